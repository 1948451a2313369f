"""GPU parity: batched small attention (attn.rs Core forward/backward and
rel_index) against the CPU oracle, at BASELINE config 2 and at the reference's
attention gradcheck shapes (check.rs:294-358)."""
import numpy as np
import pytest

from conftest import TOL, rel_frob, to_dev, to_host

pytestmark = pytest.mark.gpu


def make_case(orc, n, h, dh, th, tw, mh, mw, variant, seed):
    """Self attention (mh == th): SelfAttn buffer [n, t, 3c] with q/k/v at
    0/c/2c (attn.rs:393-404).  Cross: q [n, tq, c], memory [n, tk, 2c] with
    K at 0, V at c (attn.rs:508-519)."""
    rng = orc.Rng(seed)
    c = h * dh
    tq, tk = th * tw, mh * mw
    relidx, nrel = orc.rel_index(th, tw, mh, mw)
    selfattn = (mh == th and mw == tw)
    scale = np.float32(1.0 / np.sqrt(dh))
    if selfattn:
        qkv = rng.rand_vec(n * tq * 3 * c) * scale
        q, kv = qkv, qkv
        geo = dict(qstride=3 * c, qoff=0, kvstride=3 * c, koff=c, voff=2 * c)
    else:
        q = rng.rand_vec(n * tq * c) * scale
        kv = rng.rand_vec(n * tk * 2 * c) * scale
        geo = dict(qstride=c, qoff=0, kvstride=2 * c, koff=0, voff=c)
    if variant == "plain":   # BASELINE config 2 as specified
        tau = np.ones(h, np.float32)
        rel = np.zeros(h * nrel, np.float32)
        mask = False
    else:                    # SelfAttn/CrossAttn defaults + random rel (check.rs:300, 334)
        tau = np.full(h, 1.0 / np.sqrt(dh), np.float32)
        rel = rng.rand_vec(h * nrel)
        mask = selfattn
    dout = rng.rand_vec(n * tq * c)
    return dict(q=q, kv=kv, geo=geo, tau=tau, rel=rel, mask=mask, relidx=relidx, nrel=nrel,
                dout=dout, tq=tq, tk=tk, selfattn=selfattn)


CASES = [
    # name, n, h, dh, th, tw, mh, mw, variant
    ("cfg2_plain", 128, 4, 32, 8, 8, 8, 8, "plain"),
    ("cfg2_lsa", 128, 4, 32, 8, 8, 8, 8, "lsa"),
    ("gc_self", 3, 2, 4, 3, 3, 3, 3, "lsa"),
    ("gc_cross", 3, 2, 4, 3, 3, 6, 6, "lsa"),
    ("dh64_t16", 16, 6, 64, 4, 4, 4, 4, "lsa"),
    ("dh64_t64", 8, 4, 64, 8, 8, 8, 8, "lsa"),
    # tq or tk above 64: the composed path (batched GEMMs + row kernels)
    # tq <= 64 and tk 128 / 256 with dh 32 / 64: one fused workgroup per
    # (image, head) (attn_fwd_long_kernel) in the forward
    ("cross_tk256", 8, 4, 64, 8, 8, 16, 16, "lsa"),   # the rustvit's cross-attention
    ("cross_tk128_dh32_tq49", 4, 3, 32, 7, 7, 8, 16, "lsa"),
    ("cross_tk256_dh32_tq36", 4, 2, 32, 6, 6, 16, 16, "plain"),
    ("self_t100", 4, 2, 48, 10, 10, 10, 10, "lsa"),   # masked self-attention, 100 tokens
    ("cross_tk81_dh80", 3, 2, 80, 3, 3, 9, 9, "lsa"),
]


@pytest.mark.parametrize("name,n,h,dh,th,tw,mh,mw,variant", CASES, ids=[c[0] for c in CASES])
def test_attn_parity(rnn, orc, name, n, h, dh, th, tw, mh, mw, variant):
    cs = make_case(orc, n, h, dh, th, tw, mh, mw, variant, seed=7)
    g = cs["geo"]
    d = orc.attn_desc(h, dh, cs["tq"], cs["tk"], g["qstride"], g["qoff"], g["kvstride"],
                      g["koff"], g["voff"], cs["relidx"], cs["nrel"], cs["mask"])
    with orc.threads(8):
        p_want, o_want = orc.attn_forward(d, n, cs["q"], cs["kv"], cs["tau"], cs["rel"])
    core = rnn.Core(h, dh, cs["tq"], cs["tk"], cs["relidx"], cs["nrel"], cs["mask"])
    Q = to_dev(cs["q"])
    KV = Q if cs["selfattn"] else to_dev(cs["kv"])
    TAU, REL = to_dev(cs["tau"]), to_dev(cs["rel"])
    P, O = core.forward(n, Q, g["qstride"], g["qoff"], KV, g["kvstride"], g["koff"], g["voff"],
                        TAU, REL)
    assert rel_frob(to_host(P), p_want) < TOL, "p"
    assert rel_frob(to_host(O), o_want) < TOL, "o"

    # backward: separate dq / dkv buffers with non-zero initial content (+=)
    nq, nkv = cs["q"].size, cs["kv"].size
    r = np.random.default_rng(3)
    dq0 = r.standard_normal(nq).astype(np.float32)
    dkv0 = r.standard_normal(nkv).astype(np.float32)
    dtau0 = r.standard_normal(h).astype(np.float32)
    drel0 = r.standard_normal(h * cs["nrel"]).astype(np.float32)
    with orc.threads(8):
        dq_w, dkv_w, dtau_w, drel_w = orc.attn_backward(d, n, cs["q"], cs["kv"], cs["tau"], p_want,
                                                        cs["dout"], dq0, dkv0, dtau0, drel0)
    dq, dkv = to_dev(dq0.copy()), to_dev(dkv0.copy())
    dtau, drel = to_dev(dtau0.copy()), to_dev(drel0.copy())
    core.backward(n, Q, g["qstride"], g["qoff"], KV, g["kvstride"], g["koff"], g["voff"], TAU,
                  to_dev(p_want), to_dev(cs["dout"]), dq, dkv, dtau, drel)
    assert rel_frob(to_host(dq) - dq0, dq_w - dq0) < TOL, "dq"
    assert rel_frob(to_host(dkv) - dkv0, dkv_w - dkv0) < TOL, "dkv"
    assert rel_frob(to_host(dtau) - dtau0, dtau_w - dtau0) < TOL, "dtau"
    assert rel_frob(to_host(drel) - drel0, drel_w - drel0) < TOL, "drel"


def _cols(size, stride, offs, width):
    """Mask of the columns [off, off + width) of every row, for each off."""
    m = np.zeros((size // stride, stride), bool)
    for off in offs:
        m[:, off:off + width] = True
    return m.ravel()


SET_CASES = [c for c in CASES if c[0] in ("cfg2_lsa", "gc_cross", "dh64_t16", "cross_tk256",
                                          "self_t100")]


@pytest.mark.parametrize("flags", [1, 2, 3])
@pytest.mark.parametrize("name,n,h,dh,th,tw,mh,mw,variant", SET_CASES,
                         ids=[c[0] for c in SET_CASES])
def test_attn_backward_set(rnn, orc, flags, name, n, h, dh, th, tw, mh, mw, variant):
    """rnn_attn_backward_ex: an operand flagged for overwriting receives what
    accumulating into a zeroed buffer gives (bit for bit), and its old
    contents (NaN here) are never read; an unflagged one accumulates."""
    cs = make_case(orc, n, h, dh, th, tw, mh, mw, variant, seed=11)
    g = cs["geo"]
    d = orc.attn_desc(h, dh, cs["tq"], cs["tk"], g["qstride"], g["qoff"], g["kvstride"],
                      g["koff"], g["voff"], cs["relidx"], cs["nrel"], cs["mask"])
    with orc.threads(8):
        p_w, _ = orc.attn_forward(d, n, cs["q"], cs["kv"], cs["tau"], cs["rel"])
    core = rnn.Core(h, dh, cs["tq"], cs["tk"], cs["relidx"], cs["nrel"], cs["mask"])
    Q = to_dev(cs["q"])
    KV = Q if cs["selfattn"] else to_dev(cs["kv"])
    TAU, P, DO = to_dev(cs["tau"]), to_dev(p_w), to_dev(cs["dout"])
    nq, nkv = cs["q"].size, cs["kv"].size
    r = np.random.default_rng(5)
    set_q, set_kv = bool(flags & 1), bool(flags & 2)
    dq0 = np.zeros(nq, np.float32) if set_q else r.standard_normal(nq).astype(np.float32)
    dkv0 = np.zeros(nkv, np.float32) if set_kv else r.standard_normal(nkv).astype(np.float32)
    dtau0 = r.standard_normal(h).astype(np.float32)
    drel0 = r.standard_normal(h * cs["nrel"]).astype(np.float32)
    # the accumulating call into zeroed buffers, then the flagged call into NaN
    want = [to_dev(a.copy()) for a in (dq0, dkv0, dtau0, drel0)]
    core.backward(n, Q, g["qstride"], g["qoff"], KV, g["kvstride"], g["koff"], g["voff"], TAU, P,
                  DO, *want)
    nan = np.float32(np.nan)
    got = [to_dev(np.full(nq, nan) if set_q else dq0.copy()),
           to_dev(np.full(nkv, nan) if set_kv else dkv0.copy()),
           to_dev(dtau0.copy()), to_dev(drel0.copy())]
    core.backward(n, Q, g["qstride"], g["qoff"], KV, g["kvstride"], g["koff"], g["voff"], TAU, P,
                  DO, *got, set_dq=set_q, set_dkv=set_kv)
    width = h * dh
    mq = _cols(nq, g["qstride"], [g["qoff"]], width)
    mkv = _cols(nkv, g["kvstride"], [g["koff"], g["voff"]], width)
    for nm, a, b, m in (("dq", got[0], want[0], mq), ("dkv", got[1], want[1], mkv),
                        ("dtau", got[2], want[2], None), ("drel", got[3], want[3], None)):
        a, b = to_host(a), to_host(b)
        if m is not None:
            a, b = a[m], b[m]
        assert np.isfinite(a).all() and np.array_equal(a, b), nm
    with orc.threads(8):
        dq_w, dkv_w, _, _ = orc.attn_backward(d, n, cs["q"], cs["kv"], cs["tau"], p_w, cs["dout"],
                                              dq0, dkv0, dtau0, drel0)
    assert rel_frob(to_host(got[0])[mq] - dq0[mq], dq_w[mq] - dq0[mq]) < TOL
    assert rel_frob(to_host(got[1])[mkv] - dkv0[mkv], dkv_w[mkv] - dkv0[mkv]) < TOL


@pytest.mark.parametrize("n,h,dh,t", [(32, 4, 32, 8), (4, 2, 48, 10)])
def test_attn_aliased_dq_dkv(rnn, orc, n, h, dh, t):
    """SelfAttn accumulates dq and dk/dv into one fused-QKV gradient buffer
    (attn.rs:418-438); the device path may take them aliased (both the
    register-resident kernels and, at 100 tokens, the composed path)."""
    cs = make_case(orc, n, h, dh, t, t, t, t, "lsa", seed=13)
    g = cs["geo"]
    T = t * t
    d = orc.attn_desc(h, dh, T, T, g["qstride"], 0, g["kvstride"], g["koff"], g["voff"],
                      cs["relidx"], cs["nrel"], True)
    p_w, _ = orc.attn_forward(d, n, cs["q"], cs["kv"], cs["tau"], cs["rel"])
    z = np.zeros(cs["q"].size, np.float32)
    dq_w, dkv_w, _, _ = orc.attn_backward(d, n, cs["q"], cs["kv"], cs["tau"], p_w, cs["dout"], z, z,
                                          np.zeros(h, np.float32),
                                          np.zeros(h * cs["nrel"], np.float32))
    want = dq_w + dkv_w  # attn.rs:438
    core = rnn.Core(h, dh, T, T, cs["relidx"], cs["nrel"], True)
    Q = to_dev(cs["q"])
    dab = to_dev(z.copy())
    dtau = to_dev(np.zeros(h, np.float32))
    drel = to_dev(np.zeros(h * cs["nrel"], np.float32))
    core.backward(n, Q, g["qstride"], 0, Q, g["kvstride"], g["koff"], g["voff"], to_dev(cs["tau"]),
                  to_dev(p_w), to_dev(cs["dout"]), dab, dab, dtau, drel)
    assert rel_frob(to_host(dab), want) < TOL


@pytest.mark.parametrize("th,tw,mh,mw", [(8, 8, 8, 8), (8, 8, 16, 16), (4, 4, 4, 4), (3, 3, 6, 6),
                                         (3, 3, 3, 3), (2, 5, 4, 10)])
def test_rel_index_bit_exact(rnn, orc, th, tw, mh, mw):
    want, nrel_w = orc.rel_index(th, tw, mh, mw)
    got, nrel = rnn.rel_index(th, tw, mh, mw)
    assert nrel == nrel_w and np.array_equal(got, want)
    dev = to_host(rnn.dbg_rel_index(th, tw, mh, mw)).view(np.uint32)
    assert np.array_equal(dev, want)


def test_attn_unsupported_shape_raises(rnn, orc):
    relidx, nrel = orc.rel_index(8, 8, 8, 8)  # dh = 80 at tq = tk = 64: beyond the kernel
    core = rnn.Core(1, 80, 64, 64, relidx, nrel, False)
    q = to_dev(np.zeros(64 * 80, np.float32))
    kv = to_dev(np.zeros(64 * 160, np.float32))
    with pytest.raises(rnn.RnnError):
        core.forward(1, q, 80, 0, kv, 160, 0, 80, to_dev(np.ones(1, np.float32)),
                     to_dev(np.zeros(nrel, np.float32)))


# The long-key backward's key half: one query, a whole k step of 32, one more,
# a partial second one; an infinity and a NaN in dO (which have no split).
@pytest.mark.parametrize("h,dh,th,tw,mh,mw,acc,special", [
    (2, 64, 1, 1, 16, 16, False, False), (3, 32, 4, 8, 8, 16, True, False),
    (2, 64, 3, 11, 16, 16, False, False), (1, 64, 7, 9, 8, 16, True, False),
    (3, 32, 5, 6, 16, 16, False, False), (2, 64, 8, 8, 16, 16, False, True),
    (2, 32, 5, 8, 8, 16, True, True)])
def test_attn_long_key_gradients(rnn, h, dh, th, tw, mh, mw, acc, special):
    import torch
    n, tq, tk, c = 3, th * tw, mh * mw, h * dh
    idx, nrel = rnn.rel_index(th, tw, mh, mw)
    core = rnn.Core(h, dh, tq, tk, idx, nrel, False)
    gen = torch.Generator(device="cuda").manual_seed(tq + tk)
    rnd = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
    q, kv, do = rnd(n, tq, c), rnd(n, tk, 2 * c), rnd(n, tq, c)
    tau, rel = torch.full((h,), dh ** -0.5, device="cuda"), rnd(h * nrel) * 0.2
    if special:
        do[0, tq - 1, 1], do[1, 0, c - 1] = float("inf"), float("nan")
    lay = (c, 0, kv, 2 * c, 0, c)
    p, _ = core.forward(n, q, *lay, tau, rel)
    dq, dtau, drel = torch.zeros_like(q), torch.zeros_like(tau), torch.zeros_like(rel)
    dkv = torch.full_like(kv, 1.0 if acc else float("nan"))
    core.backward(n, q, *lay, tau, p, do, dq, dkv, dtau, drel, set_dkv=not acc)
    heads = lambda t, at: t[..., at:at + c].reshape(n, -1, h, dh).transpose(1, 2).double()
    P, O, Q = p.view(n, h, tq, tk).double(), heads(do, 0), heads(q, 0)
    dp = O @ heads(kv, c).transpose(2, 3).contiguous()
    ds = P * (dp - (P * dp).sum(-1, keepdim=True)) * tau.view(1, h, 1, 1)
    for at, a, b in ((c, P, O), (0, ds, Q)):
        got = to_host(heads(dkv, at)) - (1.0 if acc else 0.0)
        want = to_host(a.transpose(2, 3).contiguous() @ b)
        fine = np.isfinite(want)
        assert np.array_equal(got[~fine], want[~fine], equal_nan=True)
        # sums of tq rounded products, each rounding 2^-24 of a partial sum; dS
        # from a dP of dh such terms; the added 1 is far larger than dK
        tol = 2.0 ** -24 * (np.sqrt(tq) + 4 * np.sqrt(dh) + 8)
        size = np.linalg.norm(want[fine]) + (np.sqrt(fine.sum()) if acc else 0.0)
        assert np.linalg.norm(got[fine] - want[fine]) < tol * size


# The long-key forward: one query, a query past a wave's 16, a partial last
# wave; infinities and a NaN in K and V (which have no split).
@pytest.mark.parametrize("h,dh,th,tw,mh,mw,special", [
    (2, 64, 1, 1, 16, 16, False), (3, 32, 3, 6, 8, 16, False), (1, 64, 7, 9, 8, 16, False),
    (3, 32, 8, 8, 16, 16, False), (2, 64, 8, 8, 16, 16, True), (2, 32, 5, 8, 8, 16, True)])
def test_attn_long_key_forward(rnn, h, dh, th, tw, mh, mw, special):
    import torch
    n, tq, tk, c = 3, th * tw, mh * mw, h * dh
    idx, nrel = rnn.rel_index(th, tw, mh, mw)
    core = rnn.Core(h, dh, tq, tk, idx, nrel, False)
    gen = torch.Generator(device="cuda").manual_seed(tq + tk)
    rnd = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
    q, kv = rnd(n, tq, c), rnd(n, tk, 2 * c)
    if special:
        kv[0, tk - 3, 5], kv[1, 2, c + 1] = float("inf"), float("-inf")
        kv[2, tk - 1, 2 * c - 1] = float("nan")
    tau, rel = torch.full((h,), dh ** -0.5, device="cuda"), rnd(h * nrel) * 0.2
    p, o = core.forward(n, q, c, 0, kv, 2 * c, 0, c, tau, rel)
    heads = lambda t, at: t[..., at:at + c].reshape(n, -1, h, dh).transpose(1, 2).double()
    s = heads(q, 0) @ heads(kv, 0).transpose(2, 3).contiguous() * tau.view(1, h, 1, 1)
    bias = rel.view(h, nrel)[:, torch.as_tensor(np.asarray(idx).astype(np.int64), device="cuda")]
    want_p = torch.softmax(s + bias.view(1, h, tq, tk), -1)
    want_o = want_p @ heads(kv, c)
    # scores of size 6 at most, each term's and sum's rounding 2^-24 of it; the
    # exponential carries them into P, the sums over keys add 2^-24 sqrt(tk)
    tol = 2.0 ** -24 * (np.sqrt(dh) + np.sqrt(tk) + 6 * 8)
    for got, want in ((p.view(n, h, tq, tk), want_p), (o.reshape(n, tq, h, dh).transpose(1, 2),
                                                       want_o)):
        got, want = to_host(got), to_host(want)
        fine = np.isfinite(want)
        assert np.array_equal(got[~fine], want[~fine], equal_nan=True)
        assert np.linalg.norm(got[fine] - want[fine]) < tol * np.linalg.norm(want[fine])


@pytest.mark.parametrize("dh,th,mh", [(32, 4, 8), (64, 8, 16)])
@pytest.mark.parametrize("sq,sk,sv,so", [(1.0, 1.0, 1e-36, 1.0), (1.0, 1.0, 1e-36, 1e30),
                                         (1e-38, 1e30, 1.0, 1e-36), (1e28, 1e-41, 1.0, 1e-8)])
def test_attn_long_key_exponent_range(rnn, dh, th, mh, sq, sk, sv, so):
    """Q, K, V and dO far from 1, down to denormal ones."""
    import torch
    n, h, tw = 2, 2, 8
    tq, tk, c = th * tw, mh * 16, h * dh
    idx, nrel = rnn.rel_index(th, tw, mh, 16)
    core = rnn.Core(h, dh, tq, tk, idx, nrel, False)
    gen = torch.Generator(device="cuda").manual_seed(tk + dh)
    rnd = lambda s, *sh: (torch.randn(sh, generator=gen, device="cuda").double() * s).float()
    q, do = rnd(sq, n, tq, c), rnd(so, n, tq, c)
    kv = torch.cat([rnd(sk, n, tk, c), rnd(sv, n, tk, c)], -1)
    tau, rel = torch.full((h,), dh ** -0.5, device="cuda"), rnd(0.2, h * nrel)
    lay = (c, 0, kv, 2 * c, 0, c)
    p, o = core.forward(n, q, *lay, tau, rel)
    dq, dkv = torch.empty_like(q), torch.empty_like(kv)
    core.backward(n, q, *lay, tau, p, do, dq, dkv, torch.zeros_like(tau), torch.zeros_like(rel),
                  set_dq=True, set_dkv=True)
    heads = lambda t, at=0: t[..., at:at + c].reshape(n, -1, h, dh).transpose(1, 2).double()
    t = lambda a: a.transpose(2, 3).contiguous()
    Q, K, V, O = heads(q), heads(kv), heads(kv, c), heads(do)
    P = p.view(n, h, tq, tk).double()
    dp = O @ t(V)
    ds = P * (dp - (P * dp).sum(-1, keepdim=True)) * tau.view(1, h, 1, 1)
    # sums of at most tk products, dS from sums of dh; the spacing of denormals
    tol = 2.0 ** -24 * (np.sqrt(tk) + 4 * np.sqrt(dh) + 8)
    for got, want in ((heads(o.view(n, tq, c)), P @ V), (heads(dq), ds @ K),
                      (heads(dkv), t(ds) @ Q), (heads(dkv, c), t(P) @ O)):
        got, want = to_host(got.contiguous()), to_host(want.contiguous())
        size = np.linalg.norm(want) + 2.0 ** -145 * np.sqrt(want.size) / tol
        assert np.linalg.norm(got - want) < tol * size


def test_attn_long_key_one_query(rnn):
    """One query: dV and dK are single products, rounded once (dV = P dO)."""
    import torch
    n, h, dh, tk = 3, 2, 64, 256
    c = h * dh
    idx, nrel = rnn.rel_index(1, 1, 16, 16)
    core = rnn.Core(h, dh, 1, tk, idx, nrel, False)
    gen = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
    q, kv, do = rnd(n, 1, c), rnd(n, tk, 2 * c), rnd(n, 1, c)
    tau, rel = torch.full((h,), 0.125, device="cuda"), rnd(h * nrel) * 0.2
    lay = (c, 0, kv, 2 * c, 0, c)
    p, _ = core.forward(n, q, *lay, tau, rel)
    dkv = torch.empty_like(kv)
    core.backward(n, q, *lay, tau, p, do, torch.empty_like(q), dkv, torch.zeros_like(tau),
                  torch.zeros_like(rel), set_dq=True, set_dkv=True)
    want = p.view(n, h, tk, 1) * do.view(n, h, 1, dh)
    assert torch.equal(dkv[..., c:].reshape(n, tk, h, dh).transpose(1, 2), want)
