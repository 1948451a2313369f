"""The work that users of the framework have it do, as cases that can be timed.

Each case is one call, or one forward and backward, through the package's
public entry points: the dense products, the token Linear, the convolutions,
the attention core, a ViT block, the Newton-Schulz iteration of the optimiser,
and the ResNet as a whole (a train step; evaluation of a batch).  All data is
float32, which is the only type that the framework computes in.

``listed()`` are the sizes of the repository's own networks at their training
batch, with ragged and smallest ones beside them; ``draw(rng)`` gives others
of the same ranges.
"""
import math

import torch

import rustnn_amd as R
from rustnn_amd import model, nn, optim, vit

DEV = "cuda"
D = torch.float64
CLASSES = 100  # fine classes of the image sets that the networks train on
SMOOTH, LR, MOM, WD = 0.1, 0.2, 0.0, 5e-4


def listed():
    return [
        # One image's logits: the least a serving program asks for.
        dict(name="resnet_eval_one", kind="resnet_eval", n=1, depth=3, width=32, img=32),
        # The ResNet-20 train step at its training batch.
        dict(name="resnet_train", kind="resnet_train", n=128, depth=3, width=32, img=32),
        # A stage-3 transformer block with a memory reader, forward and backward.
        dict(name="vit_block_reader", kind="block", n=128, dim=256, heads=4, th=8, mh=16),
        # The fused QKV Linear of a stage-3 block, forward and backward.
        dict(name="linear_qkv", kind="linear", rows=8192, fin=256, fout=768),
        # The largest dense product.
        dict(name="matmul_large", kind="matmul", m=4096, n=4096, k=4096, at=False, bt=False),
        # A dense product of sizes that no tile or 16-byte load divides.
        dict(name="matmul_ragged", kind="matmul", m=1003, n=517, k=771, at=False, bt=True),
        # A first-stage convolution layer, forward, dX and dW.
        dict(name="conv_stage1", kind="conv", n=128, cin=32, cout=32, k=3, stride=1, h=32, w=32),
        # The strided convolution that opens the third stage.
        dict(name="conv_down", kind="conv", n=128, cin=64, cout=128, k=3, stride=2, h=16, w=16),
        # A convolution over a last, partial batch of images of another format.
        dict(name="conv_ragged", kind="conv", n=37, cin=48, cout=80, k=3, stride=1, h=23, w=29),
        # Self-attention over 8 x 8 tokens, diagonal masked, forward and backward.
        dict(name="attn_self", kind="attn", n=128, heads=4, dh=64, th=8, mh=0),
        # Cross-attention of 8 x 8 tokens over a 16 x 16 memory.
        dict(name="attn_cross", kind="attn", n=128, heads=4, dh=64, th=8, mh=16),
        # The optimiser's orthogonalisation of a stage's SwiGLU matrices.
        dict(name="newton_schulz", kind="ns", count=5, rows=704, cols=256, steps=3),
    ]


def _log(rng, lo, hi, mult=1):
    """A size of [lo, hi], even over its logarithm, a multiple of mult."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(mult, int(round(v / mult)) * mult)


def draw(rng):
    """One more case, its batch halved until it is no larger than a listed one."""
    c = _draw(rng)
    while c["kind"] in ("conv", "block") and work(c)["flops"] > 4.5e10:
        c["n"] = (c["n"] + 1) // 2
    return c


def _draw(rng):
    kind = rng.choice(["matmul", "linear", "conv", "conv", "attn", "attn", "block", "ns",
                       "resnet_eval", "resnet_train"])
    mult = rng.choice([1, 1, 4, 32])  # ragged sizes and whole tiles
    if kind == "matmul":
        return dict(kind=kind, m=_log(rng, 16, 8192, mult), n=_log(rng, 16, 2048, mult),
                    k=_log(rng, 16, 4096, mult), at=rng.random() < 0.3, bt=rng.random() < 0.5)
    if kind == "linear":
        return dict(kind=kind, rows=_log(rng, 8, 16384, mult), fin=_log(rng, 32, 1152, mult),
                    fout=_log(rng, 20, 1152, mult))
    if kind == "conv":
        s = _log(rng, 6, 34)
        k, stride = rng.choice([(3, 1), (3, 1), (3, 2), (1, 2), (1, 1)])
        return dict(kind=kind, n=_log(rng, 1, 256), cin=_log(rng, 3, 128, mult),
                    cout=_log(rng, 16, 256, mult), k=k, stride=stride, h=s,
                    w=rng.choice([s, _log(rng, 6, 34)]))
    if kind == "attn":
        th = rng.randint(2, 8)
        return dict(kind=kind, n=_log(rng, 1, 256), heads=rng.choice([3, 4, 6]),
                    dh=rng.choice([32, 64]), th=th, mh=rng.choice([0, 0, 2 * th]))
    if kind == "block":
        heads = rng.choice([2, 4, 6])
        th = rng.choice([4, 6, 8])
        return dict(kind=kind, n=_log(rng, 1, 128), dim=64 * heads, heads=heads, th=th,
                    mh=rng.choice([0, 2 * th]))
    if kind == "ns":
        return dict(kind=kind, count=rng.randint(1, 6), rows=_log(rng, 64, 1152, mult),
                    cols=_log(rng, 64, 512, mult), steps=3)
    return dict(kind=kind, n=_log(rng, 1, 128), depth=rng.randint(1, 3),
                width=rng.choice([16, 32]), img=32)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEV) * std


def _conv_inputs(c, seed):
    """Activations after a ReLU, Kaiming weights, a small output gradient."""
    g = _gen(seed)
    k = c["k"]
    oh, ow = _out(c["h"], k, c["stride"]), _out(c["w"], k, c["stride"])
    return (_normal(g, (c["n"], c["cin"], c["h"], c["w"])).relu_(),
            _normal(g, (c["cout"], c["cin"], k, k), math.sqrt(2.0 / (c["cin"] * k * k))),
            _normal(g, (c["n"], c["cout"], oh, ow), 1e-3))


def _out(s, k, stride):
    return (s + 2 * (k // 2) - k) // stride + 1


def _linear_inputs(c, seed):
    g = _gen(seed)
    return (_normal(g, (c["rows"], c["fin"])), _normal(g, (c["fout"], c["fin"]), 0.02),
            _normal(g, c["fout"], 0.02), _normal(g, (c["rows"], c["fout"]), 1e-3))


def _matmul_inputs(c, seed):
    g = _gen(seed)
    m, n, k = c["m"], c["n"], c["k"]
    return (_normal(g, (k, m) if c["at"] else (m, k)),
            _normal(g, (n, k) if c["bt"] else (k, n), 0.02))


def _grids(c):
    """Query and key grid sides of an attention case (mh = 0: self)."""
    return c["th"], c["mh"] or c["th"]


def _attn_inputs(c, seed):
    """Self-attention's [n, t, 3c] buffer, or queries and the [n, tk, 2c]
    memory; temperature about 1 / sqrt(dh) and a learned bias."""
    g = _gen(seed)
    th, mh = _grids(c)
    ch, n = c["heads"] * c["dh"], c["n"]
    if c["mh"]:
        q, kv = _normal(g, (n, th * th, ch)), _normal(g, (n, mh * mh, 2 * ch))
    else:
        q = kv = _normal(g, (n, th * th, 3 * ch))
    _, nrel = R.rel_index(th, th, mh, mh)
    tau = c["dh"] ** -0.5 * (1.0 + _normal(g, c["heads"], 0.1))
    return q, kv, tau, _normal(g, c["heads"] * nrel, 0.2), _normal(g, (n, th * th, ch), 1e-3)


def _block_inputs(c, seed):
    g = _gen(seed)
    t, d = c["th"] ** 2, c["dim"]
    mem = _normal(g, (c["n"], c["mh"] ** 2, 2 * d)) if c["mh"] else None
    return _normal(g, (c["n"], t, d)), mem, _normal(g, (c["n"], t, d), 1e-3)


def _make_block(c, seed):
    """A Block of a seed's weights, its LayerScales as training leaves them."""
    b = vit.Block(c["dim"], c["heads"], c["th"], c["th"], (c["mh"], c["mh"]) if c["mh"] else None,
                  7, 0.0, 1, 0.1, seed)
    ps = []
    b.for_each_param(ps.append)
    return b, ps


def _images(c, seed):
    g = _gen(seed)
    return (_normal(g, (c["n"], 3, c["img"], c["img"])),
            torch.randint(0, CLASSES, (c["n"],), generator=g, device=DEV, dtype=torch.int32))


def _make_resnet(c, seed):
    """A ResNet with the gammas away from their initial 1 and 0 and the
    running statistics away from 0 and 1, as in training."""
    net = model.ResNet(c["depth"], c["width"], CLASSES, seed)
    g = _gen(seed + 1)
    v = net.params()
    at = 0
    for ln, decay in net.tensor_lens():
        if not decay:
            v[at:at + ln] += _normal(g, ln, 0.1) + 0.2
        at += ln
    net.set_params(v)
    b = net.buffers()
    net.set_buffers((b + torch.rand(b.shape, generator=g, device=DEV) * 0.5).contiguous())
    return net


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"c": c}
    if kind == "matmul":
        a, b = _matmul_inputs(c, seed)
        s.update(a=a, b=b, y=torch.empty(c["m"], c["n"], device=DEV))
    elif kind == "linear":
        x, w, b, dy = _linear_inputs(c, seed)
        s.update(x=x, dy=dy, lin=R.Linear(c["fin"], c["fout"], True, w.reshape(-1), b))
    elif kind == "conv":
        x, w, dy = _conv_inputs(c, seed)
        s.update(x=x, dy=dy, conv=R.Conv2d(c["cin"], c["cout"], c["k"], c["stride"], c["k"] // 2,
                                           w.view(c["cout"], -1)))
    elif kind == "attn":
        th, mh = _grids(c)
        q, kv, tau, rel, do = _attn_inputs(c, seed)
        idx, nrel = R.rel_index(th, th, mh, mh)
        core = R.Core(c["heads"], c["dh"], th * th, mh * mh, idx, nrel, not c["mh"])
        dq = torch.empty_like(q)
        s.update(q=q, kv=kv, tau=tau, rel=rel, do=do, core=core, dq=dq,
                 dkv=torch.empty_like(kv) if c["mh"] else dq, dtau=torch.zeros_like(tau),
                 drel=torch.zeros_like(rel))
    elif kind == "block":
        x, mem, dz = _block_inputs(c, seed)
        blk, ps = _make_block(c, seed)
        s.update(x=x, mem=mem, dz=dz, blk=blk, ps=ps,
                 dmem=torch.empty_like(mem) if c["mh"] else None)
    elif kind == "ns":
        g = _normal(_gen(seed), (c["count"], c["rows"] * c["cols"]), 1e-3)
        s.update(g=g, m=torch.empty_like(g))
    else:
        x, labels = _images(c, seed)
        net = _make_resnet(c, seed)
        s.update(x=x, labels=labels, net=net, p0=net.params(), loss=torch.zeros(1, device=DEV))
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["c"]
    return _RUN[c["kind"]](c, s)


def _run_matmul(c, s):
    return R.matmul(c["m"], c["n"], c["k"], s["a"], c["at"], s["b"], c["bt"], s["y"])


def _run_linear(c, s):
    lin = s["lin"]
    torch._foreach_zero_([lin.gw, lin.gb])
    y = lin.forward(s["x"], c["rows"])
    dx = lin.backward(s["dy"])
    return dict(y=y, dx=dx, dw=lin.gw, db=lin.gb)


def _run_conv(c, s):
    conv = s["conv"]
    conv.g.zero_()
    y = conv.forward(s["x"], c["n"], c["h"], c["w"])
    dx = conv.backward(s["dy"])
    return dict(y=y, dx=dx, dw=conv.g)


def _run_attn(c, s):
    ch = c["heads"] * c["dh"]
    lay = (ch, 0, s["kv"], 2 * ch, 0, ch) if c["mh"] else (3 * ch, 0, s["kv"], 3 * ch, ch, 2 * ch)
    torch._foreach_zero_([s["dtau"], s["drel"]])
    p, o = s["core"].forward(c["n"], s["q"], *lay, s["tau"], s["rel"])
    s["core"].backward(c["n"], s["q"], *lay, s["tau"], p, s["do"], s["dq"], s["dkv"], s["dtau"],
                       s["drel"], set_dq=True, set_dkv=True)
    return dict(p=p, o=o, dq=s["dq"], dkv=s["dkv"], dtau=s["dtau"], drel=s["drel"])


def _run_block(c, s):
    blk = s["blk"]
    grads = [p.g for p in s["ps"]]
    torch._foreach_zero_(grads)
    blk.ctx.set_defer(True)  # as the ViT's train step runs its blocks
    y = blk.forward(s["x"], s["mem"], True, 0)
    dx = blk.backward(s["dz"], s["mem"], s["dmem"], set_dmem=True)
    blk.ctx.set_defer(False)
    return dict(y=y, dx=dx, dmem=s["dmem"], grads=grads)


def _run_ns(c, s):
    s["m"].copy_(s["g"])
    return optim.newton_schulz(s["m"], c["rows"], c["cols"], c["steps"])


def _run_resnet_eval(c, s):
    return s["net"].forward(s["x"], False)


def _run_resnet_train(c, s):
    """One step from the prepared weights (so that every pass is the same
    step): the loss, the new weights and the momenta (without momentum, the
    gradients plus the weight decay)."""
    net = s["net"]
    net.set_params(s["p0"])
    net.train_step(s["x"], s["labels"], SMOOTH, LR, MOM, WD, s["loss"])
    return dict(loss=s["loss"], params=net.params(), momenta=net.momenta())


_RUN = dict(matmul=_run_matmul, linear=_run_linear, conv=_run_conv, attn=_run_attn,
            block=_run_block, ns=_run_ns, resnet_eval=_run_resnet_eval,
            resnet_train=_run_resnet_train)


# ------------------------------------------------------------------ its least work
def _resnet_work(c):
    """(parameters, forward multiply-adds of an image)."""
    img, w = c["img"], c["width"]
    par, mac = 27 * w, 27 * w * img * img
    cin = w
    for stage in range(3):
        co = w << stage
        for b in range(c["depth"]):
            s = 2 if stage and not b else 1
            img //= s
            k = 9 * cin * co + 9 * co * co + (cin * co if s == 2 or cin != co else 0)
            par, mac = par + k, mac + k * img * img
            cin = co
    return par + cin * CLASSES, mac + cin * CLASSES


def work(case):
    c, kind = case, case["kind"]
    if kind == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "linear":
        r, i, o = c["rows"], c["fin"], c["fout"]
        return {"bytes": 4 * (2 * r * i + 2 * r * o + 2 * i * o + 2 * o), "flops": 6 * r * i * o}
    if kind == "conv":
        k = c["k"]
        oh, ow = _out(c["h"], k, c["stride"]), _out(c["w"], k, c["stride"])
        x, y = c["n"] * c["cin"] * c["h"] * c["w"], c["n"] * c["cout"] * oh * ow
        wt = c["cout"] * c["cin"] * k * k
        return {"bytes": 4 * (2 * x + 2 * y + 2 * wt), "flops": 6 * wt * c["n"] * oh * ow}
    if kind == "attn":
        th, mh = _grids(c)
        tq, tk, ch, n = th * th, mh * mh, c["heads"] * c["dh"], c["n"]
        # q, k, v, their gradients, o and do; the probabilities are an output
        return {"bytes": 4 * n * (ch * (4 * tq + 4 * tk) + c["heads"] * tq * tk),
                "flops": 12 * n * ch * tq * tk}
    if kind == "block":
        n, d, t, tm = c["n"], c["dim"], c["th"] ** 2, c["mh"] ** 2
        hid = -(-(4 * d // 3) // 16) * 16
        par = d * (4 * d + 3 * hid + 9) + (2 * d * d if tm else 0)
        mac = n * t * (par + 2 * d * (t + tm))
        return {"bytes": 4 * (4 * n * t * d + 4 * n * tm * d + 2 * par), "flops": 6 * mac}
    if kind == "ns":
        a, b = min(c["rows"], c["cols"]), max(c["rows"], c["cols"])
        # X X^T and its square are symmetric: half their products
        return {"bytes": 8 * c["count"] * a * b,
                "flops": c["count"] * c["steps"] * (a * a * b + a ** 3 + 2 * a * a * b)}
    par, mac = _resnet_work(c)
    x = c["n"] * 3 * c["img"] ** 2
    if kind == "resnet_eval":
        return {"bytes": 4 * (x + par + c["n"] * CLASSES), "flops": 2 * c["n"] * mac}
    return {"bytes": 4 * (x + 5 * par), "flops": 6 * c["n"] * mac}


def tolerance(case):
    return dict(_TOL[case["kind"]])


# About four times the distance from the same pass in 64 bits, over drawn cases too.  In the
# train step a value at a ReLU that another rounding moves to the other side of zero counts.
_TOL = dict(matmul={"rel": 4e-6}, linear={"rel": 4e-6}, conv={"rel": 4e-6}, attn={"rel": 4e-6},
            block={"rel": 8e-6}, ns={"rel": 4e-6}, resnet_eval={"rel": 4e-6},
            resnet_train={"rel": 2e-3})


# ------------------------------------------------------------------ in 64 bits
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _leaf(t):
    return t.to(D).requires_grad_(True)


def _grad(out, dout, leaves):
    return [g.detach() for g in torch.autograd.grad(out, leaves, dout.to(D))]


def _exact_matmul(c, seed):
    a, b = (t.to(D) for t in _matmul_inputs(c, seed))
    return (a.T if c["at"] else a) @ (b.T if c["bt"] else b)


def _exact_linear(c, seed):
    x, w, b, dy = (t.to(D) for t in _linear_inputs(c, seed))
    return dict(y=(x @ w.T + b).reshape(-1), dx=(dy @ w).reshape(-1), dw=(dy.T @ x).reshape(-1),
                db=dy.sum(0))


def _conv64(x, w, stride):
    """A convolution with "same" padding as one product over its windows."""
    co, ci, k, _ = w.shape
    n, _, h, wd = x.shape
    cols = torch.nn.functional.unfold(x, k, padding=k // 2, stride=stride)
    cols = cols.permute(1, 0, 2).reshape(ci * k * k, -1)
    y = w.reshape(co, -1) @ cols
    return y.view(co, n, _out(h, k, stride), _out(wd, k, stride)).permute(1, 0, 2, 3)


def _exact_conv(c, seed):
    x, w, dy = _conv_inputs(c, seed)
    x, w = _leaf(x), _leaf(w)
    y = _conv64(x, w, c["stride"])
    dx, dw = _grad(y, dy, [x, w])
    return dict(y=y.detach().reshape(-1), dx=dx.reshape(-1), dw=dw.view(c["cout"], -1))


def _core64(q, k, v, tau, rel, idx, masked):
    """q [n, tq, h, d], k and v [n, tk, h, d] -> (p, o)."""
    q, k, v = (t.permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    x = tau.view(1, -1, 1, 1) * (q @ k.transpose(2, 3).contiguous())
    x = x + rel.view(tau.numel(), -1)[:, idx]
    if masked:
        x = x.masked_fill(torch.eye(x.shape[-1], dtype=torch.bool, device=x.device), -math.inf)
    p = torch.softmax(x, -1)
    return p, (p @ v).permute(0, 2, 1, 3)


def _rel64(th, mh):
    """The bias slot of (query, key): their distance on the finer grid."""
    r = 1 if mh == th else 2
    q, m = torch.arange(th, device=DEV) * r, torch.arange(mh, device=DEV)
    dif = q[:, None] - m[None, :] + mh - 1
    span = r * (th - 1) + mh
    return (dif[:, None, :, None] * span + dif[None, :, None, :]).reshape(th * th, mh * mh)


def _exact_attn(c, seed):
    th, mh = _grids(c)
    h, d, n, ch = c["heads"], c["dh"], c["n"], c["heads"] * c["dh"]
    q, kv, tau, rel, do = _attn_inputs(c, seed)
    leaves = [_leaf(q), _leaf(kv) if c["mh"] else None, _leaf(tau), _leaf(rel)]
    ql, kvl, taul, rell = leaves
    if c["mh"]:
        qq, kk, vv = ql, kvl[..., :ch], kvl[..., ch:]
    else:
        qq, kk, vv = ql.split(ch, -1)
    p, o = _core64(*(t.reshape(n, -1, h, d) for t in (qq, kk, vv)), taul, rell, _rel64(th, mh),
                   not c["mh"])
    got = _grad(o.reshape(n, -1, ch), do, [t for t in leaves if t is not None])
    dq, dkv = got[0], got[1] if c["mh"] else got[0]
    return dict(p=p.detach().reshape(-1), o=o.detach().reshape(-1), dq=dq, dkv=dkv, dtau=got[-2],
                drel=got[-1])


def _exact_block(c, seed):
    d, h, n, th = c["dim"], c["heads"], c["n"], c["th"]
    t, dh, F = th * th, d // h, torch.nn.functional
    x, mem, dz = _block_inputs(c, seed)
    ps = [_leaf(p.v) for p in _make_block(c, seed)[1]]
    it = iter(ps)
    x = _leaf(x)
    mem = _leaf(mem) if c["mh"] else None

    def lin(v, fout):
        w, b = next(it), next(it)
        return v @ w.view(fout, -1).T + b

    def norm(v):
        return F.layer_norm(v, (d,), next(it), next(it), 1e-5)

    def heads(*ts):
        return [u.reshape(n, -1, h, dh) for u in ts]

    hh = norm(x)
    qkv = lin(hh, 3 * d)
    wp, bp, tau, rel = next(it), next(it), next(it), next(it)
    _, o = _core64(*heads(*qkv.split(d, -1)), tau, rel, _rel64(th, th), True)
    a = o.reshape(n, t, d) @ wp.view(d, d).T + bp
    w9, b9 = next(it).view(9, d), next(it)
    img = F.pad(hh.view(n, th, th, d), (0, 0, 1, 1, 1, 1))
    dw = b9 + sum(w9[3 * i + j] * img[:, i:i + th, j:j + th] for i in range(3) for j in range(3))
    gamma, ls1 = next(it), next(it)
    y = x + ls1 * (a + gamma * dw.reshape(n, t, d))
    if mem is not None:
        q = lin(hh, d)
        wp, bp, tau, rel = next(it), next(it), next(it), next(it)
        _, o = _core64(*heads(q, mem[..., :d], mem[..., d:]), tau, rel, _rel64(th, c["mh"]), False)
        y = y + next(it) * (o.reshape(n, t, d) @ wp.view(d, d).T + bp)
    h2 = norm(y)
    hid = -(-(4 * d // 3) // 16) * 16
    gate, up = lin(h2, 2 * hid).split(hid, -1)
    m = lin(F.silu(gate) * up, d)
    z = y + next(it) * m
    got = _grad(z, dz, [x] + ([mem] if mem is not None else []) + ps)
    dmem = got.pop(1) if mem is not None else None
    return dict(y=z.detach(), dx=got[0], dmem=dmem, grads=got[1:])


def _exact_ns(c, seed):
    g = _normal(_gen(seed), (c["count"], c["rows"] * c["cols"]), 1e-3).to(D)
    x = g.view(c["count"], c["rows"], c["cols"])
    tall = c["rows"] > c["cols"]
    x = (x.transpose(1, 2) if tall else x).contiguous()
    x = x / (x.flatten(1).norm(dim=1) + 1e-7).view(-1, 1, 1)
    for _ in range(c["steps"]):
        a = x @ x.transpose(1, 2).contiguous()
        b = -4.7750 * a + 2.0315 * (a @ a)
        x = 3.4445 * x + b @ x
    x = x.transpose(1, 2) if tall else x
    return x.reshape(c["count"], -1)


def _resnet64(c, seed, train):
    """The network in 64 bits: (logits, its parameters)."""
    net = _make_resnet(c, seed)
    flat, stats = net.params(), net.buffers().to(D)
    lens = [ln for ln, _ in net.tensor_lens()]
    net.close()
    ps = [_leaf(v) for v in flat.split(lens)]
    it, at = iter(ps), 0

    def conv_bn(h, co, k, s):
        nonlocal at
        y = _conv64(h, next(it).view(co, h.shape[1], k, k), s)
        g, b = next(it).view(1, -1, 1, 1), next(it).view(1, -1, 1, 1)
        if train:
            mean = y.mean((0, 2, 3), keepdim=True)
            var = ((y - mean) ** 2).mean((0, 2, 3), keepdim=True)
        else:
            mean = stats[at:at + co].view(1, -1, 1, 1)
            var = stats[at + co:at + 2 * co].view(1, -1, 1, 1)
            at += 2 * co
        return (y - mean) / torch.sqrt(var + 1e-5) * g + b

    x, labels = _images(c, seed)
    h = conv_bn(x.to(D), c["width"], 3, 1).relu()
    for stage in range(3):
        co = c["width"] << stage
        for b in range(c["depth"]):
            s = 2 if stage and not b else 1
            y = conv_bn(conv_bn(h, co, 3, s).relu(), co, 3, 1)
            h = (y + (conv_bn(h, co, 1, s) if s == 2 or h.shape[1] != co else h)).relu()
    w, bias = next(it).view(CLASSES, -1), next(it)
    return h.mean((2, 3)) @ w.T + bias, ps, labels.long()


def _exact_resnet_eval(c, seed):
    with torch.no_grad():
        return _resnet64(c, seed, False)[0]


def _exact_resnet_train(c, seed):
    net = _make_resnet(c, seed)
    decay = [d for _, d in net.tensor_lens()]
    net.close()
    z, ps, labels = _resnet64(c, seed, True)
    loss = torch.nn.functional.cross_entropy(z, labels, label_smoothing=SMOOTH)
    g = [v + (WD * p.detach() if d else 0.0)
         for v, p, d in zip(torch.autograd.grad(loss, ps), ps, decay)]
    # a gradient jumps where a value at a ReLU rounds to the other side of zero (about one in
    # 1e7 of them does at 32 bits): no momenta; the weights move by a fifth of them
    return dict(loss=loss.detach().view(1), momenta=None,
                params=torch.cat([p.detach() - LR * v for p, v in zip(ps, g)]))


_EXACT = dict(matmul=_exact_matmul, linear=_exact_linear, conv=_exact_conv, attn=_exact_attn,
              block=_exact_block, ns=_exact_ns, resnet_eval=_exact_resnet_eval,
              resnet_train=_exact_resnet_train)
