"""GPU parity: dense GEMM drivers (gemm.rs matmul / gemm_small / matmul_dw),
the Linear layer (linear.rs) and the PackedA/PackedB layouts, through the C ABI,
against the CPU oracle (restated reference) on identical seeded inputs."""
import numpy as np
import pytest

from conftest import TOL, rel_frob, to_dev, to_host

pytestmark = pytest.mark.gpu

# check.rs:147 gemmcheck shapes: partial 6x16 tiles and a K>256 block split
GEMMCHECK = [(23, 37, 19), (64, 48, 96), (7, 16, 259)]


def naive64(m, n, k, a, at, b, bt):
    A = a.reshape(k, m).T if at else a.reshape(m, k)
    B = b.reshape(n, k).T if bt else b.reshape(k, n)
    return (A.astype(np.float64) @ B.astype(np.float64)).ravel()


@pytest.mark.parametrize("m,n,k", GEMMCHECK)
@pytest.mark.parametrize("at", [False, True])
@pytest.mark.parametrize("bt", [False, True])
def test_matmul_gemmcheck(rnn, orc, m, n, k, at, bt):
    rng = orc.Rng(1234 ^ 0x1234)
    a, b = rng.rand_vec(m * k), rng.rand_vec(k * n)
    want = orc.matmul(m, n, k, a, at, b, bt)
    c = to_dev(np.zeros(m * n, np.float32))
    rnn.matmul(m, n, k, to_dev(a), at, to_dev(b), bt, c)
    got = to_host(c)
    assert rel_frob(got, want) < TOL
    assert rel_frob(got, naive64(m, n, k, a, at, b, bt)) < TOL
    # check.rs max_rel metric, tolerance 5e-3
    assert np.abs(got - want).max() / max(np.abs(want).max(), 1e-6) < 5e-3


@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_integer_bit_exact(rnn, orc, at, bt):
    m, n, k = 133, 97, 300
    r = np.random.default_rng(5)
    a = r.integers(-3, 4, m * k).astype(np.float32)
    b = r.integers(-3, 4, k * n).astype(np.float32)
    c0 = r.integers(-3, 4, m * n).astype(np.float32)
    for acc in (False, True):
        want = orc.matmul(m, n, k, a, at, b, bt, c0, acc)
        c = to_dev(c0.copy())
        rnn.matmul(m, n, k, to_dev(a), at, to_dev(b), bt, c, acc)
        assert np.array_equal(to_host(c), want)


def test_matmul_edge_cases(rnn, orc):
    c0 = np.full(12, 7.0, np.float32)
    # k == 0: C zeroed unless acc (gemm.rs:449-454)
    c = to_dev(c0.copy())
    rnn.matmul(3, 4, 0, to_dev(np.zeros(1, np.float32)), False, to_dev(np.zeros(1, np.float32)),
               False, c, False)
    assert np.array_equal(to_host(c), np.zeros(12, np.float32))
    c = to_dev(c0.copy())
    rnn.matmul(3, 4, 0, to_dev(np.zeros(1, np.float32)), False, to_dev(np.zeros(1, np.float32)),
               False, c, True)
    assert np.array_equal(to_host(c), c0)
    # m == 0 / n == 0: untouched
    c = to_dev(c0.copy())
    rnn.matmul(0, 4, 3, to_dev(np.ones(12, np.float32)), False, to_dev(np.ones(12, np.float32)),
               False, c, False)
    assert np.array_equal(to_host(c), c0)


@pytest.mark.parametrize("m,n,k,at,bt", [
    (16384, 768, 256, False, True),    # bench.rs:18 S3 qkv fwd
    (16384, 256, 768, False, False),   # bench.rs:20 S3 qkv dX
    (768, 256, 16384, True, False),    # bench.rs:21 S3 qkv dW (matmul with at)
    (4096, 384, 1024, False, True),    # bench.rs:23 merge fwd
])
def test_matmul_gemmbench_shapes(rnn, orc, m, n, k, at, bt):
    rng = orc.Rng(7)
    a, b = rng.rand_vec(m * k), rng.rand_vec(k * n)
    with orc.threads(8):
        want = orc.matmul(m, n, k, a, at, b, bt)
    c = to_dev(np.zeros(m * n, np.float32))
    rnn.matmul(m, n, k, to_dev(a), at, to_dev(b), bt, c)
    assert rel_frob(to_host(c), want) < TOL


def test_gemm_small_batched_attention_shapes(rnn, orc):
    # 512 (image, head) problems: QK^T (bt), PV, P^T dO (at)
    cnt = 512
    rng = orc.Rng(11)
    for (m, n, k, at, bt) in [(64, 64, 32, False, True), (64, 32, 64, False, False),
                              (64, 32, 64, True, False), (9, 9, 4, False, True)]:
        a = rng.rand_vec(cnt * m * k)
        b = rng.rand_vec(cnt * k * n)
        c = to_dev(np.zeros(cnt * m * n, np.float32))
        rnn.gemm_small_batched(cnt, m, n, k, to_dev(a), m * k, at, to_dev(b), k * n, bt, c, m * n)
        got = to_host(c).reshape(cnt, m * n)
        for i in (0, 1, 255, cnt - 1):
            want = orc.gemm_small(m, n, k, a[i * m * k:(i + 1) * m * k], at,
                                  b[i * k * n:(i + 1) * k * n], bt)
            assert rel_frob(got[i], want) < TOL


def test_gemm_small_k0_leaves_c(rnn, orc):
    c0 = np.arange(8, dtype=np.float32)
    c = to_dev(c0.copy())
    one = to_dev(np.ones(8, np.float32))
    rnn.gemm_small_batched(2, 2, 2, 0, one, 0, False, one, 0, False, c, 4)
    assert np.array_equal(to_host(c), c0)
    assert np.array_equal(orc.gemm_small(2, 2, 0, np.zeros(0, np.float32), False,
                                         np.zeros(0, np.float32), False, c0[:4]), c0[:4])


@pytest.mark.parametrize("m,n,k", [(768, 256, 8192), (5, 6, 3), (64, 700, 1000), (300, 40, 257)])
def test_matmul_dw(rnn, orc, m, n, k):
    rng = orc.Rng(3)
    a, b, c0 = rng.rand_vec(k * m), rng.rand_vec(k * n), rng.rand_vec(m * n)
    with orc.threads(8):
        want = orc.matmul_dw(m, n, k, a, b, c0)
    c = to_dev(c0.copy())
    rnn.matmul_dw(m, n, k, to_dev(a), to_dev(b), c)
    got = to_host(c)
    assert rel_frob(got, want) < TOL
    # deterministic: same inputs, same bits
    c2 = to_dev(c0.copy())
    rnn.matmul_dw(m, n, k, to_dev(a), to_dev(b), c2)
    assert np.array_equal(to_host(c2), got)


def test_matmul_dw_integer_exact(rnn, orc):
    m, n, k = 40, 72, 5000
    r = np.random.default_rng(9)
    a = r.integers(-2, 3, k * m).astype(np.float32)
    b = r.integers(-2, 3, k * n).astype(np.float32)
    c0 = r.integers(-2, 3, m * n).astype(np.float32)
    want = orc.matmul_dw(m, n, k, a, b, c0)
    c = to_dev(c0.copy())
    rnn.matmul_dw(m, n, k, to_dev(a), to_dev(b), c)
    assert np.array_equal(to_host(c), want)


# db is summed by the dW GEMM itself on its direct-to-LDS path (fout and fin
# multiples of 4): split-K (8192 rows; 4096 rows with a partial last row
# tile), one launch (27 rows), 128 x 128 tiles (4096 x 4096); fout = 30 takes
# the column-sum kernels.
@pytest.mark.parametrize("rows,fin,fout,bias", [(8192, 256, 768, True), (27, 8, 24, True),
                                                 (64, 384, 1024, False), (4096, 36, 100, True),
                                                 (64, 4096, 4096, True), (100, 64, 30, True)])
def test_linear(rnn, orc, rows, fin, fout, bias):
    rng = orc.Rng(21)
    x, w = rng.rand_vec(rows * fin), rng.rand_vec(fout * fin) * np.float32(0.02)
    b = rng.rand_vec(fout) if bias else None
    dy = rng.rand_vec(rows * fout)
    dw0, db0 = rng.rand_vec(fout * fin), (rng.rand_vec(fout) if bias else None)
    with orc.threads(8):
        y_want = orc.linear_forward(rows, fin, fout, x, w, b)
        dw_want, db_want, dx_want = orc.linear_backward(rows, fin, fout, dy, x, w, dw0, db0)
    y = rnn.linear_forward(rows, fin, fout, to_dev(x), to_dev(w), to_dev(b) if bias else None)
    assert rel_frob(to_host(y), y_want) < TOL
    dw = to_dev(dw0.copy())
    db = to_dev(db0.copy()) if bias else None
    dx = rnn.linear_backward(rows, fin, fout, to_dev(dy), to_dev(x), to_dev(w), dw, db)
    assert rel_frob(to_host(dw), dw_want) < TOL
    assert rel_frob(to_host(dx), dx_want) < TOL
    if bias:
        assert rel_frob(to_host(db), db_want) < TOL


@pytest.mark.parametrize("rows,fin,fout", [(8192, 256, 768), (100, 64, 30), (27, 6, 10)])
def test_linear_backward_acc(rnn, orc, rows, fin, fout):
    """rnn_linear_backward_ex with RNN_LINEAR_ACC_DX: dx0 + the dx that
    rnn_linear_backward writes, bit for bit (dW and db as the plain call's,
    bit for bit), and within TOL of the oracle."""
    rng = orc.Rng(22)
    x, w = rng.rand_vec(rows * fin), rng.rand_vec(fout * fin) * np.float32(0.02)
    dy, dx0 = rng.rand_vec(rows * fout), rng.rand_vec(rows * fin)
    X, W, DY = to_dev(x), to_dev(w), to_dev(dy)
    dw1, db1 = to_dev(np.zeros(fout * fin, np.float32)), to_dev(np.zeros(fout, np.float32))
    dx = to_host(rnn.linear_backward(rows, fin, fout, DY, X, W, dw1, db1))
    dw2, db2 = to_dev(np.zeros(fout * fin, np.float32)), to_dev(np.zeros(fout, np.float32))
    DX = to_dev(dx0.copy())
    out = rnn.linear_backward(rows, fin, fout, DY, X, W, dw2, db2, dx=DX, acc_dx=True)
    assert out is DX
    assert np.array_equal(to_host(DX), (dx0 + dx).astype(np.float32))
    assert np.array_equal(to_host(dw1), to_host(dw2)) and np.array_equal(to_host(db1), to_host(db2))
    with orc.threads(8):
        _, _, dx_want = orc.linear_backward(rows, fin, fout, dy, x, w, np.zeros(fout * fin, np.float32),
                                            np.zeros(fout, np.float32))
    assert rel_frob(to_host(DX) - dx0, dx_want) < TOL


@pytest.mark.parametrize("rows,fin,fout,rpi,masked", [(8192, 352, 256, 64, True),
                                                      (2048, 256, 384, 16, False),
                                                      (300, 40, 36, 10, True),
                                                      (96, 6, 20, 32, True)])
def test_linear_forward_residual(rnn, orc, rows, fin, fout, rpi, masked):
    """rnn_linear_forward_residual == rnn_linear_forward then
    rnn_residual_add_scaled(out, y, ...), bit for bit (rpi 10: the two-pass
    fallback; fin 6: the register-staged GEMM's epilogue), y within TOL of the
    oracle."""
    import ctypes as C
    from rustnn_amd import _ptr, lib
    rng = orc.Rng(23)
    x, w = rng.rand_vec(rows * fin), rng.rand_vec(fout * fin) * np.float32(0.05)
    b, l, out0 = rng.rand_vec(fout), rng.rand_vec(fout), rng.rand_vec(rows * fout)
    n = rows // rpi
    mask = np.where(np.arange(n) % 3 == 1, 0.0, 1.25).astype(np.float32)
    X, W, B, L = to_dev(x), to_dev(w), to_dev(b), to_dev(l)
    M = to_dev(mask) if masked else None
    y1 = rnn.linear_forward(rows, fin, fout, X, W, B)
    O1 = to_dev(out0.copy())
    ctx = rnn.default_ctx()
    ctx.check(lib().rnn_residual_add_scaled(ctx.h, rows, fout, _ptr(O1, rows * fout, "x"),
                                            _ptr(y1, rows * fout, "a"), _ptr(L, fout, "l"),
                                            _ptr(M, n, "m") if masked else None, rpi,
                                            _ptr(O1, rows * fout, "y")))
    O2 = to_dev(out0.copy())
    y2 = rnn.linear_forward_residual(rows, fin, fout, X, W, B, O2, L, M, rpi)
    assert np.array_equal(to_host(y1), to_host(y2))
    assert np.array_equal(to_host(O1), to_host(O2))
    with orc.threads(8):
        yw = orc.linear_forward(rows, fin, fout, x, w, b)
    assert rel_frob(to_host(y2), yw) < TOL


@pytest.mark.parametrize("m,k", [(32, 288), (288, 32), (7, 259), (1, 1), (13, 600)])
@pytest.mark.parametrize("tr", [False, True])
def test_pack_bit_exact(rnn, orc, m, k, tr):
    rng = orc.Rng(m * 1000 + k)
    a = rng.rand_vec(m * k)
    assert np.array_equal(to_host(rnn.dbg_pack_a(to_dev(a), m, k, tr)), orc.pack_a(a, m, k, tr))
    assert np.array_equal(to_host(rnn.dbg_pack_b(to_dev(a), m, k, tr)), orc.pack_b(a, m, k, tr))


def test_destroy_flushes_deferred_reductions(rnn, orc):
    """A context destroyed with deferral on and reductions still queued runs
    them first: the Linear backward's dW (split over rows) and bias
    gradient equal the immediate path's, bit for bit."""
    rows, fin, fout = 8192, 64, 96
    rng = orc.Rng(31)
    x, dy = to_dev(rng.rand_vec(rows * fin)), to_dev(rng.rand_vec(rows * fout))
    w = to_dev(rng.rand_vec(fout * fin))
    got = []
    for defer in (False, True):
        ctx = rnn.Context(0)
        dw = to_dev(np.zeros(fout * fin, np.float32))
        db = to_dev(np.zeros(fout, np.float32))
        ctx.set_defer(defer)
        rnn.linear_backward(rows, fin, fout, dy, x, w, dw, db, ctx=ctx)
        ctx.close()  # no flush: destroy runs what is queued
        got.append((to_host(dw), to_host(db)))
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])
    assert got[1][1].any()


# The direct-to-LDS tiles at their edges: a quad past the last whole tile, one
# short of it, the shortest k, k off a stage; 32 x 64, 64 x 64, 128 x 128 and
# 256 x 128 tiles by size.
# Then sizes that no 16-byte quad divides (one float a lane and DMA).
@pytest.mark.parametrize("m,n,k", [(4, 4, 4), (36, 68, 12), (516, 2052, 132), (2044, 2180, 1028),
                                   (16388, 1028, 36), (1, 1, 1), (33, 65, 67), (1001, 1030, 35),
                                   (70, 31, 2051)])
@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_split_tiles(rnn, m, n, k, at, bt):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn((k, m) if at else (m, k), generator=g, device="cuda")
    b = torch.randn((n, k) if bt else (k, n), generator=g, device="cuda")
    c = torch.full((m, n), 7.0, device="cuda")
    rnn.matmul(m, n, k, a, at, b, bt, c)
    want = (a.T if at else a).double() @ (b.T if bt else b).double()
    # k sums of rounded products, each rounding 2^-24 of a partial sum: as a
    # random walk 2^-24 sqrt(k) of the result, with 2^-23 for the part
    # products left out (below 2^-22 of their product each, 2^-24 in the root
    # mean square over random operands)
    assert rel_frob(to_host(c), to_host(want)) < 2.0 ** -24 * np.sqrt(k) + 2.0 ** -23


@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (512, 2048, 256), (2048, 2176, 1024),
                                   (16384, 1024, 32)])
def test_matmul_split_special_values(rnn, m, n, k):
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randint(-3, 4, (m, k), generator=g, device="cuda").float()
    b = torch.randint(-3, 4, (k, n), generator=g, device="cuda").float()
    a[5, 3], a[17, 1], b[2, 9] = float("inf"), float("nan"), float("-inf")
    a[40], a[40, 7], b[7] = 0.0, torch.finfo(torch.float32).max, 1.0
    c = torch.empty((m, n), device="cuda")
    rnn.matmul(m, n, k, a, False, b, False, c)
    # infinities and NaN land where IEEE products and sums put them, finite
    # integer results are exact, the largest float comes through whole
    want = (a.double() @ b.double()).float()
    assert np.array_equal(to_host(c), to_host(want), equal_nan=True)


@pytest.mark.parametrize("rows,fin,fout", [(35, 33, 31), (2050, 130, 67), (5, 513, 2)])
def test_linear_backward_ragged_bias(rnn, rows, fin, fout):
    """db rides in the dW product for ragged sizes too, also split over rows."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows)
    dy = torch.randn((rows, fout), generator=g, device="cuda")
    x = torch.randn((rows, fin), generator=g, device="cuda")
    w = torch.randn((fout, fin), generator=g, device="cuda")
    dw, db = torch.ones(fout * fin, device="cuda"), torch.ones(fout, device="cuda")
    dx = rnn.linear_backward(rows, fin, fout, dy, x, w, dw, db)
    # sums of at most `rows` rounded products (test_matmul_split_tiles); db in f64
    tol = lambda k: 2.0 ** -24 * np.sqrt(k) + 2.0 ** -23
    d = dy.double()
    assert rel_frob(to_host(dw) - 1, to_host(d.T @ x.double())) < 2 * tol(rows)
    assert rel_frob(to_host(db), to_host(d.sum(0) + 1)) < 2.0 ** -23
    assert rel_frob(to_host(dx), to_host(d @ w.double())) < tol(fout)


# Operands far from 1, down to denormal ones, whose lower parts have no bf16 of
# their own exponent: 32 x 64, 64 x 64, 128 x 128, 256 x 128 and ragged tiles.
@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (2048, 640, 64), (2048, 2048, 1024),
                                   (16384, 1024, 32), (65, 67, 63)])
@pytest.mark.parametrize("sa,sb", [(1e-36, 1.0), (1e-36, 1e30), (1e30, 3e-39), (1e-41, 1e30),
                                   (1e25, 1e10)])
def test_matmul_split_exponent_range(rnn, m, n, k, sa, sb):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + k)
    rnd = lambda r, c, s: (torch.randn((r, c), generator=g, device="cuda").double() * s).float()
    a, b = rnd(m, k, sa), rnd(k, n, sb)
    c = torch.empty((m, n), device="cuda")
    rnn.matmul(m, n, k, a, False, b, False, c)
    # as test_matmul_split_tiles; results from 1e24 on are fp32 products
    want = a.double() @ b.double()
    assert rel_frob(to_host(c), to_host(want)) < 2.0 ** -24 * np.sqrt(k) + 2.0 ** -22


@pytest.mark.parametrize("m,n,k", [(512, 512, 16), (512, 512, 256), (513, 515, 65), (8192, 256, 48),
                                   (2048, 2048, 1024), (16384, 1024, 64)])
def test_matmul_split_same_sign(rnn, m, n, k):
    """What the split leaves out does not add up over terms of one sign."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + k)
    a = torch.randn((m, k), generator=g, device="cuda").abs()
    b = torch.randn((k, n), generator=g, device="cuda").abs()
    c = torch.empty((m, n), device="cuda")
    rnn.matmul(m, n, k, a, False, b, False, c)
    want = a.double() @ b.double()
    # each result's error is a random walk of sqrt(k) roundings, their mean over
    # rows and columns that share operands at most its 1/sqrt(min(m, n)) part
    tol = 2.0 ** -24 * np.sqrt(k) / np.sqrt(min(m, n)) + 2.0 ** -27
    assert abs(((c.double() - want) / want).mean().item()) < tol
    # a mantissa whose parts below the leading one are as large as they get
    x = 1.0 + 2.0 ** -7 - 2.0 ** -23
    a.fill_(x)
    b.fill_(x)
    rnn.matmul(m, n, k, a, False, b, False, c)
    assert rel_frob(to_host(c), np.full((m, n), k * x * x)) < 2.0 ** -22


# Short k: one product is rounded once, and sums of a few are no further off
# than a chain of fp32 roundings.
@pytest.mark.parametrize("m,n", [(4, 4), (64, 68), (8192, 256), (4096, 4096), (1, 3), (511, 513)])
@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("k", [1, 2, 4, 5])
def test_matmul_short_k(rnn, m, n, k, at, bt):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn((k, m) if at else (m, k), generator=g, device="cuda")
    b = torch.randn((n, k) if bt else (k, n), generator=g, device="cuda")
    c = torch.full((m, n), 7.0, device="cuda")
    rnn.matmul(m, n, k, a, at, b, bt, c)
    want = (a.T if at else a).double() @ (b.T if bt else b).double()
    if k == 1:
        assert torch.equal(c, want.float())
    elif m * n > 256:
        # rounding j of k is 2^-24 / sqrt(3) of a partial sum of j of the k terms
        # at most, 0.7 of that where mantissas are spread over a binade
        tol = 2.0 ** -24 / np.sqrt(3) * np.sqrt((k + 1) / 2)
        assert ((c.double() - want).norm() / want.norm()).item() < tol


# Both sides of the lines between the tiles: fp32 and split ones at k = 4 / 8
# and, with up to 256 tiles, 24 / 28; tiles without shares up to k = 64, or 128;
# 32 x 64 and 64 x 64 ones at 256 and 272 tiles; ragged sizes at k = 12 / 13.
# With infinities and a NaN.
@pytest.mark.parametrize("m,n,k", [(1024, 1088, 4), (1024, 1088, 8), (512, 512, 24), (512, 512, 28),
                                   (1024, 1020, 128), (1024, 1020, 132), (1024, 1088, 64),
                                   (1024, 1088, 68), (255, 257, 12), (255, 257, 13),
                                   (2047, 1029, 131)])
@pytest.mark.parametrize("at,bt", [(False, False), (False, True), (True, False)])
def test_matmul_tile_lines(rnn, m, n, k, at, bt):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-3, 4, (k, m) if at else (m, k), generator=g, device="cuda").float()
    b = torch.randint(-3, 4, (n, k) if bt else (k, n), generator=g, device="cuda").float()
    c = torch.empty((m, n), device="cuda")
    for special in (False, True):
        if special:
            av, bv = a.T if at else a, b.T if bt else b
            av[5, 3], av[m - 1, k - 1] = float("inf"), float("nan")
            bv[2, 9], bv[k - 1, n - 2] = float("-inf"), float("inf")
        rnn.matmul(m, n, k, a, at, b, bt, c)
        want = ((a.T if at else a).double() @ (b.T if bt else b).double()).float()
        assert np.array_equal(to_host(c), to_host(want), equal_nan=True)


@pytest.mark.parametrize("rows,fin,fout", [(1, 32, 64), (3, 33, 31), (48, 33, 31), (49, 33, 31),
                                           (64, 64, 128)])
def test_linear_backward_few_rows(rnn, rows, fin, fout):
    """dW and db of a short batch, with db beside dW and in a sum of its own."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(rows + fin)
    dy = torch.randint(-3, 4, (rows, fout), generator=g, device="cuda").float()
    x = torch.randint(-3, 4, (rows, fin), generator=g, device="cuda").float()
    w = torch.randint(-3, 4, (fout, fin), generator=g, device="cuda").float()
    dw, db = torch.ones(fout * fin, device="cuda"), torch.ones(fout, device="cuda")
    dx = rnn.linear_backward(rows, fin, fout, dy, x, w, dw, db)
    assert torch.equal(dw.view(fout, fin), dy.T.contiguous() @ x + 1)
    assert torch.equal(db, dy.sum(0) + 1)
    assert torch.equal(dx.view(rows, fin), dy @ w)


_REGISTER_KERNEL = """
import sys
import torch
import rustnn_amd as R
worst = 0.0
for m, n, k in ((64, 64, 64), (132, 68, 36), (2176, 2176, 48), (1, 1, 1), (33, 65, 67),
                (2177, 2177, 31), (70, 31, 2051)):
    for at in (False, True):
        for bt in (False, True):
            g = torch.Generator(device="cuda").manual_seed(m + n + k)
            a = torch.randint(-3, 4, (k, m) if at else (m, k), generator=g, device="cuda").float()
            b = torch.randint(-3, 4, (n, k) if bt else (k, n), generator=g, device="cuda").float()
            want = ((a.T if at else a).double() @ (b.T if bt else b).double()).float()
            for acc in (False, True):
                c = torch.full((m, n), 7.0, device="cuda")
                R.matmul(m, n, k, a, at, b, bt, c, acc)
                assert torch.equal(c, want + 7.0 if acc else want), (m, n, k, at, bt, acc)
for rows, fin, fout in ((64, 32, 48), (35, 33, 31), (2050, 130, 67)):
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, w, dy = (torch.randint(-3, 4, sh, generator=g, device="cuda").float()
                for sh in ((rows, fin), (fout, fin), (rows, fout)))
    bias = torch.arange(fout, device="cuda").float()
    y = R.linear_forward(rows, fin, fout, x, w, bias)
    assert torch.equal(y.view(rows, fout), x @ w.T.contiguous() + bias)
    dw, db = torch.ones(fout * fin, device="cuda"), torch.ones(fout, device="cuda")
    dx = R.linear_backward(rows, fin, fout, dy, x, w, dw, db)
    assert torch.equal(dx.view(rows, fin), dy @ w) and torch.equal(db, dy.sum(0) + 1)
    assert torch.equal(dw.view(fout, fin), dy.T.contiguous() @ x + 1)
print("register kernel ok", flush=True)
"""


def test_register_staged_kernel():
    """gemm_kernel, which operands of 2 GiB and more take, at every tile,
    layout and alignment: a process in which no product takes the other one."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", _REGISTER_KERNEL], cwd=root, capture_output=True,
                       text=True, timeout=100, env=dict(os.environ, RNN_GEMM_NODMA="1"))
    assert r.returncode == 0 and "register kernel ok" in r.stdout, r.stderr[-2000:]
