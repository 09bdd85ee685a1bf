"""Matrix products on the GPU against the CPU oracle: the reference's cases
(tests/test_mlu.py:238-300) and configs 4 and 5a of the benchmark at full
size.

Bars (north_star): float32 products within 2e-3 and bfloat16 / float16
products (float32 accumulation) within 1e-2, both as max |got - want| /
max |want| against the float64 product of the same stored inputs.  Full-size
products are checked on 4096 sampled entries computed exactly by the oracle
and, over the whole matrix, with Freivalds' test C x = A (B x) in float64.
"""

import numpy as np
import pytest

from _check import BF16, F16, F32

pytestmark = pytest.mark.gpu

DTYPES = [F32, BF16, F16]
BAR = {F32: 2e-3, BF16: 1e-2, F16: 1e-2}


def sample(orc, shape, dtype, seed, scale=1.0):
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32) * np.float32(scale)
    return orc.from_float(x, dtype)


def rel_err(orc, got, want, dtype):
    g = orc.to_float(got, dtype)
    w = orc.to_float(want, dtype) if want.dtype != np.float64 else want
    return float(np.max(np.abs(g - w)) / max(np.max(np.abs(w)), 1e-30))


def check(orc, got, want, dtype, what):
    e = rel_err(orc, got, want, dtype)
    assert e <= BAR[dtype], f"{what}: relative error {e:.3g} > {BAR[dtype]}"
    return e


def exact(orc, a, b, dtype, ta=False, tb=False):
    """float64 product of the stored operands (op = transpose when t*)."""
    A = orc.to_float(a, dtype)
    B = orc.to_float(b, dtype)
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    return A @ B


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,k,n", [(37, 19, 23), (128, 64, 96), (200, 72, 136), (256, 256, 256),
                                   (64, 520, 24), (8, 16, 8)])
def test_mm_transposes(dev, ops, orc, dtype, ta, tb, m, k, n):
    a = sample(orc, (k, m) if ta else (m, k), dtype, 1)
    b = sample(orc, (n, k) if tb else (k, n), dtype, 3)
    da = dev.from_numpy(a, dtype=dtype)
    db = dev.from_numpy(b, dtype=dtype)
    got = ops.mm(da.t() if ta else da, db.t() if tb else db).numpy()
    want = orc.gemm(dtype, a, b, ta, tb)
    assert got.shape == (m, n)
    check(orc, got, want, dtype, f"mm ta={ta} tb={tb}")
    check(orc, got, exact(orc, a, b, dtype, ta, tb), dtype, "mm vs float64")


@pytest.mark.parametrize("dtype", DTYPES)
def test_addmm_bmm_matmul(dev, ops, orc, dtype):
    bias, a, b = sample(orc, (23,), dtype, 0), sample(orc, (37, 19), dtype, 1), sample(orc, (19, 23), dtype, 2)
    d = lambda x: dev.from_numpy(x, dtype=dtype)  # noqa: E731
    got = ops.addmm(d(bias), d(a), d(b), beta=0.5, alpha=2.0).numpy()
    check(orc, got, orc.gemm(dtype, a, b, alpha=2.0, beta=0.5, cin=bias), dtype, "addmm")
    want64 = 0.5 * orc.to_float(bias, dtype) + 2.0 * exact(orc, a, b, dtype)
    check(orc, got, want64, dtype, "addmm vs float64")
    x, y = sample(orc, (4, 9, 6), dtype, 4), sample(orc, (4, 6, 5), dtype, 5)
    check(orc, ops.bmm(d(x), d(y)).numpy(), orc.gemm(dtype, x, y), dtype, "bmm")
    w = sample(orc, (6, 5), dtype, 6)
    got = ops.matmul(d(x), d(w)).numpy()
    assert got.shape == (4, 9, 5)
    check(orc, got, exact(orc, x, w, dtype), dtype, "matmul 3d @ 2d")
    v = sample(orc, (2, 1, 6, 3), dtype, 7)
    got = ops.matmul(d(x), d(v)).numpy()
    assert got.shape == (2, 4, 9, 3)
    check(orc, got, exact(orc, x, v, dtype), dtype, "matmul broadcast batch")
    u = sample(orc, (6,), dtype, 8)
    got = ops.matmul(d(x), d(u)).numpy()
    assert got.shape == (4, 9)
    check(orc, got, exact(orc, x, u, dtype), dtype, "matmul 3d @ 1d")
    got = ops.matmul(d(u), d(w)).numpy()
    assert got.shape == (5,)
    check(orc, got, exact(orc, u, w, dtype), dtype, "matmul 1d @ 2d")


@pytest.mark.parametrize("dtype", DTYPES)
def test_linear(dev, ops, orc, dtype):
    x, w, b = sample(orc, (3, 5, 64), dtype, 0), sample(orc, (48, 64), dtype, 1), sample(orc, (48,), dtype, 2)
    d = lambda t: dev.from_numpy(t, dtype=dtype)  # noqa: E731
    want = exact(orc, x, w, dtype, tb=True)
    got = ops.linear(d(x), d(w), d(b)).numpy()
    assert got.shape == (3, 5, 48)
    check(orc, got, want + orc.to_float(b, dtype), dtype, "linear with bias")
    check(orc, ops.linear(d(x), d(w)).numpy(), want, dtype, "linear")
    got = ops.linear(d(x)[0, 0], d(w), d(b)).numpy()
    assert got.shape == (48,)
    check(orc, got, want[0, 0] + orc.to_float(b, dtype), dtype, "linear 1-d input")


@pytest.mark.parametrize("dtype", DTYPES)
def test_bmm_shapes(dev, ops, orc, dtype):
    for (bt, m, k, n) in ((32, 512, 64, 512), (1, 256, 4096, 1024), (3, 1, 7, 5)):
        a = sample(orc, (bt, m, k), dtype, 1, k ** -0.5)
        b = sample(orc, (bt, k, n), dtype, 2)
        got = ops.bmm(dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)).numpy()
        check(orc, got, exact(orc, a, b, dtype), dtype, f"bmm {bt}x{m}x{k}x{n}")
    a, b = sample(orc, (4, 9, 6), dtype, 3), sample(orc, (4, 5, 6), dtype, 4)
    got = ops.bmm(dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype).transpose(1, 2)).numpy()
    check(orc, got, exact(orc, a, b, dtype, tb=True), dtype, "bmm transposed operand")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,k,n", [(2, 1024, 1024), (128, 1024, 256), (256, 4096, 1024),
                                   (1024, 4096, 128)])
def test_mm_shapes(dev, ops, orc, dtype, m, k, n):
    a, b = sample(orc, (m, k), dtype, 1), sample(orc, (k, n), dtype, 2)
    got = ops.mm(dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)).numpy()
    check(orc, got, exact(orc, a, b, dtype), dtype, f"mm {m}x{k}x{n}")


def test_k_zero_and_empty(dev, ops, orc):
    a = dev.from_numpy(np.zeros((4, 0), np.float32))
    b = dev.from_numpy(np.zeros((0, 3), np.float32))
    assert np.array_equal(ops.mm(a, b).numpy(), np.zeros((4, 3), np.float32))
    bias = dev.from_numpy(np.arange(3, dtype=np.float32))
    got = ops.addmm(bias, a, b, beta=2.0).numpy()
    assert np.array_equal(got, np.broadcast_to(np.arange(3, dtype=np.float32) * 2, (4, 3)))


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16", "fp16"])
def test_product_planner_layouts(dev, ops, orc, dtype):
    """Layouts the product planner reads where they lie, or copies, with NaN
    in every stored element outside the views (a read outside the view
    shows up as NaN in the result)."""
    d = lambda t: dev.from_numpy(t, dtype=dtype)  # noqa: E731
    f = lambda t: orc.to_float(t, dtype)  # noqa: E731

    def no_nan(got, what):
        assert not np.isnan(f(got)).any(), f"{what}: read outside the view"

    # mm on column slices: leading dimensions wider than the rows.
    a = _padded(orc, (70, 40), 9, dtype, 1)
    b = _padded(orc, (40, 33), 7, dtype, 2)
    got = ops.mm(d(a)[:, :40], d(b)[:, :33]).numpy()
    no_nan(got, "mm column slices")
    check(orc, got, f(a)[:, :40] @ f(b)[:, :33], dtype, "mm column slices")
    # bmm over every other matrix of a stack (batch stride 2 m k).
    x = sample(orc, (8, 16, 24), dtype, 3)
    y = sample(orc, (8, 24, 12), dtype, 4)
    got = ops.bmm(d(x)[::2], d(y)[1::2]).numpy()
    check(orc, got, f(x)[::2] @ f(y)[1::2], dtype, "bmm strided batch")
    # [B, M, K] stored as transposes against a shared [K, N]: the batch does
    # not fold into the rows, the shared side is read with batch stride 0.
    xt = sample(orc, (5, 24, 16), dtype, 5)
    w = _padded(orc, (24, 20), 4, dtype, 6)
    got = ops.matmul(d(xt).transpose(1, 2), d(w)[:, :20]).numpy()
    assert got.shape == (5, 16, 20)
    no_nan(got, "matmul unfoldable batch")
    check(orc, got, np.swapaxes(f(xt), 1, 2) @ f(w)[:, :20], dtype, "matmul unfoldable batch")
    # [1, M, K] against [B, K, N] (left side shared), and [K] against [B, K, N].
    l1 = sample(orc, (1, 16, 24), dtype, 7)
    got = ops.matmul(d(l1), d(y)).numpy()
    assert got.shape == (8, 16, 12)
    check(orc, got, f(l1) @ f(y), dtype, "matmul shared left side")
    v = sample(orc, (24,), dtype, 8)
    got = ops.matmul(d(v), d(y)).numpy()
    assert got.shape == (8, 12)
    check(orc, got, f(v) @ f(y), dtype, "matmul vector @ stack")
    # Batch axes that do not merge into one stride ([2, 3] from a permuted
    # [3, 2] stack): copied dense first.
    s = sample(orc, (3, 2, 16, 24), dtype, 9)
    got = ops.matmul(d(s).permute(1, 0, 2, 3), d(y)[:6].view(2, 3, 24, 12)).numpy()
    want = np.swapaxes(f(s), 0, 1) @ f(y)[:6].reshape(2, 3, 24, 12)
    check(orc, got, want, dtype, "matmul unmergeable batch")
    # linear on a permuted 3-D input with bias, and with an input whose rows
    # are a column slice.
    xin = sample(orc, (6, 4, 32), dtype, 10)
    wt = sample(orc, (10, 32), dtype, 11)
    bias = sample(orc, (10,), dtype, 12)
    got = ops.linear(d(xin).permute(1, 0, 2), d(wt), d(bias)).numpy()
    assert got.shape == (4, 6, 10)
    want = np.swapaxes(f(xin), 0, 1) @ f(wt).T + f(bias)
    check(orc, got, want, dtype, "linear permuted input")
    xs = _padded(orc, (12, 32), 6, dtype, 13)
    got = ops.linear(d(xs)[:, :32], d(wt), d(bias)).numpy()
    no_nan(got, "linear column-slice input")
    check(orc, got, f(xs)[:, :32] @ f(wt).T + f(bias), dtype, "linear column-slice input")


def test_planner_empty_sums(dev, ops, orc):
    """An inner size of 0 gives zeros, or beta * bias; linear keeps the
    input's rows; addmm with beta = 0 never reads (or shape-checks) the
    bias."""
    z = lambda *s: dev.from_numpy(np.zeros(s, np.float32))  # noqa: E731
    bias = np.array([1.0, -2.0, 3.0], np.float32)
    got = ops.linear(z(4, 0), z(3, 0), dev.from_numpy(bias)).numpy()
    assert np.array_equal(got, np.broadcast_to(bias, (4, 3)))
    assert np.array_equal(ops.linear(z(2, 5, 0), z(3, 0)).numpy(), np.zeros((2, 5, 3), np.float32))
    assert np.array_equal(ops.matmul(z(2, 4, 0), z(0, 3)).numpy(), np.zeros((2, 4, 3), np.float32))
    a = np.random.default_rng(0).standard_normal((4, 6)).astype(np.float32)
    b = np.random.default_rng(1).standard_normal((6, 3)).astype(np.float32)
    odd_bias = dev.from_numpy(np.full((7,), np.nan, np.float32))
    got = ops.addmm(odd_bias, dev.from_numpy(a), dev.from_numpy(b), beta=0.0, alpha=2.0).numpy()
    check(orc, got, 2.0 * (a.astype(np.float64) @ b), F32, "addmm beta 0")


# ---- full-size configs ------------------------------------------------------------


def sampled_entries(orc, got, a, b, dtype, ta=False, tb=False, alpha=1.0, beta=0.0, cin=None,
                    count=4096, seed=0):
    m, n = got.shape[-2:]
    g = np.random.default_rng(seed)
    idx = np.stack([np.zeros(count, np.int64), g.integers(0, m, count), g.integers(0, n, count)], 1)
    want = orc.gemm_entries(dtype, a, b, idx, ta, tb, alpha, beta, cin)
    have = orc.to_float(got, dtype)[idx[:, 1], idx[:, 2]]
    return float(np.max(np.abs(have - want)) / np.max(np.abs(want)))


def freivalds(orc, got, a, b, dtype, ta=False, tb=False, bias=None):
    """max |C x - A (B x)| relative to max |A (B x)|, in float64."""
    x = np.random.default_rng(7).standard_normal(got.shape[-1])
    A = orc.to_float(a, dtype)
    B = orc.to_float(b, dtype)
    A = A.T if ta else A
    B = B.T if tb else B
    ref = A @ (B @ x)
    if bias is not None:
        ref = ref + float(orc.to_float(bias, dtype) @ x)
    lhs = orc.to_float(got, dtype) @ x
    return float(np.max(np.abs(lhs - ref)) / np.max(np.abs(ref)))


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
def test_config4_mm_4096(dev, ops, orc, dtype):
    K = 4096
    a = sample(orc, (K, K), dtype, 1, K ** -0.25)
    b = sample(orc, (K, K), dtype, 2, K ** -0.25)
    da, db = dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)
    got = ops.mm(da, db).numpy()
    assert sampled_entries(orc, got, a, b, dtype) <= BAR[dtype]
    assert freivalds(orc, got, a, b, dtype) <= BAR[dtype]
    # A stored [K, M] and read in place through .t()
    at = np.ascontiguousarray(a.T)
    got_t = ops.mm(dev.from_numpy(at, dtype=dtype).t(), db).numpy()
    assert sampled_entries(orc, got_t, at, b, dtype, ta=True) <= BAR[dtype]
    # addmm with a [4096] bias
    bias = sample(orc, (K,), dtype, 3)
    got_b = ops.addmm(dev.from_numpy(bias, dtype=dtype), da, db).numpy()
    assert sampled_entries(orc, got_b, a, b, dtype, beta=1.0, cin=bias) <= BAR[dtype]


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
def test_config4_linear(dev, ops, orc, dtype):
    x = sample(orc, (8192, 4096), dtype, 1, 4096 ** -0.25)
    w = sample(orc, (11008, 4096), dtype, 2, 4096 ** -0.25)
    b = sample(orc, (11008,), dtype, 3)
    got = ops.linear(dev.from_numpy(x, dtype=dtype), dev.from_numpy(w, dtype=dtype),
                     dev.from_numpy(b, dtype=dtype)).numpy()
    assert got.shape == (8192, 11008)
    assert sampled_entries(orc, got, x, w, dtype, tb=True, beta=1.0, cin=b) <= BAR[dtype]
    assert freivalds(orc, got, x, w, dtype, tb=True, bias=b) <= BAR[dtype]


def test_config5_bmm_bf16(dev, ops, orc):
    a = sample(orc, (64, 512, 128), BF16, 1, 128 ** -0.25)
    b = sample(orc, (64, 128, 512), BF16, 2, 128 ** -0.25)
    got = ops.bmm(dev.from_numpy(a, dtype=BF16), dev.from_numpy(b, dtype=BF16)).numpy()
    check(orc, got, exact(orc, a, b, BF16), BF16, "bmm 64x512x128x512")


# ---- the 256 x 256 four-wave kernel through the kernel C-ABI ---------------------


def _padded(orc, shape, pad, dtype, seed):
    """Random values of ``shape`` stored with ``pad`` extra NaN columns: the
    array returned is the storage, the view of its first columns the
    operand.  A kernel that reads the padding produces NaNs."""
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32) * np.float32(0.25)
    store = np.full(shape[:-1] + (shape[-1] + pad,), np.nan, np.float32)
    store[..., :shape[-1]] = x
    return orc.from_float(store, dtype)


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("bt,m,n,k", [(256, 256, 256, 256), (256, 256, 256, 384), (64, 512, 512, 320)],
                         ids=["big-tiles", "big-tiles-6-steps", "K-tail-fallback"])
def test_gemm_abi_padded_batched(amd, dev, orc, dtype, ta, tb, bt, m, n, k):
    """tp_amd_launch_gemm on a batch of products with padded leading
    dimensions (NaN padding), alpha = 0.5 and beta = 2 with a full Cin.  The
    first two shapes have one 256 x 256 tile per CU and four or six K tiles
    (the four-wave kernel: its loads of A for the K tile after next go out
    after each step's barrier, so the step pairs, the last two steps and
    the prologue all issue differently); the third, K = 320, is not a
    multiple of 128 and takes the eight-wave kernel."""
    lib = amd.load()
    pad, alpha, beta = 8, 0.5, 2.0
    a = _padded(orc, (bt, k, m) if ta else (bt, m, k), pad, dtype, 1)
    b = _padded(orc, (bt, n, k) if tb else (bt, k, n), pad, dtype, 2)
    cin = sample(orc, (bt, m, n), dtype, 3)
    lda, ldb = a.shape[-1], b.shape[-1]
    da, db, dc = (dev.from_numpy(x, dtype=dtype) for x in (a, b, cin))
    out = dev.empty((bt, m, n), dtype=dtype)
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, alpha, da.data_ptr, lda, a.shape[-2] * lda,
                                int(ta), db.data_ptr, ldb, b.shape[-2] * ldb, int(tb), beta,
                                dc.data_ptr, n, 1, m * n, out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    A = orc.to_float(a, dtype)[..., :(m if ta else k)]
    B = orc.to_float(b, dtype)[..., :(k if tb else n)]
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    want = alpha * np.matmul(A, B) + beta * orc.to_float(cin, dtype)
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "padding leaked into the product"
    check(orc, got, want, dtype, f"gemm abi {bt}x{m}x{n}x{k} ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("bt,m,n,k,pad,bcast", [(1, 515, 517, 509, 3, False), (1, 520, 512, 512, 3, False),
                                                (4, 300, 270, 255, 5, True)],
                         ids=["odd-K", "odd-ld", "odd-K-batch-broadcast"])
def test_gemm_abi_repacked_operands(amd, dev, orc, dtype, ta, tb, bt, m, n, k, pad, bcast):
    """Operands that are not whole packets (odd K, odd leading dimensions, NaN
    in the padding), read where they lie at these sizes: alpha = 0.5, beta =
    2 with a full Cin, and in the batched case a B broadcast over the batch
    (stride 0)."""
    lib = amd.load()
    alpha, beta = 0.5, 2.0
    a = _padded(orc, (bt, k, m) if ta else (bt, m, k), pad, dtype, 1)
    b = _padded(orc, (1 if bcast else bt, n, k) if tb else (1 if bcast else bt, k, n), pad, dtype, 2)
    cin = sample(orc, (bt, m, n), dtype, 3)
    lda, ldb = a.shape[-1], b.shape[-1]
    da, db, dc = (dev.from_numpy(x, dtype=dtype) for x in (a, b, cin))
    out = dev.empty((bt, m, n), dtype=dtype)
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, alpha, da.data_ptr, lda, a.shape[-2] * lda,
                                int(ta), db.data_ptr, ldb, 0 if bcast else b.shape[-2] * ldb, int(tb),
                                beta, dc.data_ptr, n, 1, m * n, out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    A = orc.to_float(a, dtype)[..., :(m if ta else k)]
    B = orc.to_float(b, dtype)[..., :(k if tb else n)]
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    want = alpha * np.matmul(A, B) + beta * orc.to_float(cin, dtype)
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "padding leaked into the product"
    check(orc, got, want, dtype, f"gemm abi {bt}x{m}x{n}x{k} ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)], ids=["NN", "TT"])
def test_gemm_abi_odd_k_in_place_mn_major(amd, dev, orc, dtype, ta, tb):
    """An odd K with one operand stored M/N-contiguous and aligned: only the
    K-major operand is copied (zero-padded to whole packets), the other is
    read in place up to row K -- its storage has NaN rows right after row
    K, which must never reach the product."""
    lib = amd.load()
    bt, m, n, k, alpha, beta = 2, 264, 256, 509, 0.5, 2.0  # M, N and their lds whole packets
    g = np.random.default_rng(5)
    # the K-major operand: ordinary storage, ld = K
    km = g.standard_normal((bt, n, k) if tb else (bt, m, k)).astype(np.float32) * np.float32(0.25)
    km = orc.from_float(km, dtype)
    # the MN-major operand: [K + 5, MN + 8] per batch, NaN past row K and column MN
    mn_len = m if ta else n
    store = np.full((bt, k + 5, mn_len + 8), np.nan, np.float32)
    store[:, :k, :mn_len] = g.standard_normal((bt, k, mn_len)).astype(np.float32) * np.float32(0.25)
    mnm = orc.from_float(store, dtype)
    cin = sample(orc, (bt, m, n), dtype, 3)
    d_km, d_mn, dc = (dev.from_numpy(x, dtype=dtype) for x in (km, mnm, cin))
    out = dev.empty((bt, m, n), dtype=dtype)
    ld_mn, sb_mn = mn_len + 8, (k + 5) * (mn_len + 8)
    if ta:   # A stored [K, M] (M contiguous) in place, B stored [N, K] (K-major)
        args = (d_mn.data_ptr, ld_mn, sb_mn, 1, d_km.data_ptr, k, n * k, 1)
    else:    # A stored [M, K] (K-major), B stored [K, N] (N contiguous) in place
        args = (d_km.data_ptr, k, m * k, 0, d_mn.data_ptr, ld_mn, sb_mn, 0)
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, alpha, *args, beta, dc.data_ptr, n, 1, m * n,
                                out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    K = orc.to_float(km, dtype)
    Mv = orc.to_float(mnm, dtype)[:, :k, :mn_len]
    A = np.swapaxes(Mv, 1, 2) if ta else K
    B = np.swapaxes(K, 1, 2) if tb else Mv
    want = alpha * np.matmul(A, B) + beta * orc.to_float(cin, dtype)
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "rows past K leaked into the product"
    check(orc, got, want, dtype, f"odd K in place ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
def test_mm_skinny_odd_k(dev, ops, orc, dtype):
    """dX = dY W for a one-row dY and a vocabulary-sized odd K (W stored
    [K, N], N contiguous): read in place, checked against the float64
    product."""
    dy = sample(orc, (1, 3001), dtype, 21)
    w = sample(orc, (3001, 256), dtype, 22, 3001 ** -0.5)
    got = ops.mm(dev.from_numpy(dy, dtype=dtype), dev.from_numpy(w, dtype=dtype)).numpy()
    check(orc, got, exact(orc, dy, w, dtype), dtype, "skinny odd K")


@pytest.mark.parametrize("m,n,k,pad", [(1664, 1408, 520, 0), (1701, 1300, 776, 1)], ids=["aligned", "odd-M-ldc"])
def test_fp32_nn_as_transposed_product(amd, dev, ops, orc, m, n, k, pad):
    """float32 A [M, K] @ B [K, N] with enough tiles to fill the GPU runs as
    C^T = B^T A^T with C written transposed: ragged M and N, addmm's bias,
    a full Cin with beta = 2 through the kernel ABI into a C whose rows are
    ldc = N + pad apart (pad 1: rows not 16-byte aligned, element stores;
    the pad column must stay untouched), and a batch of two."""
    lib = amd.load()
    a, b = sample(orc, (m, k), F32, 31, k ** -0.5), sample(orc, (k, n), F32, 32)
    da, db = dev.from_numpy(a), dev.from_numpy(b)
    want = a.astype(np.float64) @ b.astype(np.float64)
    check(orc, ops.mm(da, db).numpy(), want, F32, "mm")
    bias = sample(orc, (n,), F32, 33)
    check(orc, ops.addmm(dev.from_numpy(bias), da, db, beta=0.5, alpha=2.0).numpy(),
          2.0 * want + 0.5 * bias.astype(np.float64), F32, "addmm")
    cin = sample(orc, (m, n), F32, 34)
    ldc = n + pad
    out = dev.from_numpy(np.full((m, ldc), 7.0, np.float32))
    st = lib.tp_amd_launch_gemm(0, F32, 1, m, n, k, 0.5, da.data_ptr, k, 0, 0, db.data_ptr, n, 0, 0, 2.0,
                                dev.from_numpy(cin).data_ptr, n, 1, 0, out.data_ptr, ldc, 0)
    assert st == 0, lib.tp_mlu_last_error()
    got = out.numpy()
    assert np.all(got[:, n:] == 7.0), "the pad column was written"
    check(orc, np.ascontiguousarray(got[:, :n]), 0.5 * want + 2.0 * cin.astype(np.float64), F32, "full Cin")
    x, y = sample(orc, (2, m, k), F32, 35, k ** -0.5), sample(orc, (2, k, n), F32, 36)
    check(orc, ops.bmm(dev.from_numpy(x), dev.from_numpy(y)).numpy(),
          np.matmul(x.astype(np.float64), y.astype(np.float64)), F32, "bmm")


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
def test_mm_2047_cube(dev, ops, orc, dtype):
    """mm 2047^3 (odd everything) through ops.mm, checked on sampled
    entries and with Freivalds' test."""
    a = sample(orc, (2047, 2047), dtype, 11, 0.05)
    b = sample(orc, (2047, 2047), dtype, 12, 0.05)
    got = ops.mm(dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)).numpy()
    assert sampled_entries(orc, got, a, b, dtype) <= BAR[dtype]
    assert freivalds(orc, got, a, b, dtype) <= BAR[dtype]


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("cin_kind", ["full", "bias-row"])
def test_gemm_fp32_split_k(amd, dev, orc, ta, tb, cin_kind):
    """A float32 product with few 128 x 128 tiles and a long K (256 x 384
    outputs, K = 4096: 6 tiles) is split over K into float32 partials that are
    added in slice order: the result matches the float64 product at the fp32
    bar with alpha = 0.5, beta = 2 and a full Cin or a row-broadcast bias,
    NaN-padded leading dimensions, and two runs give the same bits."""
    lib = amd.load()
    m, n, k, pad, alpha, beta = 256, 384, 4096, 4, 0.5, 2.0
    a = _padded(orc, (k, m) if ta else (m, k), pad, F32, 7)
    b = _padded(orc, (n, k) if tb else (k, n), pad, F32, 8)
    if cin_kind == "full":
        cin = sample(orc, (m, n), F32, 9)
        rs, cs = n, 1
        cin_f = cin
    else:
        cin = sample(orc, (n,), F32, 9)
        rs, cs = 0, 1
        cin_f = np.broadcast_to(cin, (m, n))
    da, db, dc = dev.from_numpy(a), dev.from_numpy(b), dev.from_numpy(cin)
    A = a[:, :m] if ta else a[:, :k]
    B = b[:, :k] if tb else b[:, :n]
    A = A.T if ta else A
    B = B.T if tb else B
    want = alpha * (A.astype(np.float64) @ B.astype(np.float64)) + beta * cin_f.astype(np.float64)
    outs = []
    for _ in range(2):
        out = dev.empty((m, n), dtype=F32)
        st = lib.tp_amd_launch_gemm(0, F32, 1, m, n, k, alpha, da.data_ptr, a.shape[-1], 0, int(ta),
                                    db.data_ptr, b.shape[-1], 0, int(tb), beta, dc.data_ptr, rs, cs, 0,
                                    out.data_ptr, n, 0)
        assert st == 0, lib.tp_mlu_last_error()
        outs.append(out.numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32)), "split-K sum is not deterministic"
    check(orc, outs[0], want, F32, f"split-K fp32 ta={ta} tb={tb} {cin_kind}")


# One size for each tile shape and split the planner picks on 256 CUs, with
# ragged edges: M and N a few elements past or short of whole tiles, K with a
# partial last slab (16-bit slabs are 64 deep, float32 ones 32) and K shorter
# than one.  (m, n, k); an M/N-major operand needs its extent in packets.
TILE16 = [(2056, 2200, 72), (1496, 1512, 200), (1112, 1000, 264), (712, 136, 8), (3000, 2904, 40),
          (200, 304, 4104), (1208, 1000, 5000), (1496, 1512, 4104), (40, 8200, 1032), (200, 328, 24),
          (136, 264, 49160), (1128, 624, 4104), (200, 3000, 9000), (1200, 1104, 9000)]
TILE32 = [(2052, 2044, 36), (1500, 1504, 100), (712, 132, 4), (300, 304, 4004), (20, 8204, 2052),
          (44, 4100, 4108), (1500, 1504, 2100), (132, 60, 28), (132, 140, 40004), (24, 4100, 1028), (36, 8204, 260),
          (4100, 24, 4100), (36, 196, 516)]


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("dtype,m,n,k", [(BF16 if i % 2 else F16, *t) for i, t in enumerate(TILE16)]
                         + [(F32, *t) for t in TILE32], ids=lambda v: str(v))
def test_gemm_tiles_with_ragged_edges(amd, dev, orc, dtype, ta, tb, m, n, k):
    """Every tile shape and split in the four layouts: NaN-padded leading
    dimensions (a load past an edge that reached the product would show),
    alpha and a row-broadcast bias, sampled columns against float64, and the
    same bits twice."""
    lib = amd.load()
    pad, alpha, beta = 8, 0.5, 2.0
    a = _padded(orc, (k, m) if ta else (m, k), pad, dtype, 61)
    b = _padded(orc, (n, k) if tb else (k, n), pad, dtype, 62)
    bias = sample(orc, (n,), dtype, 63)
    A = orc.to_float(a, dtype)[:, :(m if ta else k)]
    B = orc.to_float(b, dtype)[:, :(k if tb else n)]
    A = A.T if ta else A
    B = B.T if tb else B
    da, db, dbias = (dev.from_numpy(v, dtype=dtype) for v in (a, b, bias))
    outs = []
    for _ in range(2):
        out = dev.empty((m, n), dtype=dtype)
        st = lib.tp_amd_launch_gemm(0, dtype, 1, m, n, k, alpha, da.data_ptr, a.shape[-1], 0, int(ta),
                                    db.data_ptr, b.shape[-1], 0, int(tb), beta, dbias.data_ptr, 0, 1, 0,
                                    out.data_ptr, n, 0)
        assert st == 0, lib.tp_mlu_last_error()
        outs.append(out.numpy())
    assert np.array_equal(outs[0], outs[1]), "two runs differ"
    got = orc.to_float(outs[0], dtype)
    assert not np.isnan(got).any(), "an edge leaked into the product"
    rng = np.random.default_rng(64)
    cols = np.unique(np.concatenate([np.arange(min(n, 8)), np.arange(max(0, n - 70), n), rng.integers(0, n, 40)]))
    want = alpha * (A.astype(np.float64) @ B[:, cols].astype(np.float64)) + beta * orc.to_float(bias, dtype)[cols]
    check(orc, np.ascontiguousarray(outs[0][:, cols]), want, dtype, f"{m}x{n}x{k} ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("bt,m,n,k", [(9, 1000, 64, 200), (70, 72, 136, 40), (33, 320, 80, 328), (5, 40, 48, 4104)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)], ids=["NN", "TT"])
def test_gemm_tiles_batched(amd, dev, orc, dtype, bt, m, n, k, ta, tb):
    """Batches of attention-sized products on the tile kernel, few columns
    among them, each batch with its own full Cin."""
    lib = amd.load()
    a = _padded(orc, (bt, k, m) if ta else (bt, m, k), 8, dtype, 65)
    b = _padded(orc, (bt, n, k) if tb else (bt, k, n), 8, dtype, 66)
    cin = sample(orc, (bt, m, n), dtype, 67)
    A = orc.to_float(a, dtype)[..., :(m if ta else k)].astype(np.float64)
    B = orc.to_float(b, dtype)[..., :(k if tb else n)].astype(np.float64)
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    want = 0.5 * np.matmul(A, B) + 2.0 * orc.to_float(cin, dtype)
    da, db, dc = (dev.from_numpy(v, dtype=dtype) for v in (a, b, cin))
    out = dev.empty((bt, m, n), dtype=dtype)
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, 0.5, da.data_ptr, a.shape[-1], a.shape[-1] * a.shape[-2],
                                int(ta), db.data_ptr, b.shape[-1], b.shape[-1] * b.shape[-2], int(tb), 2.0,
                                dc.data_ptr, n, 1, m * n, out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "an edge leaked into the product"
    for i in (0, bt // 2, bt - 1):
        check(orc, got[i], want[i], dtype, f"batch {i} of {bt}x{m}x{n}x{k} ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("cin_kind", ["none", "full", "bias-row"])
@pytest.mark.parametrize("k", [4096, 4000, 3001])
def test_gemm16_split_k(amd, dev, orc, dtype, ta, tb, cin_kind, k):
    """A 16-bit product with few 128 x 128 tiles and a long K (200 x 384
    outputs: 6 tiles) is split over K into float32 partials, added in slice
    order and rounded once: within the 16-bit bar of the float64 product
    with alpha = 0.5 and beta = 2 (a full Cin or a row-broadcast bias),
    NaN-padded leading dimensions, a ragged M, and two runs giving the same
    bits.  K = 4096 splits into four slices of 1024; K = 4000 into three of
    1024 and a last of 928; K = 3001 (odd: K-major operands are copied with
    zero padding first, M/N-major ones read in place) into 1536 and 1465."""
    lib = amd.load()
    m, n, pad, alpha = 200, 384, 8, 0.5
    a = _padded(orc, (k, m) if ta else (m, k), pad, dtype, 17)
    b = _padded(orc, (n, k) if tb else (k, n), pad, dtype, 18)
    A = orc.to_float(a, dtype).astype(np.float64)
    B = orc.to_float(b, dtype).astype(np.float64)
    A = A[:, :m].T if ta else A[:, :k]
    B = B[:, :k].T if tb else B[:, :n]
    want = alpha * (A @ B)
    if cin_kind == "none":
        beta, cin, rs, cs = 0.0, None, 0, 0
    elif cin_kind == "full":
        beta, cin, rs, cs = 2.0, sample(orc, (m, n), dtype, 19), n, 1
        want = want + beta * orc.to_float(cin, dtype)
    else:
        beta, cin, rs, cs = 2.0, sample(orc, (n,), dtype, 19), 0, 1
        want = want + beta * orc.to_float(cin, dtype)
    da, db = dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)
    dc = dev.from_numpy(cin, dtype=dtype) if cin is not None else None
    outs = []
    for _ in range(2):
        out = dev.empty((m, n), dtype=dtype)
        st = lib.tp_amd_launch_gemm(0, dtype, 1, m, n, k, alpha, da.data_ptr, a.shape[-1], 0, int(ta),
                                    db.data_ptr, b.shape[-1], 0, int(tb), beta,
                                    dc.data_ptr if dc is not None else 0, rs, cs, 0, out.data_ptr, n, 0)
        assert st == 0, lib.tp_mlu_last_error()
        outs.append(out.numpy())
    assert np.array_equal(outs[0], outs[1]), "split-K sum is not deterministic"
    assert not np.isnan(orc.to_float(outs[0], dtype)).any(), "padding leaked into the product"
    check(orc, outs[0], want, dtype, f"16-bit split-K k={k} ta={ta} tb={tb} {cin_kind}")


@pytest.mark.parametrize("dtype", [BF16, F16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("k", [64, 128])
@pytest.mark.parametrize("cin_kind", ["none", "bias-row", "full"])
@pytest.mark.parametrize("bt,m,n", [(64, 512, 512), (257, 256, 256)], ids=["xcd-order", "plain-order"])
def test_gemm_abi_small_k(amd, dev, orc, dtype, ta, tb, k, cin_kind, bt, m, n):
    """Batched 16-bit products with K = 64 or 128 (attention-sized: the
    one-barrier kernel that holds all of K in LDS) through
    tp_amd_launch_gemm: NaN-padded leading dimensions, the four layouts,
    alpha = 0.5 and beta = 0 / a per-column bias shared by the batch / a full
    Cin with beta = 2.  64 x 512 x 512 has 256 tiles (numbered so each batch
    stays on one XCD); 257 x 256 x 256 has a tile count that is not a
    multiple of 8 and is numbered in order."""
    lib = amd.load()
    pad, alpha = 8, 0.5
    a = _padded(orc, (bt, k, m) if ta else (bt, m, k), pad, dtype, 11)
    b = _padded(orc, (bt, n, k) if tb else (bt, k, n), pad, dtype, 12)
    lda, ldb = a.shape[-1], b.shape[-1]
    da, db = dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)
    A = orc.to_float(a, dtype)[..., :(m if ta else k)]
    B = orc.to_float(b, dtype)[..., :(k if tb else n)]
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    want = alpha * np.matmul(A, B)
    if cin_kind == "none":
        beta, cin, rs, cs, sb = 0.0, None, 0, 0, 0
    elif cin_kind == "bias-row":
        beta, cin, rs, cs, sb = 1.0, sample(orc, (n,), dtype, 13), 0, 1, 0
        want = want + orc.to_float(cin, dtype)
    else:
        beta, cin, rs, cs, sb = 2.0, sample(orc, (bt, m, n), dtype, 13), n, 1, m * n
        want = want + beta * orc.to_float(cin, dtype)
    dc = dev.from_numpy(cin, dtype=dtype) if cin is not None else None
    cptr = dc.data_ptr if dc is not None else 0
    out = dev.empty((bt, m, n), dtype=dtype)
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, alpha, da.data_ptr, lda, a.shape[-2] * lda,
                                int(ta), db.data_ptr, ldb, b.shape[-2] * ldb, int(tb), beta,
                                cptr, rs, cs, sb, out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "padding leaked into the product"
    check(orc, got, want, dtype, f"small-K gemm {bt}x{m}x{n}x{k} ta={ta} tb={tb} {cin_kind}")


def _embedded(orc, shape, ld, lead, dtype, seed):
    """A matrix (or batch of them) with rows ``ld`` apart that starts ``lead``
    elements into its storage and ends with it; NaN in the gaps.  Returns the
    storage and the matrix."""
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32) * np.float32(0.25)
    rows, cols = int(np.prod(shape[:-1])), shape[-1]
    flat = np.full(lead + (rows - 1) * ld + cols, np.nan, np.float32)
    np.lib.stride_tricks.as_strided(flat[lead:], (rows, cols), (4 * ld, 4))[:] = x.reshape(rows, cols)
    x = orc.to_float(orc.from_float(x, dtype), dtype)
    return orc.from_float(flat, dtype), x


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("bt,m,n,k,pad,lead", [
    (1, 129, 67, 64, 0, 1), (1, 65, 127, 65, 1, 1), (1, 66, 131, 71, 0, 0), (1, 97, 33, 1, 1, 1), (1, 35, 70, 129, 3, 1),
    (3, 63, 65, 193, 0, 1), (1, 257, 255, 4099, 0, 1), (1, 2601, 2603, 2602, 1, 1)],
    ids=["whole-K-tile", "one-past", "odd-K", "K-1", "two-tiles-and-one", "batch", "split", "copies"])
def test_gemm_operands_at_any_element(amd, dev, orc, dtype, ta, tb, bt, m, n, k, pad, lead):
    """Operands that start, end and step at odd elements, with NaN around
    them, are read in place (the largest 16-bit one through aligned copies),
    up to the last element and no further."""
    lib = amd.load()
    lda, ldb = (m if ta else k) + pad, (n if tb is False else k) + pad
    a, A = _embedded(orc, (bt, k, m) if ta else (bt, m, k), lda, lead, dtype, 21)
    b, B = _embedded(orc, (bt, n, k) if tb else (bt, k, n), ldb, lead, dtype, 22)
    da, db = dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype)
    out = dev.empty((bt, m, n), dtype=dtype)
    e = 4 if dtype == F32 else 2
    st = lib.tp_amd_launch_gemm(0, dtype, bt, m, n, k, 1.0, da.data_ptr + lead * e, lda, (k if ta else m) * lda, int(ta),
                                db.data_ptr + lead * e, ldb, (n if tb else k) * ldb, int(tb), 0.0, 0, 0, 0, 0,
                                out.data_ptr, n, m * n)
    assert st == 0, lib.tp_mlu_last_error()
    A = np.swapaxes(A, -1, -2) if ta else A
    B = np.swapaxes(B, -1, -2) if tb else B
    rows = np.r_[0:2, 61:67, m - 3:m] if m > 1000 else np.arange(m)
    rows = rows[rows < m]
    want = np.matmul(A[:, rows].astype(np.float64), B.astype(np.float64))
    got = out.numpy()[:, rows]
    assert not np.isnan(orc.to_float(got, dtype)).any(), "an element outside the operands reached the product"
    check(orc, got, want, dtype, f"odd gemm {bt}x{m}x{n}x{k} ta={ta} tb={tb}")


def _spread(dev, ops, orc, shape, ld, lead, dtype, seed):
    """A device matrix whose rows lie ``ld`` elements apart, ``lead`` elements
    into its storage, with NaN in the gaps; and its values."""
    x = sample(orc, shape, dtype, seed, 0.25)
    store = dev.empty((lead + (shape[0] - 1) * ld + shape[1],), dtype=dtype)
    ops.fill_(store, float("nan"))
    rows = store._view(shape, (ld, 1), lead)
    ops.copy_(rows, dev.from_numpy(x, dtype=dtype))
    return store, rows, orc.to_float(x, dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("m,n,k,odd", [(130, 66, 136, 0), (67, 129, 71, 1)], ids=["even", "odd"])
def test_gemm_rows_far_apart(amd, dev, ops, orc, dtype, ta, tb, m, n, k, odd):
    """Operands whose rows are too far apart for one 4 GiB buffer resource a
    panel (from 2^23 elements for rows of K, 2^25 for rows of M or N), with
    odd ends and a row longer than 512 MiB among them; alpha, and a bias."""
    lib = amd.load()
    e = 4 if dtype == F32 else 2
    k_apart, mn_apart = (1 << 23) + 8 + odd, (1 << 25) + 8 + odd
    if ta == tb:  # one of them past 2^29 bytes
        mn_apart = max(mn_apart, (1 << 29) // e + 8 + odd) if e == 2 else mn_apart
    lda, ldb = mn_apart if ta else k_apart, k_apart if tb else mn_apart
    sa, da, A = _spread(dev, ops, orc, (k, m) if ta else (m, k), lda, odd, dtype, 71)
    sb, db, B = _spread(dev, ops, orc, (n, k) if tb else (k, n), ldb, odd, dtype, 72)
    bias = sample(orc, (n,), dtype, 73)
    dbias = dev.from_numpy(bias, dtype=dtype)
    out = dev.empty((m, n), dtype=dtype)
    st = lib.tp_amd_launch_gemm(0, dtype, 1, m, n, k, 0.5, da.data_ptr, lda, 0, int(ta), db.data_ptr, ldb, 0, int(tb),
                                2.0, dbias.data_ptr, 0, 1, 0, out.data_ptr, n, 0)
    assert st == 0, lib.tp_mlu_last_error()
    got = out.numpy()
    assert not np.isnan(orc.to_float(got, dtype)).any(), "a gap reached the product"
    want = 0.5 * ((A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64))
    check(orc, got, want + 2.0 * orc.to_float(bias, dtype), dtype, f"far gemm {m}x{n}x{k} ta={ta} tb={tb}")


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False)], ids=["NT", "NN", "TN"])
def test_gemm_of_a_very_long_k(amd, dev, ops, orc, dtype, ta, tb):
    """K past 2^23, where rows of K leave the reach of one resource: operands
    of -1, 0 and 1 with a period of 1000 in K make every sum an integer under
    2^24, so the product is exact in any order."""
    m, n, period, reps, tail = 70, 66, 1000, 8400, 37
    k = period * reps + tail
    g = np.random.default_rng(74)
    a0, b0 = (g.integers(-1, 2, (rows, period)).astype(np.float32) for rows in (m, n))

    def build(x0, kmajor):
        x0 = orc.from_float(x0, dtype)
        rows = x0.shape[0]
        x = dev.empty((rows, k) if kmajor else (k, rows), dtype=dtype)
        step = 1 if kmajor else rows
        src = dev.from_numpy(x0, dtype=dtype)
        ops.copy_(x._view((rows, reps, period), (k if kmajor else 1, period * step, step)),
                  src._view((rows, reps, period), (period, 0, 1)))
        ops.copy_(x._view((rows, tail), (k if kmajor else 1, step), period * reps * step),
                  src._view((rows, tail), (period, 1)))
        return x if kmajor else x.t()

    got = ops.mm(build(a0, not ta), build(b0, tb).t()).numpy()
    want = reps * (a0 @ b0.T) + a0[:, :tail] @ b0[:, :tail].T
    assert np.abs(want).max() < 2**24
    assert np.array_equal(got, orc.from_float(want.astype(np.float32), dtype))


def test_gemm_without_room_for_scratch(amd, dev, orc):
    """With the device's memory taken up to a few MiB, products that would be
    cut into slices of K or copied to aligned rows run without: the same
    results to rounding, no error."""
    lib = amd.load()
    # 28 MB of slices (16-bit), 35 MB of slices (float32), 27 MB of copies
    cases = []
    for dtype, m, n, k in ((BF16, 776, 3000, 11000), (F32, 1500, 1500, 4000), (BF16, 2601, 2603, 2602)):
        a, b = sample(orc, (m, k), dtype, 81, 0.25), sample(orc, (n, k), dtype, 82, 0.25)
        da, db, out = dev.from_numpy(a, dtype=dtype), dev.from_numpy(b, dtype=dtype), dev.empty((m, n), dtype=dtype)
        cases.append((dtype, m, n, k, da, db, out))

    def run():
        for dtype, m, n, k, da, db, out in cases:
            st = lib.tp_amd_launch_gemm(0, dtype, 1, m, n, k, 1.0, da.data_ptr, k, 0, 0, db.data_ptr, k, 0, 1, 0.0, 0, 0,
                                        0, 0, out.data_ptr, n, 0)
            assert st == 0, lib.tp_mlu_last_error()
        return [orc.to_float(out.numpy(), dtype) for dtype, *_, out in cases]

    want = run()
    lib.tp_mlu_empty_cache()
    held, size = [], 1 << 36
    while size >= 8 << 20:
        try:
            held.append(dev.empty((size,), dtype="uint8"))
        except RuntimeError:
            size //= 2
    try:
        got = run()
    finally:
        held.clear()
        lib.tp_mlu_empty_cache()
    for (dtype, m, n, k, *_), g, w in zip(cases, got, want):
        assert np.linalg.norm(g - w) <= (1e-5 if dtype == F32 else 4e-3) * np.linalg.norm(w), (m, n, k)
    assert any(not np.array_equal(g, w) for g, w in zip(got, want)), "the slices' memory was there"


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("m,n,k,cin_kind", [(4096, 4096, 1024, "none"), (4090, 4081, 1001, "full"),
                                            (4090, 4081, 1001, "bias-row"), (2047, 4000, 4100, "full"),
                                            (4096, 1000, 7000, "none")],
                         ids=["whole-tiles", "ragged-full", "ragged-bias", "ragged-long", "wide-long"])
def test_large_float32_product(amd, dev, orc, ta, tb, m, n, k, cin_kind):
    """Large float32 products in the four layouts.  Rows across the edges of
    tiles against float64: the error stays under that of a sum rounded term
    by term, 2^-24 sqrt(k) of the rows' norm."""
    lib = amd.load()
    rng = np.random.default_rng(31)
    lead = 1 if k % 2 else 0
    lda, ldb = (m if ta else k) + lead, (k if tb else n) + lead
    a, A = _embedded(orc, (k, m) if ta else (m, k), lda, lead, F32, 32)
    b, B = _embedded(orc, (n, k) if tb else (k, n), ldb, lead, F32, 33)
    scale = rng.uniform(0.5, 2.0, n).astype(np.float32)
    da, db = dev.from_numpy(a, dtype=F32), dev.from_numpy(b, dtype=F32)
    cin, rs, cs, beta = {"none": (None, 0, 0, 0.0), "full": (rng.standard_normal((m, n)).astype(np.float32), n, 1, 2.0),
                         "bias-row": (scale, 0, 1, -1.0)}[cin_kind]
    dc = dev.from_numpy(cin, dtype=F32) if cin is not None else None
    out = dev.empty((m, n), dtype=F32)
    st = lib.tp_amd_launch_gemm(0, F32, 1, m, n, k, 0.5, da.data_ptr + 4 * lead, lda, 0, int(ta), db.data_ptr + 4 * lead,
                                ldb, 0, int(tb), beta, dc.data_ptr if dc is not None else 0, rs, cs, 0, out.data_ptr, n, 0)
    assert st == 0, lib.tp_mlu_last_error()
    rows = np.r_[0, 127, 255, 256, 1792, m - 2, m - 1]
    want = 0.5 * (np.asarray(A.T if ta else A)[rows].astype(np.float64) @ np.asarray(B.T if tb else B).astype(np.float64))
    if cin is not None:
        want += beta * (cin[rows] if rs else cin).astype(np.float64)
    got = out.numpy()[rows].astype(np.float64)
    assert np.isfinite(got).all()
    error = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert error.max() <= 2.0**-24 * np.sqrt(k), error


@pytest.mark.parametrize("m,n,k", [(4096, 4096, 1024), (2048, 4096, 4096), (256, 1024, 4096), (40, 8200, 2048)])
@pytest.mark.parametrize("small", [1.0, 2.0**-60], ids=["ones", "2^-120"])
def test_float32_product_of_one_term_is_rounded_once(dev, ops, m, n, k, small):
    """A row with one non-zero element (a diagonal, selected or masked
    operand) makes each result one product of two float32 numbers, exact in
    float64: the result is that product rounded once, whatever the kernel
    and the slices of K, also for products down to 2^-121."""
    g = np.random.default_rng(35)
    at = g.integers(0, k, m)
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), at] = (g.uniform(0.5, 1.5, m) * small).astype(np.float32)
    b = (g.uniform(0.5, 1.5, (k, n)) * g.choice([-small, small], (k, n))).astype(np.float32)
    got = ops.mm(dev.from_numpy(a), dev.from_numpy(b)).numpy()
    want = (a[np.arange(m), at].astype(np.float64)[:, None] * b[at].astype(np.float64)).astype(np.float32)
    assert np.array_equal(got, want), f"{np.mean(got != want):.1%} of the results are not the rounded product"


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38, 1e-36, 1e-42])
def test_large_float32_product_with_extreme_values(dev, ops, value):
    """Infinities and NaN land where IEEE arithmetic puts them, and a row of
    very large, very small or subnormal values keeps its precision."""
    m, n, k = 4096, 4096, 1024
    rng = np.random.default_rng(34)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = (rng.standard_normal((k, n)) * 0.25).astype(np.float32)
    if abs(value) < 1:
        a[300] *= np.float32(value)
    else:
        a[300, 17] = value
    b[17, 40] = 0.0
    got = ops.mm(dev.from_numpy(a), dev.from_numpy(b)).numpy()[[0, 300, m - 1]]
    with np.errstate(invalid="ignore", over="ignore"):
        want = a[[0, 300, m - 1]].astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    big = ~np.isfinite(want) | (np.abs(want) > 3.4e38)
    assert np.array_equal(np.isinf(got), big & ~np.isnan(want))
    for g, w in zip(got, want):
        ok = np.isfinite(g) & np.isfinite(w)
        # 1e-42 leaves a float32 few bits: half a step of 2^-149 a rounding
        bar = 2.0**-24 * np.sqrt(k) * np.linalg.norm(w[ok]) + 2.0**-150 * k * np.sqrt(n)
        assert np.linalg.norm(g[ok].astype(np.float64) - w[ok]) <= bar


@pytest.mark.parametrize("m,n,k,dtype", [(64, 64, 64, F32), (512, 512, 512, F32), (512, 512, 512, BF16),
                                         (4096, 4096, 256, BF16), (1024, 1024, 1024, F32)],
                         ids=["fma-fp32", "mfma-fp32", "mfma-bf16", "big-bf16", "mfma-fp32-1024"])
def test_nan_and_inf_propagate(dev, ops, orc, m, n, k, dtype):
    """NaN and infinities in the operands reach the same entries of C as
    in IEEE arithmetic: a NaN fills its row (or column), an infinity fills
    its row except where it meets a 0 (NaN) -- on the FMA kernel, the MFMA
    kernels and the big bf16 kernel."""
    rng = np.random.default_rng(k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    a[3, 5], a[7, 9], b[9, 11] = np.nan, np.inf, 0.0
    a[20, :] = 0.0
    a[20, 30] = -np.inf
    b[40, 50] = np.nan
    A, B = orc.from_float(a, dtype), orc.from_float(b, dtype)
    got = orc.to_float(ops.mm(dev.from_numpy(A, dtype=dtype), dev.from_numpy(B, dtype=dtype)).numpy(), dtype)
    with np.errstate(invalid="ignore", over="ignore"):
        want = orc.to_float(A, dtype) @ orc.to_float(B, dtype)
    assert np.array_equal(np.isnan(got), np.isnan(want)), "NaN in other places"
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf), "infinities in other places"
    assert np.array_equal(got[inf], want[inf]), "signs of the infinities"

