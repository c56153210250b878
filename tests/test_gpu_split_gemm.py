"""The split-f16 Q4 GEMM (k_q4_gemm and the kernels around it) at the sizes
where its tiles end: row blocks of 16, row tiles of up to 80, the rows where
the K runs change, half chunks of 64 rows of K, K segments of 256, partial
column tiles, widths that leave stores unaligned.

Each element is held to its own bound against 64 bits.  A staged value is
within 2^-22 of the f32 it stands for (hi + lo, and lo lo dropped) plus 2^-39
of the largest of its row's 256 columns (lo's subnormal step), and an element
is at most 24 accumulations a segment (8 chunks of 32, three products) plus
one per segment, each rounded to f32: |error| <= 2 (2^-22 + (24 + segments)
2^-24) sum_k |x_k w_k| + sum over segments 2^-39 max |x| sum_k |w_k|, the
factor 2 for the sums inside one matrix instruction.
"""
import numpy as np
import pytest

import qtts
from qtts import synth
from test_zz_no_alloc import DevBuf, hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(ctx_factory):
    return ctx_factory(256)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def check(Y, X, w):
    W, X = w.dequant().astype(np.float64), X.astype(np.float64)
    bound = 2 * (2.0 ** -22 + (24 + -(-w.k // 256)) * 2.0 ** -24) * (np.abs(X) @ np.abs(W))
    for k in range(0, w.k, 256):
        bound += 2.0 ** -39 * np.abs(X[:, k:k + 256]).max(axis=1)[:, None] * np.abs(W[k:k + 256]).sum(axis=0)
    err = np.abs(Y.astype(np.float64) - X @ W)
    assert (err <= bound).all(), f"largest error {np.max(err / np.maximum(bound, 1e-300)):.3g} of its bound"


@pytest.mark.parametrize("k,n", [(64, 32), (96, 160), (256, 96), (288, 1500), (2048, 128), (2080, 1000), (6144, 64)])
def test_rows_and_shapes(ctx, k, n):
    rng = np.random.Generator(np.random.PCG64(k + n))
    w = synth.q4_random(rng, k, n)
    dw = ctx.upload(w)
    X = rng.standard_normal((225, k)).astype(np.float32)
    X *= np.exp2(rng.integers(-20, 20, (225, 1))).astype(np.float32)   # every row has its own range
    whole = ctx.gemm(dw, X, path="mfma")
    check(whole, X, w)
    assert not whole[:, n // 32 * 32:].any()
    for rows in (1, 2, 15, 16, 17, 31, 33, 48, 63, 64, 65, 80, 81, 96, 97, 161):
        print(f"k={k} n={n} rows={rows}", flush=True)
        Y = ctx.gemm(dw, X[:rows], path="mfma")
        assert np.array_equal(bits(Y), bits(whole[:rows])), f"{rows} rows: not the bits of the same rows among 225"
    dw.free()


@pytest.mark.parametrize("k,n,rows", [(6144, 2048, 450), (2048, 12288, 600), (6144, 64, 2900)])
def test_rows_in_batches(ctx, k, n, rows):
    """More rows than run one workgroup per K segment, and more (2900 x 6144)
    than the workspaces hold at once: the same bits as in batches of 100, with
    and without the call's own allocations."""
    rng = np.random.Generator(np.random.PCG64(rows))
    w = synth.q4_random(rng, k, n)
    dw = ctx.upload(w)
    X = rng.standard_normal((rows, k)).astype(np.float32)
    whole = ctx.gemm(dw, X, path="mfma")
    at = [0, 15, rows // 2, rows - 17, rows - 1]
    check(whole[at], X[at], w)
    for r0 in range(0, rows, 100):
        assert np.array_equal(bits(ctx.gemm(dw, X[r0:r0 + 100], path="mfma")), bits(whole[r0:r0 + 100]))
    h = hip()
    dx, dy = DevBuf(h, X.nbytes), DevBuf(h, whole.nbytes)
    dx.put(X)
    ctx.gemm_noalloc(dw, dx.ptr.value, rows, dy.ptr.value, path="mfma")
    ctx.sync()
    assert np.array_equal(bits(dy.get(whole.shape)), bits(whole))
    dx.free()
    dy.free()
    dw.free()


@pytest.mark.parametrize("rows", [5, 200])
def test_small_values_beside_an_outlier(ctx, rows):
    """A segment of 256 columns 2^30 times the others, with zero weights: the
    others keep their bits (each segment has its own factor)."""
    rng = np.random.Generator(np.random.PCG64(81))
    w = synth.q4_random(rng, 1024, 96)
    w.packed[256:512] = 0x88                      # nibbles of 8: zero
    X = rng.standard_normal((rows, 1024)).astype(np.float32)
    X[:, 256:512] *= np.float32(2.0 ** 30)
    dw = ctx.upload(w)
    check(ctx.gemm(dw, X), X, w)
    dw.free()


def test_zero_and_not_finite_rows(ctx):
    """A zero row gives zeros; an inf or NaN stays in its own row."""
    rng = np.random.Generator(np.random.PCG64(9))
    w = synth.q4_random(rng, 512, 96)
    dw = ctx.upload(w)
    X = rng.standard_normal((40, 512)).astype(np.float32)
    ref = ctx.gemm(dw, X, path="mfma")
    X[3], X[5, 7], X[21, 300] = 0.0, np.inf, np.nan
    Y = ctx.gemm(dw, X, path="mfma")
    keep = [i for i in range(40) if i not in (3, 5, 21)]
    assert np.array_equal(bits(Y[keep]), bits(ref[keep]))
    assert not Y[3].any() and not np.isfinite(Y[5]).any() and not np.isfinite(Y[21]).any()
    dw.free()


def test_noalloc_refusal_does_not_depend_on_the_path(ctx_factory, monkeypatch):
    """16 slices of 128 rows (tile G8_T128) x 33,792 columns: GEMV partial sums
    beyond the workspace.  Refused at any few rows, also those that the matrix
    cores take by themselves; asked for, the matrix cores run."""
    monkeypatch.setenv("QTTS_TILE_GEMV", "1")
    c = ctx_factory(256)
    rng = np.random.Generator(np.random.PCG64(78))
    dw = c.upload(synth.q4_random(rng, 2048, 33792))
    x = rng.standard_normal((16, 2048)).astype(np.float32)
    h = hip()
    dx, dy = DevBuf(h, x.nbytes), DevBuf(h, 16 * 33792 * 4)
    try:
        dx.put(x)
        for rows in (1, 3, 15):
            with pytest.raises(qtts.QttsError) as e:
                c.gemm_noalloc(dw, dx.ptr.value, rows, dy.ptr.value)
            assert e.value.code == qtts.ERR_CAPACITY
        for rows, path in ((3, "mfma"), (16, None)):
            c.gemm_noalloc(dw, dx.ptr.value, rows, dy.ptr.value, path=path)
            c.sync()
            assert np.array_equal(bits(dy.get((rows, 33792))), bits(c.gemm(dw, x[:rows], path="mfma")))
    finally:
        dx.free()
        dy.free()
        dw.free()


def test_weight_uploaded_behind_queued_work(ctx_factory):
    """An uploaded weight is complete on return: uploaded by a context that
    still has GEMMs queued on its stream, used at once by another one."""
    a, b = ctx_factory(256), ctx_factory(256)
    rng = np.random.Generator(np.random.PCG64(80))
    w0, w = synth.q4_random(rng, 6144, 2048), synth.q4_random(rng, 2048, 1024)
    d0 = a.upload(w0)
    h = hip()
    rows = 2000
    dx, dy = DevBuf(h, rows * 6144 * 4), DevBuf(h, rows * 2048 * 4)
    X = rng.standard_normal((20, 2048)).astype(np.float32)
    try:
        dx.put(np.zeros((rows, 6144), np.float32))
        for _ in range(50):
            a.gemm_noalloc(d0, dx.ptr.value, rows, dy.ptr.value)
        dw = a.upload(w)
        check(b.gemm(dw, X, path="mfma"), X, w)
        a.sync()
        dw.free()
    finally:
        dx.free()
        dy.free()
        d0.free()


@pytest.mark.parametrize("rows", [1000, 1022, 1023, 1040])
def test_host_arrays_around_the_staging_buffer(ctx, rows):
    """Host rows of 0.25 MB and results of 16 MB, which fill the 16 MiB
    staging buffer to within a slot, and more than it holds: the bits of the
    call on device memory."""
    rng = np.random.Generator(np.random.PCG64(82))
    w = synth.q4_random(rng, 64, 4032)
    X = rng.standard_normal((rows, 64)).astype(np.float32)
    dw = ctx.upload(w)
    h = hip()
    dx, dy = DevBuf(h, X.nbytes), DevBuf(h, rows * 4032 * 4)
    dx.put(X)
    ctx.gemm_noalloc(dw, dx.ptr.value, rows, dy.ptr.value)
    ctx.sync()
    for _ in range(2):
        assert np.array_equal(bits(ctx.gemm(dw, X)), bits(dy.get((rows, 4032))))
        assert ctx.debug_query("staging") == 0
    dx.free()
    dy.free()
    dw.free()
