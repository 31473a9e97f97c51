"""Batched DMMV (zh_dmmv_batched, zh_dmmv_fused_gate_up_swiglu_batched: the
skinny GEMM of recordBatchDispatchPush, dmmv.zig:880-925) through the C ABI.

Every column of a batched launch must equal the one-vector DMMV of that
column bit for bit (the weights are shared, the per-column arithmetic is the
one-vector kernel's), except where the one-vector path sums in another order:
Q4_K with K = 2048 / 4096 (the streaming kernel's half-super-block partial
sums), odd row counts (the team kernel), Q6_K at 56 and 64 super-blocks and
the LM head's height (the lane-per-block kernel). There the columns agree to
the f32 summation floor (2^-20 of sum |w x|). Every column meets the oracle
bar of the one-vector kernels: |gpu - ref| <= 1e-4 + 1e-3 |ref| (+ the f32
dot-product noise floor of test_gpu_kernels.assert_dot_close). Column counts
cover the matrix-unit launches of 1 to 4 groups of 4 vectors (Q6_K past 12 in
two), the tile launches of 2 and 4 and the one-vector launch."""
import numpy as np
import pytest

from test_gpu_kernels import assert_dot_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import zinc_amd
    c = zinc_amd.Context(0)
    yield c
    c.close()


def _ring(qt, K):
    """The one-vector path is the streaming kernel (zh_dmmv_ring.hip)."""
    return qt == 12 and K in (2048, 4096)


def _same(got, ref, mag, ring):
    if not ring:
        return np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    return bool(np.all(np.abs(got.astype(np.float64) - ref) <= 2.0 ** -20 * mag + 1e-30))


def _single(ctx, qt, Wb, x, M, K, y0=None):
    xb = ctx.upload(x)
    yb = ctx.upload(y0 if y0 is not None else np.zeros(M, np.float32))
    ctx.dmmv(qt, Wb, 0, xb, 0, yb, 0, M, K, 1 if y0 is not None else 0)
    out = yb.download(np.float32, M)
    ctx.free(xb)
    ctx.free(yb)
    return out


@pytest.mark.parametrize("qt,M,K", [(12, 4096, 4096), (12, 6144, 4096), (12, 1000, 768), (12, 512, 12288),
                                    (14, 4096, 12288), (14, 1024, 4096), (14, 300, 2048)])
@pytest.mark.parametrize("ncol", [1, 2, 3, 4, 5, 8])
def test_batched_equals_single_columns(ctx, orc, qt, M, K, ncol):
    print(f"batched q{qt} {M}x{K} cols {ncol}", flush=True)
    W = orc.synth_tensor(qt | 0x100 if qt == 12 else qt, M, K, 61 + ncol, 1)
    X = np.stack([orc.synth_normal_f32(K, 61, 10 + v) for v in range(ncol)])
    Wb, Xb, Yb = ctx.upload(W), ctx.upload(X), ctx.alloc(4 * M * ncol)
    ctx.dmmv_batched(qt, Wb, 0, Xb, 0, Yb, 0, M, K, ncol)
    Y = Yb.download(np.float32, M * ncol).reshape(ncol, M)
    ring = _ring(qt, K)
    mags = [orc.dmmv_absdot(W, qt, X[v], M, K) for v in range(ncol)] if ring else [None] * ncol
    for v in range(ncol):
        ref = _single(ctx, qt, Wb, X[v], M, K)
        assert _same(Y[v], ref, mags[v], ring), (v, np.abs(Y[v] - ref).max())
    # and the oracle bar on the first and last columns
    for v in {0, ncol - 1}:
        assert_dot_close(Y[v], orc.dmmv(W, qt, X[v], M, K), orc.dmmv_f64(W, qt, X[v], M, K),
                         orc.dmmv_absdot(W, qt, X[v], M, K), f"batched col {v}")
    # acc_mode 1: Y[v] += W X[v]
    Y0 = np.stack([orc.synth_normal_f32(M, 62, v) for v in range(ncol)])
    Yb.upload(Y0)
    ctx.dmmv_batched(qt, Wb, 0, Xb, 0, Yb, 0, M, K, ncol, 1)
    Y1 = Yb.download(np.float32, M * ncol).reshape(ncol, M)
    for v in range(ncol):
        ref = _single(ctx, qt, Wb, X[v], M, K, Y0[v])
        assert _same(Y1[v], ref, mags[v] + np.abs(Y0[v]) if ring else None, ring), v
    for b in (Wb, Xb, Yb):
        ctx.free(b)


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,nb,ncol", [(1, 1, 2), (15, 2, 4), (17, 3, 16), (129, 2, 5), (70, 5, 9), (33, 9, 12),
                                       (300, 15, 13), (4100, 17, 2), (50, 33, 16), (31, 49, 8), (16, 64, 3),
                                       (40, 65, 2),
                                       # every width class and group count with an even row count
                                       (2, 1, 3), (16, 2, 2), (18, 3, 12), (130, 5, 16), (34, 9, 12), (30, 31, 9),
                                       (32, 49, 8), (46, 63, 5), (48, 8, 9), (30, 16, 12), (34, 24, 13), (50, 48, 16)])
def test_batched_edges_equal_single_columns(ctx, orc, qt, M, nb, ncol):
    """Row counts off the 16-row tiles, K of 1 to 65 super-blocks (partial
    slabs of 16; past 64 one vector at a time), rows that start 2-byte aligned
    (odd Q6_K widths), every group count of 4 vectors: each column equals its
    one-vector DMMV (to the summation floor where that runs the streaming
    kernel, the team kernel of odd row counts, or the lane-per-block kernel
    of Q6_K at 56 and 64 super-blocks, which sum in another order)."""
    K = 256 * nb
    print(f"batched edges q{qt} {M}x{K} cols {ncol}", flush=True)
    W = orc.synth_tensor(qt | 0x100 if qt == 12 else qt, M, K, 91 + ncol, 1)
    X = np.stack([orc.synth_normal_f32(K, 92, 10 + v) for v in range(ncol)])
    Wb, Xb, Yb = ctx.upload(W), ctx.upload(X), ctx.alloc(4 * M * ncol)
    loose = _ring(qt, K) or (qt == 14 and nb in (56, 64)) or M % 2 == 1
    ctx.dmmv_batched(qt, Wb, 0, Xb, 0, Yb, 0, M, K, ncol)
    Y = Yb.download(np.float32, M * ncol).reshape(ncol, M)
    for v in range(ncol):
        ref = _single(ctx, qt, Wb, X[v], M, K)
        mag = orc.dmmv_absdot(W, qt, X[v], M, K) if loose else None
        assert _same(Y[v], ref, mag, loose), (v, np.abs(Y[v] - ref).max())
    if qt == 12:  # the same matrix as gate and up: silu(g) * g
        ctx.dmmv_fused_gate_up_swiglu_batched(qt, Wb, 0, Wb, 0, Xb, 0, Yb, 0, M, K, ncol)
        S = Yb.download(np.float32, M * ncol).reshape(ncol, M)
        ref = orc.swiglu(Y.ravel(), Y.ravel()).reshape(ncol, M)
        # expf and the division: a few f32 ulps of the result
        assert np.allclose(S, ref, rtol=1e-6, atol=1e-7 * np.abs(ref).max()), np.abs(S - ref).max()
    for b in (Wb, Xb, Yb):
        ctx.free(b)


def test_batched_lm_head_shape(ctx, orc):
    """The LM-head shape (M >= 65536: the one-vector path is the lane-per-block
    kernel, so the columns are held to the oracle bar only)."""
    qt, M, K, ncol = 14, 70000, 4096, 4
    W = orc.synth_tensor(qt, M, K, 71, 1)
    X = np.stack([orc.synth_normal_f32(K, 71, 10 + v) for v in range(ncol)])
    Wb, Xb, Yb = ctx.upload(W), ctx.upload(X), ctx.alloc(4 * M * ncol)
    ctx.dmmv_batched(qt, Wb, 0, Xb, 0, Yb, 0, M, K, ncol)
    Y = Yb.download(np.float32, M * ncol).reshape(ncol, M)
    for v in (0, 3):
        assert_dot_close(Y[v], orc.dmmv(W, qt, X[v], M, K, nthreads=8), orc.dmmv_f64(W, qt, X[v], M, K),
                         orc.dmmv_absdot(W, qt, X[v], M, K), f"lm-head col {v}")
    for b in (Wb, Xb, Yb):
        ctx.free(b)


@pytest.mark.parametrize("ncol", [1, 2, 3, 4, 6])
def test_batched_gate_up_equals_single(ctx, orc, ncol):
    qt, M, K = 12, 2048, 4096
    Wg = orc.synth_tensor(qt | 0x100, M, K, 81, 1)
    Wu = orc.synth_tensor(qt | 0x100, M, K, 81, 2)
    X = np.stack([orc.synth_normal_f32(K, 81, 10 + v) for v in range(ncol)])
    bg, bu, Xb, Yb = ctx.upload(Wg), ctx.upload(Wu), ctx.upload(X), ctx.alloc(4 * M * ncol)
    ctx.dmmv_fused_gate_up_swiglu_batched(qt, bg, 0, bu, 0, Xb, 0, Yb, 0, M, K, ncol)
    Y = Yb.download(np.float32, M * ncol).reshape(ncol, M)
    for v in range(ncol):
        xb, yb = ctx.upload(X[v]), ctx.alloc(4 * M)
        ctx.dmmv_fused_gate_up_swiglu(qt, bg, 0, bu, 0, xb, 0, yb, 0, M, K)
        ref = yb.download(np.float32, M)
        # the one-vector path at K = 4096 is the streaming kernel: f32 summation order differs
        assert np.allclose(Y[v], ref, rtol=2e-5, atol=2e-6 * np.abs(ref).max()), (v, np.abs(Y[v] - ref).max())
        ctx.free(xb)
        ctx.free(yb)
    g = orc.dmmv(Wg, qt, X[0], M, K)
    u = orc.dmmv(Wu, qt, X[0], M, K)
    assert np.allclose(Y[0], orc.swiglu(g, u), rtol=1e-3, atol=1e-3 * np.abs(orc.swiglu(g, u)).max())
    for b in (bg, bu, Xb, Yb):
        ctx.free(b)


@pytest.mark.parametrize("M,nb,ncol", [(1, 1, 2), (129, 2, 5), (70, 5, 9), (34, 9, 16), (300, 15, 13), (4100, 17, 2),
                                       (50, 33, 16), (30, 49, 8), (46, 48, 12), (18, 64, 3), (34, 64, 16), (520, 64, 7),
                                       (1030, 16, 9), (10, 65, 2)])
def test_batched_gate_up_edges(ctx, orc, M, nb, ncol):
    """Gate and up of different matrices over the row, width (one to four
    slabs of 16 super-blocks) and group-count classes: silu(g) * u of the two
    batched DMMVs, which test_batched_edges_equal_single_columns pins, to a few
    f32 ulps (expf and the division)."""
    qt, K = 12, 256 * nb
    print(f"batched gate/up edges {M}x{K} cols {ncol}", flush=True)
    X = np.stack([orc.synth_normal_f32(K, 96, 10 + v) for v in range(ncol)])
    Wg, Wu = (ctx.upload(orc.synth_tensor(qt | 0x100, M, K, 95, 1 + m)) for m in range(2))
    Xb, Yb = ctx.upload(X), ctx.alloc(4 * M * ncol)
    gu = []
    for W in (Wg, Wu):
        ctx.dmmv_batched(qt, W, 0, Xb, 0, Yb, 0, M, K, ncol)
        gu.append(Yb.download(np.float32, M * ncol))
    assert not np.array_equal(gu[0], gu[1])
    ctx.dmmv_fused_gate_up_swiglu_batched(qt, Wg, 0, Wu, 0, Xb, 0, Yb, 0, M, K, ncol)
    S = Yb.download(np.float32, M * ncol)
    ref = orc.swiglu(gu[0], gu[1])
    assert np.allclose(S, ref, rtol=1e-6, atol=1e-7 * np.abs(ref).max()), np.abs(S - ref).max()
    for b in (Wg, Wu, Xb, Yb):
        ctx.free(b)


def test_batched_rejects_bad_arguments(ctx):
    import zinc_amd
    W, X, Y = ctx.alloc(1 << 22), ctx.alloc(1 << 20), ctx.alloc(1 << 20)
    for args, name in [((12, 256, 4096, 0), "InvalidArgument"), ((12, 256, 4096, 17), "InvalidArgument"),
                       ((8, 256, 4096, 2), "UnsupportedQuantType"), ((13, 256, 4096, 2), "UnsupportedQuantType"),
                       ((12, 256, 300, 2), "InvalidArgument"),
                       ((12, 4096, 4096, 2), "InvalidArgument")]:  # W too small
        qt, M, K, n = args
        with pytest.raises(zinc_amd.ZincError) as e:
            ctx.dmmv_batched(qt, W, 0, X, 0, Y, 0, M, K, n)
        assert e.value.name == name, args
    with pytest.raises(zinc_amd.ZincError) as e:
        ctx.dmmv_batched(12, W, 4, X, 0, Y, 0, 256, 4096, 2)  # a_off not 16-byte aligned
    assert e.value.name == "InvalidArgument"
    for b in (W, X, Y):
        ctx.free(b)


def test_batched_allocates_nothing():
    """The first batched calls of 16 contexts leave the device's free memory
    as it is (the operands have a place from the context's creation on, also
    the largest: 16 columns of K = 16384)."""
    import ctypes as C
    import zinc_amd
    from zinc_amd.hip import lib

    def free_bytes():  # of the HIP runtime the library runs on
        free, total = C.c_size_t(), C.c_size_t()
        assert lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    M, K, ncol = 256, 16384, 16
    print("batched dmmv allocations", flush=True)
    ctxs = [zinc_amd.Context(0) for _ in range(16)]
    W, X, Y = ctxs[0].alloc(M * K // 256 * 144), ctxs[0].alloc(4 * K * ncol), ctxs[0].alloc(4 * M * ncol)
    for c in ctxs:  # each stream has run: the same kernel file's one-vector route, which needs no operands
        c.dmmv_batched(12, W, 0, X, 0, Y, 0, M, K, 1)
        c.sync()
    ctxs[0].dmmv_batched(12, W, 0, X, 0, Y, 0, M, K, ncol)  # (its code is loaded)
    ctxs[0].sync()
    free = free_bytes()
    for c in ctxs[1:]:
        c.dmmv_batched(12, W, 0, X, 0, Y, 0, M, K, ncol)
        c.sync()
    assert free - free_bytes() < 4 << 20  # (the runtime's page granularity is 2 MiB)
    for b in (W, X, Y):
        ctxs[0].free(b)
    for c in ctxs:
        c.close()
