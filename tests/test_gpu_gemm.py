"""GPU parity of the matrix-core prefill matmul (spq4k_gemm / mul_mat, T > 8).

Against the reference's own GGML_OP_MUL_MAT outputs (golden vectors) and the
CPU oracle (ggml's x86 order, pinned bit-exact to the reference) on Q8_K
activations. Tolerance: close_enough, 1e-4 relative or 1e-5 absolute
(tests/desktop/test_sp_kernels.cpp:34-48)."""
import os

import numpy as np
import pytest

from _oracle import close_enough, parity_ok

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def _check(got, exp, what, exact=None):
    """close_enough of the oracle (ggml's x86 order); with `exact`, the parity
    bar's either-or: of the oracle or of the dequant-then-dot value"""
    ok = close_enough(got, exp) if exact is None else parity_ok(got, exp, exact)
    assert ok.all(), (f"{what}: {int((~ok).sum())}/{ok.size} outside tolerance; first {np.argwhere(~ok)[0]} "
                      f"got {got[tuple(np.argwhere(~ok)[0])]} exp {exp[tuple(np.argwhere(~ok)[0])]}")


def test_gemm_golden(ctx):
    G = np.load(os.path.join(HERE, "golden", "q4k_golden.npz"))
    M, K = (int(v) for v in G["mm_MK"])
    W = ctx.upload(G["mm_W"], M, K)
    _check(ctx.mul_mat(W, G["mm_X17"]), G["mm_Y17"], "golden T=17")


@pytest.mark.parametrize("M,K,T", [(256, 4096, 9), (256, 4096, 16), (192, 4096, 33), (256, 4096, 128),
                                   (128, 12288, 64), (100, 768, 40), (64, 27648, 20)])
def test_gemm_vs_oracle(ctx, oracle, M, K, T):
    rng = np.random.default_rng(M + K + T)
    W = oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32))
    X = rng.standard_normal((T, K)).astype(np.float32)
    Wd = ctx.upload(W, M, K)
    _check(ctx.mul_mat(Wd, X), oracle.mul_mat(W, M, K, X), f"gemm M={M} K={K} T={T}",
           oracle.mul_mat_dq_f64(12, W, M, K, X))


@pytest.mark.parametrize("T", [1, 3, 8])
def test_gemm_small_t_matches_gemv(ctx, oracle, T):
    from spq4k.hip import DeviceArray
    rng = np.random.default_rng(40 + T)
    M, K = 320, 2048
    W = oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32))
    X = rng.standard_normal((T, K)).astype(np.float32)
    Wd = ctx.upload(W, M, K)
    xd = DeviceArray.from_host(X)
    yd = DeviceArray((T, M), np.float32)
    ctx.gemm_dev(Wd, xd.ptr, yd.ptr, T)
    ctx.synchronize()
    _check(yd.to_host(), oracle.mul_mat(W, M, K, X), f"gemm T={T}")


@pytest.mark.parametrize("mode", [1, 2])
def test_gemm_both_kernels(oracle, mode):
    """The skinny kernel (SPQ4K_GEMM_MODE=1: K split across the workgroup's
    waves, operands from the Q8_K planes) and the tiled kernel (=2: activations
    staged in LDS, shape chosen by size) at token counts on both sides of their default
    ranges, with ragged row and token tails."""
    from _envctx import context_with
    c = context_with({"SPQ4K_GEMM_MODE": mode})
    try:
        for M, K, T in ((70, 4096, 9), (130, 2048, 17), (64, 12288, 31), (50, 768, 47), (96, 4096, 65),
                        (33, 5120, 130)):
            rng = np.random.default_rng(M * 3 + T)
            W = oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32))
            X = rng.standard_normal((T, K)).astype(np.float32)
            Wd = c.upload(W, M, K)
            _check(c.mul_mat(Wd, X), oracle.mul_mat(W, M, K, X), f"mode={mode} M={M} K={K} T={T}")
            Wd.free()
    finally:
        c.close()


def test_gemm_repeatable(ctx, oracle):
    """Fixed reduction order across the workgroup's waves: bit-identical reruns."""
    rng = np.random.default_rng(4)
    M, K, T = 200, 12288, 24
    Wd = ctx.upload(oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32)), M, K)
    X = rng.standard_normal((T, K)).astype(np.float32)
    a = ctx.mul_mat(Wd, X)
    for _ in range(3):
        np.testing.assert_array_equal(ctx.mul_mat(Wd, X), a)


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("K,shapes,T", [(4096, (256, 64, 64), 16), (2048, (300, 300), 40), (768, (17, 100, 5, 33), 100)])
def test_gemm_multi(oracle, mode, K, shapes, T):
    """q/k/v and gate/up of a prefill batch in one call: X quantised once,
    every matrix within tolerance of the oracle (both kernels take the
    matrices as segments of one launch)."""
    from spq4k.hip import DeviceArray
    from _envctx import context_with
    c = context_with({"SPQ4K_GEMM_MODE": mode})
    try:
        rng = np.random.default_rng(K + T)
        Ws = [oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32)) for M in shapes]
        X = rng.standard_normal((T, K)).astype(np.float32)
        wd = [c.upload(w, M, K) for w, M in zip(Ws, shapes)]
        xd = DeviceArray.from_host(X)
        ys = [DeviceArray.from_host(np.full((T, M), np.nan, np.float32)) for M in shapes]
        c.gemm_multi_dev(wd, xd.ptr, [y.ptr for y in ys], T)
        c.synchronize()
        for w, M, y in zip(Ws, shapes, ys):
            _check(y.to_host(), oracle.mul_mat(w, M, K, X), f"multi mode={mode} K={K} M={M} T={T}")
    finally:
        c.close()


def _extreme_weights(oracle, rng, M, K):
    """Random Q4_K rows with every fourth super-block replaced by the largest
    one (d = dmin = 2^-6, all scales and mins 63, all nibbles 15)."""
    W = oracle.quantize_q4K((rng.standard_normal((M, K)) * 0.02).astype(np.float32)).reshape(M, K // 256, 144)
    ext = np.full(144, 0xFF, np.uint8)
    ext[0:2] = ext[2:4] = np.frombuffer(np.float16(2.0 ** -6).tobytes(), np.uint8)
    W[:, ::4] = ext
    return W.reshape(-1)


def _one_sign_tokens(rng, T, K):
    X = np.abs(rng.standard_normal((T, K))).astype(np.float32) * np.where(np.arange(T) % 2, -1, 1)[:, None]
    X[0] = 1.0
    X[-1] = -1.0
    X[T // 2, : K // 2] = 3.0 * np.sign(X[T // 2, -1])
    return X.astype(np.float32)


@pytest.mark.parametrize("cfg", list(range(14)) + [32])
def test_gemm_tiled_shapes(oracle, cfg):
    """Every launch shape of the tiled kernel (SPQ4K_GEMM_CFG) with ragged row,
    token and super-block tails (K = 768 leaves a K-split wave idle), the
    largest Q4_K blocks against constant +-1 activations (|BS_j| = 4064, the
    edge of the exact fp16 min-term split), and four matrices in one launch.
    Each token has one sign: the largest blocks dequantise to 13.78 everywhere,
    and against mixed-sign tokens their sums would cancel to far below the fp32
    rounding of the terms, which no summation order can meet at 1e-4."""
    from spq4k.hip import DeviceArray
    from _envctx import context_with
    c = context_with({"SPQ4K_GEMM_MODE": 2, "SPQ4K_GEMM_CFG": cfg})
    try:
        rng = np.random.default_rng(500 + cfg)
        for M, K, T in ((150, 4096, 70), (33, 768, 17), (200, 5120, 100), (64, 12288, 65)):
            W = _extreme_weights(oracle, rng, M, K)
            X = _one_sign_tokens(rng, T, K)
            Wd = c.upload(W, M, K)
            _check(c.mul_mat(Wd, X), oracle.mul_mat(W, M, K, X), f"cfg={cfg} M={M} K={K} T={T}")
            Wd.free()
        K, T, shapes = 2048, 50, (300, 17, 129, 64)
        Ws = [_extreme_weights(oracle, rng, M, K) for M in shapes]
        X = _one_sign_tokens(rng, T, K)
        wd = [c.upload(w, M, K) for w, M in zip(Ws, shapes)]
        xd = DeviceArray.from_host(X)
        ys = [DeviceArray.from_host(np.full((T, M), np.nan, np.float32)) for M in shapes]
        c.gemm_multi_dev(wd, xd.ptr, [y.ptr for y in ys], T)
        c.synchronize()
        for w, M, y in zip(Ws, shapes, ys):
            _check(y.to_host(), oracle.mul_mat(w, M, K, X), f"cfg={cfg} multi M={M}")
    finally:
        c.close()


@pytest.mark.parametrize("M,K,T,qtype", [(4096, 12288, 16, 12), (1000, 4096, 24, 12), (4096, 12288, 16, 14),
                                         (700, 8192, 40, 13), (2048, 4096, 16, 8)])
def test_gemm_k_split_fixup(ctx, oracle, M, K, T, qtype):
    """Matmuls the planner splits over K ranges (few output tiles: the ring
    kernel's partial planes, then gemm_reduce_kernel's sum in range order),
    Q4_K, Q6_K, Q5_K and Q8_0. The result matches the oracle; a graph of the
    call replayed three times, with eager calls of another split shape between
    the replays, gives the eager result bit for bit every time."""
    from spq4k.hip import DeviceArray, Graph
    rng = np.random.default_rng(M + K + T + qtype)
    Wf = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    X = rng.standard_normal((T, K)).astype(np.float32)
    W = oracle.quantize_q8_0(Wf, ref_encoder=True) if qtype == 8 else oracle.quantize(qtype, Wf)
    Wd = ctx.upload(W, M, K, type=qtype)
    xd = DeviceArray.from_host(X)
    yd = DeviceArray((T, M), np.float32)
    ctx.mul_mat_dev(Wd, xd.ptr, yd.ptr, T)
    ctx.synchronize()
    eager = yd.to_host()
    if qtype == 8:
        exp = oracle.mul_mat_q8_0(W, M, K, X)
        _check(eager, exp, f"Q8_0 M={M} K={K} T={T}")
    else:
        _check(eager, oracle.mul_mat_type(qtype, W, M, K, X), f"type {qtype} M={M} K={K} T={T}",
               oracle.mul_mat_dq_f64(qtype, W, M, K, X))
    # another split shape between the replays
    M2, K2, T2 = 512, 12288, 20
    W2 = oracle.quantize_q4K((rng.standard_normal((M2, K2)) * 0.02).astype(np.float32))
    W2d = ctx.upload(W2, M2, K2)
    X2 = rng.standard_normal((T2, K2)).astype(np.float32)
    exp2 = ctx.mul_mat(W2d, X2)
    yd.fill_byte(0)
    with Graph.capture(ctx.stream) as g:
        ctx.mul_mat_dev(Wd, xd.ptr, yd.ptr, T)
    for rep in range(3):
        yd.fill_byte(0)
        g.launch()
        ctx.synchronize()
        got = yd.to_host()
        assert np.array_equal(got.view(np.uint32), eager.view(np.uint32)), f"replay {rep} differs from the eager call"
        assert np.array_equal(ctx.mul_mat(W2d, X2).view(np.uint32), exp2.view(np.uint32)), f"eager call after replay {rep}"
    del g
    for a in (Wd, W2d, xd, yd):
        a.free()


@pytest.mark.parametrize("qtype", [8, 12, 13, 14])   # Q8_0, Q4_K, Q5_K, Q6_K
@pytest.mark.parametrize("M,nb,T", [(70, 5, 9), (1100, 7, 40), (520, 33, 100), (300, 11, 260), (4100, 3, 17),
                                    (2060, 16, 5), (2100, 8, 16), (4111, 13, 16), (37, 1, 4)])
def test_gemm_plan_ranges(ctx, oracle, M, nb, T, qtype):
    """Shapes whose split leaves ranges of one super-block, a shorter last
    range, or many ranges of few tiles (ragged rows and tokens), and the
    matrices small enough for the skinny kernel: against the oracle, and the no-allocation call (the same plan) bit for bit."""
    from spq4k.hip import DeviceArray
    K = 256 * nb
    rng = np.random.default_rng(M + K + T + qtype)
    Wf = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    X = rng.standard_normal((T, K)).astype(np.float32)
    W = oracle.quantize_q8_0(Wf, ref_encoder=True) if qtype == 8 else oracle.quantize(qtype, Wf)
    Wd = ctx.upload(W, M, K, type=qtype)
    xd, yd, y2 = DeviceArray.from_host(X), DeviceArray((T, M)), DeviceArray((T, M))
    ctx.mul_mat_dev(Wd, xd.ptr, yd.ptr, T)
    assert ctx.lib.spq4k_mul_mat_noalloc(ctx.handle, Wd.handle, xd.ptr, y2.ptr, T) == 0
    ctx.synchronize()
    got = yd.to_host()
    if qtype == 8:
        _check(got, oracle.mul_mat_q8_0(W, M, K, X), f"Q8_0 M={M} K={K} T={T}")
    else:
        _check(got, oracle.mul_mat_type(qtype, W, M, K, X), f"type {qtype} M={M} K={K} T={T}",
               oracle.mul_mat_dq_f64(qtype, W, M, K, X))
    assert np.array_equal(got.view(np.uint32), y2.to_host().view(np.uint32))


@pytest.mark.parametrize("cfg", list(range(33, 41)))
def test_gemm_two_stage_shapes(oracle, cfg):
    """The 64-row two-stage launch shapes of each format (SPQ4K_GEMM_CFG) with
    ragged rows, tokens and ranges, against the oracle."""
    from _envctx import context_with
    qtype = (12, 14, 13, 8)[(cfg - 33) % 4]
    c = context_with({"SPQ4K_GEMM_CFG": cfg})
    try:
        rng = np.random.default_rng(cfg)
        for M, K, T in ((130, 1280, 33), (67, 256, 65), (64, 4096, 9)):
            Wf = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
            X = rng.standard_normal((T, K)).astype(np.float32)
            W = oracle.quantize_q8_0(Wf, ref_encoder=True) if qtype == 8 else oracle.quantize(qtype, Wf)
            got = c.mul_mat(c.upload(W, M, K, type=qtype), X)
            exp = oracle.mul_mat_q8_0(W, M, K, X) if qtype == 8 else oracle.mul_mat_type(qtype, W, M, K, X)
            exact = None if qtype == 8 else oracle.mul_mat_dq_f64(qtype, W, M, K, X)
            _check(got, exp, f"cfg={cfg} M={M} K={K} T={T}", exact)
    finally:
        c.close()


@pytest.mark.parametrize("T", [5, 12])
def test_gemm_mode_tiled_small_batch(oracle, T):
    """SPQ4K_GEMM_MODE=2 keeps a small Q4_K matrix, which would take the skinny
    kernel, on the tiled kernels at every batch size: planes, matmul and the
    pass that sums the K ranges (the skinny kernel needs no third launch)."""
    import ctypes as C

    from _envctx import context_with
    from spq4k.hip import DeviceArray, Graph, _lib, check
    M, K = 4096, 2048
    rng = np.random.default_rng(T)
    W = oracle.quantize(12, (rng.standard_normal((M, K)) * 0.02).astype(np.float32))
    X = rng.standard_normal((T, K)).astype(np.float32)
    launches = []
    for mode in (0, 2):
        c = context_with({"SPQ4K_GEMM_MODE": mode})
        try:
            Wd = c.upload(W, M, K)
            xd, yd = DeviceArray.from_host(X), DeviceArray((T, M))
            with Graph.capture(c.stream) as g:
                c.mul_mat_dev(Wd, xd.ptr, yd.ptr, T)
            n = C.c_size_t()
            check(_lib().hipGraphGetNodes(C.c_void_p(g.graph), None, C.byref(n)), "hipGraphGetNodes")
            launches.append(n.value)
            g.launch()
            c.synchronize()
            _check(yd.to_host(), oracle.mul_mat_type(12, W, M, K, X), f"mode {mode} T={T}")
        finally:
            c.close()
    assert launches == [2, 3], launches
