"""GPU parity of axhip_gemm (the nn::Linear / ops::matmul path) against float64
and against the CPU oracle's matmul."""
import ctypes as C
import math

import numpy as np
import pytest

from oracle import axo
from tests import gpu_harness as gh

pytestmark = pytest.mark.gpu
F32, F16, BF16 = axo.F32, axo.F16, axo.BF16


def test_linear_known_answers():
    # tests/test_nn_layers.cpp:12-73
    x, W = np.ones((1, 3), np.float32), np.ones((2, 3), np.float32)
    assert np.all(gh.gemm(x, W, F32, trans_b=True) == 3.0)
    assert np.all(gh.gemm(x, W, F32, trans_b=True, bias=np.ones(2, np.float32)) == 4.0)
    assert np.all(gh.gemm(np.ones((2, 4), np.float32), np.full((3, 4), 0.5, np.float32), F32, trans_b=True) == 2.0)
    assert np.all(gh.gemm(np.ones((5, 8), np.float32), np.ones((8, 8), np.float32), F32) == 8.0)


@pytest.mark.parametrize("M,N,K,ta,tb", [(7, 5, 9, False, False), (64, 64, 64, False, True), (70, 130, 300, True, False),
                                          (33, 129, 65, True, True), (1500, 1280, 1280, False, True)])
def test_f32_matches_oracle(M, N, K, ta, tb):
    g = axo.PCG64(M + N)
    A = g.normal((K, M) if ta else (M, K))
    B = g.normal((N, K) if tb else (K, N)) * (0.02 if K > 1000 else 1.0)
    got = gh.gemm(A, B, F32, ta, tb)[0]
    want = axo.matmul(A, B, F32, ta, tb)
    assert np.allclose(got, want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("M,N,K,extras,batch", [(1500, 1280, 1280, False, 1), (300, 250, 36, True, 1), (260, 257, 100, True, 1),
                                                (1500, 3840, 384, False, 1), (2000, 330, 240, True, 1), (256, 256, 32, False, 1),
                                                (200, 136, 520, True, 3)])
def test_f32_mfma_path_matches_fp64(M, N, K, extras, batch):
    """fp32 x W^T on the fp32 matrix instruction: ragged tiles, k extents that are not a multiple of the 32-float
    k-tile (36, 100, 240, 520), fewer k-tiles than ring stages, every tile shape, batches against a shared weight,
    and the bias / residual / GELU epilogue.  fp32 products and sums: held to the fp32 bar against float64."""
    import math

    g = axo.PCG64(M * 3 + K)
    x = g.normal((batch, M, K)).astype(np.float32)
    W = (g.normal((N, K)) / np.sqrt(K)).astype(np.float32)
    bias = (g.normal((N,)) * 0.1).astype(np.float32) if extras else None
    res = g.normal((batch, M, N)).astype(np.float32) if extras else None
    got = gh.gemm(x, W, F32, trans_b=True, bias=bias, residual=res, epilogue="gelu" if extras else None)
    want = x.astype(np.float64) @ W.astype(np.float64).T
    if extras:
        y = want + bias + res
        want = 0.5 * y * (1 + np.vectorize(math.erf)(y / math.sqrt(2)))
    assert got.shape == (batch, M, N)
    assert np.allclose(got, want, rtol=1e-4, atol=1e-4), np.max(np.abs(got - want))


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1, 3, 8), (128, 128, 64), (130, 70, 200), (1500, 1280, 1280)])
def test_half_linear_matches_fp32_reference(dt, M, N, K):
    g = axo.PCG64(K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((N, K)) * 0.02, dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt)
    res = axo.to_bits(g.normal((M, N)), dt)
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=True, bias=bias, residual=res)[0], dt)
    xf, Wf = axo.to_f32(x, dt).astype(np.float64), axo.to_f32(W, dt).astype(np.float64)
    want = xf @ Wf.T + axo.to_f32(bias, dt) + axo.to_f32(res, dt)
    assert np.max(np.abs(got - want)) < 2e-2 + 2.0**-8 * np.max(np.abs(want))


def test_batched_shared_weight_and_gelu_epilogue():
    g = axo.PCG64(5)
    x, W = axo.to_bits(g.normal((3, 40, 64)), BF16), axo.to_bits(g.normal((48, 64)) * 0.1, BF16)
    got = axo.to_f32(gh.gemm(x, W, BF16, trans_b=True, epilogue="gelu"), BF16)
    y = axo.to_f32(x, BF16).astype(np.float64) @ axo.to_f32(W, BF16).astype(np.float64).T
    import math

    want = 0.5 * y * (1 + np.vectorize(math.erf)(y / math.sqrt(2)))
    assert np.max(np.abs(got - want)) < 2e-2


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,extras", [(2300, 3800, 192, True), (2304, 3840, 64, False), (4096, 2048, 320, False)])
def test_half_large_tile_path_matches_fp64(dt, M, N, K, extras):
    """Shapes that take the 256 x 256 work-group tiles, with ragged last tiles in both
    directions, a k extent of one and of several tiles, and the full epilogue."""
    g = axo.PCG64(M + K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((N, K)) * 0.05, dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt) if extras else None
    res = axo.to_bits(g.normal((M, N)), dt) if extras else None
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=True, bias=bias, residual=res, epilogue="relu" if extras else None)[0], dt)
    want = axo.to_f32(x, dt).astype(np.float64) @ axo.to_f32(W, dt).astype(np.float64).T
    if extras:
        want = np.maximum(want + axo.to_f32(bias, dt) + axo.to_f32(res, dt), 0.0)
    assert np.max(np.abs(got - want)) < 2e-2 + 2.0**-8 * np.max(np.abs(want))
    # and the CPU oracle's matmul (accumulates in the 16-bit type as the reference's CPU path
    # does, cpu_operations.cpp:1840-1872) stays within its own, wider, band on a corner block
    if not extras and K <= 64:
        o = axo.to_f32(axo.matmul(x[:64], W[:64], dt, False, True), dt)
        assert np.max(np.abs(o - got[:64, :64])) < 0.25


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,epilogue,with_bias,with_res", [
    (2050, 3803, 128, "gelu", True, True),    # odd row pitch of C: two-byte stores everywhere
    (2049, 3802, 256, None, False, True),     # a last column group of two: masked tail beside 8-byte stores
    (2304, 3801, 64, "silu", True, False),    # one k-tile
    (2100, 2310, 448, "tanh", False, False),
    (4096, 2048, 512, "sigmoid", True, True)])
def test_half_large_tile_epilogues_and_column_tails(dt, M, N, K, epilogue, with_bias, with_res):
    """The 256 x 256 kernel's epilogue: a lane owns four consecutive columns of a row, stored as 8 bytes where the
    row pitch and the origin allow it and as masked 2-byte stores otherwise; every activation, with and without bias
    and residual, against float64."""
    g = axo.PCG64(3 * M + N + K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((N, K)) * 0.05, dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt) if with_bias else None
    res = axo.to_bits(g.normal((M, N)), dt) if with_res else None
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=True, bias=bias, residual=res, epilogue=epilogue)[0], dt)
    want = axo.to_f32(x, dt).astype(np.float64) @ axo.to_f32(W, dt).astype(np.float64).T
    if with_bias:
        want = want + axo.to_f32(bias, dt)
    if with_res:
        want = want + axo.to_f32(res, dt)
    if epilogue == "gelu":
        from scipy.special import erf
        want = 0.5 * want * (1.0 + erf(want / np.sqrt(2.0)))
    elif epilogue == "silu":
        want = want / (1.0 + np.exp(-want))
    elif epilogue == "tanh":
        want = np.tanh(want)
    elif epilogue == "sigmoid":
        want = 1.0 / (1.0 + np.exp(-want))
    assert got.shape == want.shape
    assert np.max(np.abs(got - want)) < 2e-2 + 2.0**-8 * np.max(np.abs(want))


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,extras", [(1500, 5120, 1280, False), (1500, 1280, 5120, True), (200, 330, 256, True), (129, 257, 320, False),
                                          (1000, 2000, 448, True), (64, 128, 4096, False),
                                          (1500, 3840, 1280, False), (1500, 3700, 320, True)])
def test_half_ring_path_matches_fp64(dt, M, N, K, extras):
    """Mid-size products: the tile kernels (256 x 128 down to 64 x 128 tiles, k-tiles in a ring of LDS stages) and, for the
    few tiles of the smallest, the ones whose wavefronts share k, with k extents of exactly, fewer and more k-tiles than
    the ring has stages, ragged tiles, and the full epilogue."""
    g = axo.PCG64(M * 7 + K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((N, K)) * (2.0 / np.sqrt(K)), dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt) if extras else None
    res = axo.to_bits(g.normal((M, N)), dt) if extras else None
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=True, bias=bias, residual=res, epilogue="gelu" if extras else None)[0], dt)
    want = axo.to_f32(x, dt).astype(np.float64) @ axo.to_f32(W, dt).astype(np.float64).T
    if extras:
        import math

        y = want + axo.to_f32(bias, dt) + axo.to_f32(res, dt)
        want = 0.5 * y * (1 + np.vectorize(math.erf)(y / math.sqrt(2)))
    assert np.max(np.abs(got - want)) < 2e-2 + 2.0**-8 * np.max(np.abs(want))


@pytest.mark.parametrize("dt", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("ta,tb,K", [(False, False, 264), (True, False, 264), (True, True, 264), (False, True, 263), (True, False, 301)],
                         ids=["nn", "tn", "tt", "nt_k263", "tn_k301"])
def test_large_products_with_operands_not_along_k(dt, ta, tb, K):
    """Large products whose A is stored [k, m] and / or whose B is stored [k, n], or whose k is not a whole number of
    16-byte vectors: the library repacks such operands into temporary memory (transposed, k zero-padded) and runs the
    k-contiguous kernels; same bar as those.  Batched, with a shared B."""
    M, N, nb = 1040, 784, 3  # (above the size from which the library repacks)
    g = axo.PCG64(M + N + int(ta) + 2 * int(tb))
    A = axo.to_bits(g.normal((nb, K, M) if ta else (nb, M, K)), dt)
    B = axo.to_bits(g.normal((N, K) if tb else (K, N)) * 0.05, dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt)
    got = axo.to_f32(gh.gemm(A, B, dt, trans_a=ta, trans_b=tb, bias=bias, epilogue="relu"), dt)
    a64, b64 = axo.to_f32(A, dt).astype(np.float64), axo.to_f32(B, dt).astype(np.float64)
    want = np.maximum((a64.transpose(0, 2, 1) if ta else a64) @ (b64.T if tb else b64) + axo.to_f32(bias, dt), 0.0)
    tol = 1e-4 + 1e-4 * np.abs(want) if dt == F32 else 2e-2 + 2.0**-8 * np.abs(want)
    assert np.all(np.abs(got - want) <= tol)
    # per-batch B as well
    Bb = axo.to_bits(g.normal((nb, N, K) if tb else (nb, K, N)) * 0.05, dt)
    got = axo.to_f32(gh.gemm(A, Bb, dt, trans_a=ta, trans_b=tb), dt)
    bb64 = axo.to_f32(Bb, dt).astype(np.float64)
    want = (a64.transpose(0, 2, 1) if ta else a64) @ (bb64.transpose(0, 2, 1) if tb else bb64)
    tol = 1e-4 + 1e-4 * np.abs(want) if dt == F32 else 2e-2 + 2.0**-8 * np.abs(want)
    assert np.all(np.abs(got - want) <= tol)


@pytest.mark.parametrize("dt", [F32, BF16, F16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,N,K,extras", [(1, 1280, 1280, False), (1, 4096, 4096, True), (5, 100, 5120, True), (32, 1283, 264, False), (8, 51865, 384, False),
                                          (3, 2048, 4104, True), (1, 32, 256, False), (2, 4099, 776, True), (7, 16390, 520, False), (4, 1, 264, True)])
def test_skinny_products_of_a_decoding_step_match_fp64(dt, M, N, K, extras):
    """A few rows against a weight matrix (x W^T): up to 8 rows take the kernel that walks W's rows with whole
    wavefronts (1, 2 or 4 rows of W each, by N), ragged N and k tails, bias + residual + GELU; 32 rows stay on the
    tiled kernels; same bar for both."""
    g = axo.PCG64(M * 7 + N + K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((N, K)) * 0.05, dt)
    bias = axo.to_bits(g.normal((N,)) * 0.1, dt) if extras else None
    res = axo.to_bits(g.normal((M, N)), dt) if extras else None
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=True, bias=bias, residual=res, epilogue="gelu" if extras else None)[0], dt)
    want = axo.to_f32(x, dt).astype(np.float64) @ axo.to_f32(W, dt).astype(np.float64).T
    if extras:
        want = want + axo.to_f32(bias, dt) + axo.to_f32(res, dt)
        want = 0.5 * want * (1.0 + np.vectorize(math.erf)(want / math.sqrt(2.0)))
    if dt == F32:
        assert np.max(np.abs(got - want)) < 1e-4 + 1e-5 * np.max(np.abs(want))
    else:
        assert np.max(np.abs(got - want)) < 2e-2 + 2.0**-8 * np.max(np.abs(want))


@pytest.mark.parametrize("dt", [F32, BF16, F16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(m, 37, 264) for m in range(1, 9)] + [(2, 3001, 24576), (3, 2051, 32768), (5, 1025, 65536), (8, 1023, 65792)])
def test_skinny_sums_reach_their_row_and_column(dt, M, N, K):
    """One to eight rows of x on one row of W per wavefront, and two, three, five and eight on two (W of 64 M elements and more),
    W's last one alone or not: whole numbers whose products add up without rounding, with bias, residual and RELU."""
    g = axo.PCG64(M * 31 + N)
    x, W = np.zeros((M, K), np.float32), np.zeros((N, K), np.float32)
    hit = (np.arange(N) * 8191) % K  # row n of W picks column hit[n] of x, and its last one
    W[np.arange(N), hit] += 2.0
    W[:, K - 1] += 1.0
    x[:] = (np.arange(M)[:, None] * 37 + np.arange(K)[None, :] * 11) % 23 - 11.0
    bias, res = (np.round(4 * g.normal(s)).astype(np.float32) for s in ((N,), (M, N)))
    got = axo.to_f32(gh.gemm(*(axo.to_bits(t, dt) for t in (x, W)), dt, trans_b=True, bias=axo.to_bits(bias, dt), residual=axo.to_bits(res, dt), epilogue="relu")[0], dt)
    want = np.maximum(2.0 * x[:, hit] + x[:, K - 1 :] + bias + res, 0.0)
    assert np.array_equal(got, want)


def test_skinny_sums_of_four_rows_of_w():
    """Four rows of W per wavefront, up to 32 sums over its lanes: a setting that is read once, so it has a process of its own."""
    import os
    import subprocess
    import sys

    if os.environ.get("AXHIP_GEMM_SKINNY_ROWS"):
        pytest.skip("already inside a forced run")
    r = subprocess.run([sys.executable, "-m", "pytest", "-x", "-q", "-p", "no:cacheprovider", __file__, "-k", "test_skinny_sums_reach and 37-264"],
                       env=dict(os.environ, AXHIP_GEMM_SKINNY_ROWS="4"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0 and "24 passed" in r.stdout, r.stdout[-3000:]


@pytest.mark.parametrize("M,N,K", [(3, 3072, 4096), (5, 4376, 5720), (8, 4728, 1056), (8, 1160, 5120), (4, 20096, 560)])
def test_fp32_products_of_a_few_rows_keep_short_sums(M, N, K):
    """A lane's chain is the K / 64 products it owns, then six steps over the lanes.  An addition is off by 0.41 u of its
    result in the mean square; a chain of n terms adds up n / 2 of the final sum's variance, a step over the lanes all of it:
    u sqrt(K / 128 + 7) times 0.41, and 0.55 with room for the sample.  (Chains of K / 8: twice to four times as much.)"""
    r = np.random.default_rng(M * N)
    x, W = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((N, K)).astype(np.float32)
    want = x.astype(np.float64) @ W.T.astype(np.float64)
    got = gh.gemm(x, W, F32, trans_b=True)[0]
    assert np.linalg.norm(got - want) <= 0.55 * 2.0**-24 * np.sqrt(K / 128 + 7) * np.linalg.norm(want)


@pytest.mark.parametrize("dt", [F32, BF16, F16], ids=["f32", "bf16", "f16"])
def test_few_rows_too_far_apart_for_the_tiled_kernels(dt):
    """Four rows of x 2^21 elements apart, past the 32-bit offsets of the 16-bit tile kernels, and more outputs than the kernel
    for a few rows otherwise takes."""
    from axiom_amd import capi

    M, N, K, lda = 4, 2304, 512, 1 << 21
    r = np.random.default_rng(3)
    x, W = r.integers(-3, 4, (M, K)).astype(np.float32), r.integers(-2, 3, (N, K)).astype(np.float32)
    far = np.zeros((M, lda), np.float32)
    far[:, :K] = x
    a, b, c = gh.to_dev(axo.to_bits(far, dt)), gh.to_dev(axo.to_bits(W, dt)), gh.empty_dev((M, N), dt)
    p = capi.GemmParams()
    p.dtype, p.trans_a, p.trans_b, p.m, p.n, p.k, p.batch = dt, 0, 1, M, N, K, 1
    p.lda, p.ldb, p.ldc, p.stride_a, p.stride_b, p.stride_c = lda, K, N, M * lda, N * K, M * N
    gh.sync()
    capi.check(capi.lib().axhip_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    assert np.array_equal(axo.to_f32(gh.to_host(c, gh.np_store_dtype(dt)), dt), x @ W.T if dt == F32 else axo.to_f32(axo.to_bits(x @ W.T, dt), dt))


def test_the_fp32_ring_adds_up_odd_and_even_numbers_of_k_tiles():
    """Whole numbers, exact in every order of the sum: 64 x 64 tiles of fp32 products with one work-group per CU and
    with several, two to five k-tiles and a ragged last one, rows off the tile, with and without each epilogue step."""
    for M, N in ((1000, 980), (1500, 1284)):
        for K in (64, 96, 100, 128, 131, 160):
            r = np.random.default_rng(M + K)
            a, b = (r.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (K, N)))
            bias, res = (r.integers(-9, 10, s).astype(np.float32) for s in ((N,), (M, N)))
            assert np.array_equal(gh.gemm(a, b, F32)[0], a @ b), (M, N, K)
            got = gh.gemm(a, np.ascontiguousarray(b.T), F32, trans_b=True, bias=bias, residual=res, epilogue="relu")[0]
            assert np.array_equal(got, np.maximum(a @ b + bias + res, 0.0)), (M, N, K)


@pytest.mark.parametrize("dt", [F32, BF16, F16], ids=["f32", "bf16", "f16"])
def test_seeded_random_shapes_match_fp64(dt):
    """Forty seeded random products per dtype, shaped to land on every kernel and tile shape (matrix-core ring tiles,
    the 256 x 256 kernel, the register-staged and FMA fallbacks): ragged m and n, k with and without the alignment the
    matrix-core paths need, batches against a shared or a per-batch right operand, random epilogues."""
    import math

    r = np.random.default_rng(1234 + dt)
    erf = np.vectorize(math.erf)
    for case in range(40):
        big = case % 8 == 0
        M = int(r.integers(1, 2200 if big else 700))
        N = int(r.integers(1, 2200 if big else 700))
        K = int(r.choice([r.integers(1, 600), 8 * r.integers(1, 80), 64 * r.integers(1, 12)]))
        batch = int(r.choice([1, 1, 2, 3])) if not big else 1
        shared_w = bool(r.integers(0, 2))
        extras = bool(r.integers(0, 2))
        epi = [None, "relu", "gelu"][int(r.integers(0, 3))] if extras else None
        g = axo.PCG64(case * 7 + 1)
        x = g.normal((batch, M, K))
        W = g.normal((N, K) if shared_w else (batch, N, K)) / np.sqrt(K)
        bias = g.normal((N,)) * 0.1 if extras else None
        res = g.normal((batch, M, N)) if extras else None
        if dt == F32:
            xs, Ws = x.astype(np.float32), W.astype(np.float32)
            bs, rs = (bias.astype(np.float32), res.astype(np.float32)) if extras else (None, None)
            xf, Wf, bf, rf = xs, Ws, bs, rs
        else:
            xs, Ws = axo.to_bits(x, dt), axo.to_bits(W, dt)
            bs, rs = (axo.to_bits(bias, dt), axo.to_bits(res, dt)) if extras else (None, None)
            xf, Wf = axo.to_f32(xs, dt), axo.to_f32(Ws, dt)
            bf, rf = (axo.to_f32(bs, dt), axo.to_f32(rs, dt)) if extras else (None, None)
        got = gh.gemm(xs, Ws, dt, trans_b=True, bias=bs, residual=rs, epilogue=epi)
        got = got.astype(np.float64) if dt == F32 else axo.to_f32(got, dt).astype(np.float64)
        want = xf.astype(np.float64) @ np.swapaxes(Wf.astype(np.float64), -1, -2)
        if extras:
            want = want + bf + rf
            if epi == "relu":
                want = np.maximum(want, 0.0)
            elif epi == "gelu":
                want = 0.5 * want * (1 + erf(want / math.sqrt(2)))
        tol = 1e-4 * (1 + np.abs(want)) if dt == F32 else 2e-2 + 2.0**-8 * np.abs(want)
        assert got.shape == (batch, M, N)
        assert np.all(np.abs(got - want) <= tol), (case, M, N, K, batch, shared_w, epi, float(np.max(np.abs(got - want))))


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch", [
    (1, 9, 8, 1), (17, 33, 65, 3), (33, 64, 71, 1), (16, 63, 64, 2), (65, 72, 200, 1), (40, 2056, 1032, 1), (129, 1000, 511, 1),  # few rows or few tiles
    (300, 2104, 200, 2), (385, 5128, 264, 1), (1025, 3848, 136, 1), (1537, 5000, 72, 1),  # 64 .. 256 x 128 tiles, k not whole k-tiles
    (1500, 2001, 203, 1), (1100, 1999, 1001, 1)])  # 128 x 128 tiles through registers: rows off the 16-byte grid
def test_half_products_at_the_edges_of_tiles(dt, nn, M, N, K, batch):
    """x W^T and a b of every 16-bit kernel: one element more and fewer than tiles, pieces of k and 16-byte vectors,
    rows shorter than a tile (n of 9 and 63), bias + residual + activation.  Against float64 of the same 16-bit inputs:
    the result is rounded once (half an ulp: 2^-8 of it at most with bf16's 8 significant bits, 2^-11 with f16's 11), the sum is fp32 (K ulps of the sum of magnitudes at most)."""
    g = axo.PCG64(3 * M + 5 * N + K)
    x = axo.to_bits(g.normal((batch, M, K)), dt)
    W = axo.to_bits(g.normal((batch, K, N) if nn else (batch, N, K)) / np.sqrt(K), dt)
    bias, res = axo.to_bits(g.normal((N,)) * 0.1, dt), axo.to_bits(g.normal((batch, M, N)), dt)
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=not nn, bias=bias, residual=res, epilogue="relu"), dt).astype(np.float64)
    x64, w64 = axo.to_f32(x, dt).astype(np.float64), axo.to_f32(W, dt).astype(np.float64)
    w64 = w64 if nn else np.swapaxes(w64, -1, -2)
    b64, r64 = axo.to_f32(bias, dt).astype(np.float64), axo.to_f32(res, dt).astype(np.float64)
    want = np.maximum(x64 @ w64 + b64 + r64, 0.0)
    magnitude = np.abs(x64) @ np.abs(w64) + np.abs(b64) + np.abs(r64)
    tol = (2.0**-8 if dt == BF16 else 2.0**-11) * np.abs(want) + (K + 2) * 2.0**-24 * magnitude + (0.0 if dt == BF16 else 2.0**-25)
    assert got.shape == want.shape
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) - tol))


@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch", [
    (90, 37, 33, 1), (17, 261, 32, 3), (16, 1041, 95, 1), (65, 50, 1024, 2), (9, 700, 2049, 1),  # 16 rows: pieces of 64 and 32 k, whole and broken
    (33, 515, 64, 9), (513, 129, 100, 4), (31, 4, 600, 1), (200, 2047, 257, 1),                  # 32 rows; n of one lane's columns
    (1000, 1030, 70, 1), (385, 67, 130, 32), (1023, 961, 513, 1)])                               # 64 x 64
def test_f32_products_at_the_edges_of_tiles(nn, M, N, K, batch):
    """x W^T and a b in fp32 without shared tiles: rows, columns and k that end inside a tile, a lane's columns and a
    piece, with bias, residual and activation.  Against float64: K + 2 roundings of the sum of magnitudes at most."""
    g = axo.PCG64(7 * M + 3 * N + K)
    x, W = g.normal((batch, M, K)).astype(np.float32), (g.normal((batch, K, N) if nn else (batch, N, K)) / np.sqrt(K)).astype(np.float32)
    bias, res = (g.normal((N,)) * 0.1).astype(np.float32), g.normal((batch, M, N)).astype(np.float32)
    got = gh.gemm(x, W, F32, trans_b=not nn, bias=bias, residual=res, epilogue="relu").astype(np.float64)
    x64, w64 = x.astype(np.float64), W.astype(np.float64) if nn else np.swapaxes(W.astype(np.float64), -1, -2)
    want = np.maximum(x64 @ w64 + bias + res, 0.0)
    magnitude = np.abs(x64) @ np.abs(w64) + np.abs(bias) + np.abs(res)
    assert got.shape == want.shape
    assert np.all(np.abs(got - want) <= (K + 2) * 2.0**-24 * magnitude)


@pytest.mark.parametrize("M,N,K,batch", [(2048, 2044, 132, 1), (1000, 1100, 260, 8), (1024, 1024, 1024, 1), (1300, 4000, 44, 3), (700, 2500, 1000, 1)])
def test_f32_products_of_plain_matrices_on_the_ring(M, N, K, batch):
    """a b with b stored [k, n] in whole vectors, sizes of several of the ring kernel's tiles: k that ends inside a k-tile, rows
    and columns inside a tile; b lies in front of NaNs.  The same bound as above."""
    import ctypes as C

    import torch

    from axiom_amd import capi

    g = axo.PCG64(M + N + K)
    x, W = g.normal((batch, M, K)).astype(np.float32), (g.normal((batch, K, N)) / np.sqrt(K)).astype(np.float32)
    da, db = gh.to_dev(x), torch.full((batch * K * N + 64 * N,), float("nan"), device="cuda")
    db[: batch * K * N] = gh.to_dev(W).flatten()
    c = gh.empty_dev((batch, M, N), F32)
    p = capi.GemmParams()
    p.dtype, p.m, p.n, p.k, p.batch, p.lda, p.ldb, p.ldc = F32, M, N, K, batch, K, N, N
    p.stride_a, p.stride_b, p.stride_c = M * K, K * N, M * N
    gh.sync()
    capi.check(capi.lib().axhip_gemm(da.data_ptr(), db.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    got = c.double()
    x64, w64 = da.double(), gh.to_dev(W).double()
    assert bool(((got - x64 @ w64).abs() <= (K + 2) * 2.0**-24 * (x64.abs() @ w64.abs())).all())


@pytest.mark.parametrize("dt", [BF16, F16], ids=["bf16", "f16"])
@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("K", [9, 65, 127, 193, 257, 321, 385, 449, 513, 577, 641, 705])
def test_half_products_through_registers_of_every_number_of_k_tiles(dt, nn, K):
    """Unaligned rows on the tile kernel that loads through registers, from one k-tile to what its pipeline holds twice
    over, and the unaligned stores of C (rows of an odd number of columns, ragged last tiles).  The bound of
    test_half_products_at_the_edges_of_tiles."""
    import torch

    M, N = 1930, 2001
    g = axo.PCG64(K)
    x, W = axo.to_bits(g.normal((M, K)), dt), axo.to_bits(g.normal((K, N) if nn else (N, K)) / np.sqrt(K), dt)
    bias, res = axo.to_bits(g.normal((N,)) * 0.1, dt), axo.to_bits(g.normal((M, N)), dt)
    got = axo.to_f32(gh.gemm(x, W, dt, trans_b=not nn, bias=bias, residual=res), dt).reshape(M, N)
    on = lambda t: torch.from_numpy(np.ascontiguousarray(axo.to_f32(t, dt))).cuda().double()
    x64, w64, extra = on(x), on(W) if nn else on(W).t().contiguous(), on(bias) + on(res)
    want, magnitude = x64 @ w64 + extra, x64.abs() @ w64.abs() + on(bias).abs() + on(res).abs()
    tol = (2.0**-8 if dt == BF16 else 2.0**-11) * want.abs() + (K + 2) * 2.0**-24 * magnitude + (0.0 if dt == BF16 else 2.0**-25)
    assert bool(((torch.from_numpy(got).cuda().double() - want).abs() <= tol).all())


@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch", [
    (1025, 1027, 33, 1), (1000, 1001, 95, 2), (513, 2049, 127, 1), (1919, 1921, 129, 1), (1920, 1920, 730, 1),  # 64 x 64 and 64 x 128, K of every remainder of 4
    (2300, 130, 161, 8), (700, 2813, 385, 1), (4000, 3999, 1001, 1)])
def test_f32_products_of_rows_that_start_anywhere_on_the_ring(nn, M, N, K, batch):
    """The ring kernel without 16-byte alignment: k that ends inside a chunk (what lies behind it in memory are other rows,
    here with infinities and NaNs next to the operands), column tiles moved left to end with the rows, bias and residual.
    The bound of the tests above; its sums are chains of 32 and then one per k-tile, so the error is also held to that of
    chains that long: (32 + K / 32 + 4) half ulps of the sum of magnitudes."""
    import ctypes as C

    import torch

    from axiom_amd import capi

    g = axo.PCG64(M + 3 * N + K)
    x, W = g.normal((batch, M, K)).astype(np.float32), (g.normal((batch, K, N) if nn else (batch, N, K)) / np.sqrt(K)).astype(np.float32)
    def off_grid(t):  # one float into a buffer of NaNs
        buf = torch.full((t.size + 600,), float("nan"), device="cuda")
        buf[1:1 + t.size] = gh.to_dev(t).flatten()
        return buf, buf[1:1 + t.size].view(t.shape)
    (_, da), (_, db) = off_grid(x), off_grid(W)
    bias, res = gh.to_dev((g.normal((N,)) * 0.1).astype(np.float32)), gh.to_dev(g.normal((batch, M, N)).astype(np.float32))
    c = gh.empty_dev((batch, M, N), F32)
    p = capi.GemmParams()
    p.dtype, p.m, p.n, p.k, p.batch, p.lda, p.ldb, p.ldc, p.trans_b = F32, M, N, K, batch, K, N if nn else K, N, int(not nn)
    p.stride_a, p.stride_b, p.stride_c = M * K, K * N, M * N
    p.bias, p.residual = bias.data_ptr(), res.data_ptr()
    torch.cuda.synchronize()
    gh.sync()
    capi.check(capi.lib().axhip_gemm(da.data_ptr(), db.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    for b in range(batch):
        x64, w64 = da[b].double(), db[b].double() if nn else db[b].double().t().contiguous()
        want, magnitude = x64 @ w64 + bias.double() + res[b].double(), x64.abs() @ w64.abs() + bias.double().abs() + res[b].double().abs()
        err = (c[b].double() - want).abs()
        assert bool((err <= min(K + 2, 36 + K / 32) * 2.0**-24 * magnitude).all())


@pytest.mark.parametrize("dtype", [F32, F16, BF16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch,shared", [
    (16, 16, 64, 3, False), (40, 72, 96, 5, True), (50, 200, 128, 7, False),    # one tile a product, fewer products than XCDs
    (192, 1536, 264, 9, False), (130, 390, 200, 11, True), (640, 320, 512, 8, False), # 3 .. 15 tiles: products change inside an XCD's range
    (513, 700, 130, 3, False), (257, 2050, 2112, 2, True), (16, 64, 32, 1000, False)])
def test_batches_are_dealt_over_all_xcds(dtype, nn, M, N, K, batch, shared):
    """Every tile of every product is computed once, with its own residual; `shared`: one b for the whole batch (stride 0).
    The bound of the tests above: K + 2 roundings of fp32 on the sum of magnitudes, half an ulp of the stored type."""
    import ctypes as C

    import torch

    from axiom_amd import capi

    g = axo.PCG64(M + 3 * N + K + batch)
    nb = 1 if shared else batch
    half_ulp = {F32: 0.0, F16: 2.0**-11, BF16: 2.0**-8}[dtype]
    td = {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[dtype]
    da = gh.to_dev(g.normal((batch, M, K)).astype(np.float32)).to(td)
    db = gh.to_dev((g.normal((nb, K, N) if nn else (nb, N, K)) / np.sqrt(K)).astype(np.float32)).to(td)
    bias, res = gh.to_dev((g.normal((N,)) * 0.1).astype(np.float32)).to(td), gh.to_dev(g.normal((batch, M, N)).astype(np.float32)).to(td)
    c = torch.full((batch, M, N), float("nan"), device="cuda", dtype=td)
    p = capi.GemmParams()
    p.dtype, p.m, p.n, p.k, p.batch, p.lda, p.ldb, p.ldc, p.trans_b = dtype, M, N, K, batch, K, N if nn else K, N, int(not nn)
    p.stride_a, p.stride_b, p.stride_c = M * K, 0 if shared else K * N, M * N
    p.bias, p.residual = bias.data_ptr(), res.data_ptr()
    torch.cuda.synchronize()
    gh.sync()
    capi.check(capi.lib().axhip_gemm(da.data_ptr(), db.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    for b in range(batch):
        x, w = da[b].double(), db[0 if shared else b].double()
        w = w if nn else w.t().contiguous()
        want = x @ w + bias.double() + res[b].double()
        magnitude = x.abs() @ w.abs() + bias.double().abs() + res[b].double().abs()
        assert bool(((c[b].double() - want).abs() <= (K + 2) * 2.0**-24 * magnitude + half_ulp * want.abs() + 2.0**-24).all())


# Every tile that multiplies parts, and four products that stay with fp32 ones: k-tiles (of 32 on
# 128 x 128, of 64 on the other two rings) of every remainder by how many are on their way (three, two, three), k of every
# remainder by 4, rows and columns inside a tile, columns off the 16-byte grid (b as [k, n]: the last tile moved left)
PARTS = [(346, 2137, 98, 4, "ring_128x128_parts"), (206, 1581, 133, 8, "ring_128x128_parts"), (321, 1054, 163, 8, "ring_128x128_parts"), (2048, 2044, 225, 1, "ring_128x128_parts"),
         (51, 2093, 244, 8, "ring_64x128_parts"), (103, 1073, 289, 8, "ring_64x128_parts"), (257, 4100, 700, 1, "ring_64x128_parts"), (1000, 1028, 1090, 1, "ring_64x128_parts"),
         (817, 614, 354, 1, "ring_64x64_parts"), (291, 1665, 418, 1, "ring_64x64_parts"), (1845, 263, 493, 1, "ring_64x64_parts"), (867, 579, 628, 1, "ring_64x64_parts"),
         (300, 1280, 1285, 1, "f32_32x64_parts"), (130, 1984, 2050, 1, "f32_32x64_parts"), (21, 1071, 690, 8, "f32_32x64_parts"), (1684, 165, 547, 1, "f32_32x64_parts"),
         (1024, 1020, 1023, 1, "ring_64x64"), (513, 132, 995, 8, "ring_64x64"), (1153, 129, 256, 16, "ring_64x64"), (64, 241, 145, 32, "f32_32x64")]


@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch,kernel", PARTS)
def test_f32_products_of_parts(nn, M, N, K, batch, kernel):
    """Products by way of bf16 parts are no further from the exact ones than fp32 sums of 32 products and then one per
    32 k: (36 + K / 32) half ulps of the sum of magnitudes, for inputs of both signs, of one sign, so small that their
    last parts would be below bf16's smallest normal number, had they not been scaled, denormal ones, and some on either side of 2^112, from which
    on there are no parts."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + 3 * N + K)
    scales = {"small": (2.0**-118, 2.0**40), "denormal": (2.0**-70, 2.0**100), "large": (2.0**111, 2.0**-30)}
    for kind in ("normal", "positive", *scales):
        if kind == "denormal" and "parts" not in kernel:
            continue
        x, W = torch.empty((batch, M, K), device="cuda"), torch.empty((batch, K, N) if nn else (batch, N, K), device="cuda")
        for t in (x, W):
            t.uniform_(0.0, 1.0, generator=gen) if kind == "positive" else t.normal_(generator=gen)
        if kind in scales:
            x *= scales[kind][0]
            W *= scales[kind][1]
        if kind == "denormal":
            x *= scales[kind][0]
            assert bool((x.abs() < 2.0**-130).all()) and bool((x != 0).any())
        c = _f32_product(x, W, nn, kernel)
        for b in range(0, batch, 5):
            x64, w64 = x[b].double(), W[b].double() if nn else W[b].double().t().contiguous()
            assert bool(((c[b].double() - x64 @ w64).abs() <= min(K + 2, 36 + K / 32) * 2.0**-24 * (x64.abs() @ w64.abs())).all()), kind


@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch,kernel", PARTS)
def test_f32_products_of_parts_with_one_product_to_an_output(nn, M, N, K, batch, kernel):
    """Rows of x with a single entry: the result is one product, rounded once.  By parts the last addition rounds by half
    an ulp and the seven before it, of numbers below 2^-5 where the result is 1 or more, by 2^-30 each at most: 0.5 + 7 / 128 ulp.  Among
    random factors some whose second and third parts are as large as they get (0x1.01ffp0 squared is 2 ulp off without their products)."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + 3 * N + K)
    x, W = torch.zeros((batch, M, K), device="cuda"), torch.empty((batch, K, N) if nn else (batch, N, K), device="cuda").normal_(generator=gen)
    at = torch.randint(0, K, (batch, M, 1), device="cuda", generator=gen)
    value = torch.empty((batch, M, 1), device="cuda").normal_(generator=gen)
    hard = float.fromhex("0x1.01ffp0")
    value[:, ::3] = hard
    (W[:, :, ::3] if nn else W[:, ::3]).fill_(hard)
    x.scatter_(2, at, value)
    c = _f32_product(x, W, nn, kernel)
    for b in range(0, batch, 5):
        want = value[b].double() * (W[b].t() if not nn else W[b]).contiguous()[at[b, :, 0]].double()
        nearest = want.float().abs()
        ulp = (torch.nextafter(nearest, torch.full_like(nearest, float("inf"))) - nearest).double()
        assert bool(((c[b].double() - want).abs() <= (0.5 + 7 / 128) * ulp).all())


@pytest.mark.parametrize("again", [False, True], ids=["once", "again"])
@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch,kernel", PARTS)
def test_f32_products_of_parts_of_whole_numbers(nn, M, N, K, batch, kernel, again):
    """Whole numbers with one to three parts, sums below 2^24: exact, with bias, residual and activation, also (`again`) where a tile is
    computed a second time because one of its rows is infinite."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + 3 * N + K)
    whole = lambda shape, to: torch.randint(-to, to + 1, shape, device="cuda", generator=gen).float()
    for wide in ("x", "W"):
        x, W = whole((batch, M, K), 900 if wide == "x" else 4), whole((batch, K, N) if nn else (batch, N, K), 4 if wide == "x" else 900)
        (x if wide == "x" else W.transpose(1, 2) if nn else W)[..., 1:K:K // 3] += 2.0**17 + 1 # (at most four in each sum)
        bias, residual = whole((N,), 9), whole((batch, M, N), 9)
        if again:
            x[batch // 2, M - 1, K - 2], (W[:, K - 2] if nn else W[:, :, K - 2])[...] = float("inf"), 1.0
        c = _f32_product(x, W, nn, kernel, bias, residual, "relu")
        for b in {0, batch // 2, batch - 1}:
            want = (x[b].double() @ (W[b].double() if nn else W[b].double().t().contiguous()) + bias + residual[b]).clamp_min(0.0)
            assert bool((want[torch.isfinite(want)] < 2.0**24).all()) and bool(torch.isinf(want[M - 1]).all()) == (again and b == batch // 2)
            assert bool((c[b].double() == want).all()), (wide, b)


@pytest.mark.parametrize("nn", [False, True], ids=["nt", "nn"])
@pytest.mark.parametrize("M,N,K,batch,kernel", PARTS)
def test_f32_products_of_parts_that_are_not_finite(nn, M, N, K, batch, kernel):
    """Infinities, NaN and numbers near the largest, whose parts have none: the same places of the result are infinite or NaN as in
    float64, and everything else keeps its bound, in the tiles that are computed again and in the others."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + 3 * N + K)
    x, W = torch.empty((batch, M, K), device="cuda").normal_(generator=gen), torch.empty((batch, K, N) if nn else (batch, N, K), device="cuda").normal_(generator=gen)
    last = batch - 1
    x[0, 3, 5], x[last, M - 1, K - 1], x[0, min(40, M - 2), :] = float("inf"), float("nan"), 3.0e38
    W[0] = W[0].abs() * 2.0**-20
    W[last, 0, 0] = -float("inf") if batch > 1 else W[last, 0, 0]
    c = _f32_product(x, W, nn, kernel)
    for b in {0, last // 2, last}:
        x64, w64 = x[b].double(), W[b].double() if nn else W[b].double().t().contiguous()
        want = x64 @ w64
        finite = torch.isfinite(want) & (want.abs() < 3.0e38)
        beyond = want.abs() > 3.5e38
        assert bool((torch.isnan(c[b]) == torch.isnan(want)).all())
        assert bool((c[b][beyond].double() == torch.sign(want[beyond]) * float("inf")).all())
        bound = min(K + 2, 36 + K / 32) * 2.0**-24 * torch.nan_to_num(x64, nan=0.0, posinf=0.0).abs() @ torch.nan_to_num(w64, neginf=0.0).abs()
        assert bool(((c[b].double() - want).abs() <= bound)[finite].all())


def _f32_product(x, W, nn, kernel, bias=None, residual=None, act=None):
    import ctypes as C

    import torch

    from axiom_amd import capi

    batch, M, K = x.shape
    N = W.shape[2] if nn else W.shape[1]
    c = torch.full((batch, M, N), 7.0, device="cuda")
    p = capi.GemmParams()
    p.dtype, p.m, p.n, p.k, p.batch, p.lda, p.ldb, p.ldc, p.trans_b = F32, M, N, K, batch, K, N if nn else K, N, int(not nn)
    p.stride_a, p.stride_b, p.stride_c = M * K, K * N, M * N
    p.bias, p.residual, p.epilogue_op = None if bias is None else bias.data_ptr(), None if residual is None else residual.data_ptr(), 0 if act is None else capi.OP[act]
    torch.cuda.synchronize()
    gh.sync()
    capi.check(capi.lib().axhip_gemm(x.data_ptr(), W.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    assert capi.lib().axhip_gemm_last_kernel() == kernel.encode()
    return c
