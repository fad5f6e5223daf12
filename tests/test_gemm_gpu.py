"""GPU parity of the MFMA GEMM family (MatMul, BatchMatMul, fused epilogues, int8) against the
CPU oracle, through the C ABI.

Inputs are scaled so outputs are O(1); fp32 must agree to 1e-4 (accumulation order only),
fp16 to 4e-3 and bf16 to 3e-2 max-abs (one storage rounding of an O(1..4) value); int8
accumulators are compared bit-exactly against an integer brute force.
"""
import ctypes

import numpy as np
import pytest
import torch

from helpers import ALL_DTYPES, TORCH_DTYPES, TTMI_DTYPES, dev, host, max_abs, ok, ptr, rounded, stream
from turbotransformers_amd import capi

pytestmark = pytest.mark.gpu

GEMM_TOL = {"f32": 1e-4, "f16": 4e-3, "bf16": 3e-2}


def _ab(rng, M, N, K, b_trans):
    A = rng.standard_normal((M, K), np.float32)
    B = (rng.standard_normal((N, K) if b_trans else (K, N), np.float32) / np.sqrt(K)).astype(np.float32)
    return A, B


def test_matmul_known_answer(ttmi):
    # layers/kernels/mat_mul_test.cpp:29-40: [1,2;3,4] x [2,3;4,5] = [10,13;22,29]
    A, B = np.array([[1, 2], [3, 4]], np.float32), np.array([[2, 3], [4, 5]], np.float32)
    for dt in ALL_DTYPES:
        C = torch.zeros((2, 2), dtype=dev(A, dt).dtype, device="cuda")
        ok(ttmi.ttmi_gemm(ptr(dev(A, dt)), ptr(dev(B, dt)), ptr(C), 2, 2, 2, 2, 2, 2, 0, 1.0, 0.0, TTMI_DTYPES[dt], stream()))
        assert np.array_equal(host(C), np.array([[10, 13], [22, 29]], np.float32))
        ok(ttmi.ttmi_gemm(ptr(dev(A, dt)), ptr(dev(np.ascontiguousarray(B.T), dt)), ptr(C), 2, 2, 2, 2, 2, 2, 1, 1.0, 0.0,
                          TTMI_DTYPES[dt], stream()))
        assert np.array_equal(host(C), np.array([[10, 13], [22, 29]], np.float32))


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("b_trans", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (5, 768, 768), (20, 3072, 768), (20, 768, 3072), (128, 2304, 768), (300, 256, 64), (257, 129, 72),
    (33, 65, 50), (1, 8, 8), (2048, 2304, 768), (8192, 2304, 768), (4100, 1024, 1024), (500, 500, 500)])
def test_matmul(ttmi, oracle, dt, b_trans, M, N, K):
    rng = np.random.default_rng(M + N + K + b_trans)
    A, B = _ab(rng, M, N, K, b_trans)
    dA, dB = dev(A, dt), dev(B, dt)
    C = torch.full((M, N), 3.0, dtype=dA.dtype, device="cuda")
    ok(ttmi.ttmi_gemm(ptr(dA), ptr(dB), ptr(C), M, N, K, K, K if b_trans else N, N, b_trans, 1.0, 0.0,
                      TTMI_DTYPES[dt], stream()))
    want = oracle.matmul(rounded(A, dt), rounded(B, dt), bool(b_trans))
    assert max_abs(host(C), want) <= GEMM_TOL[dt]


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,K", [(128, 768, 3072), (128, 768, 768), (1, 768, 3072), (100, 2304, 768), (200, 3072, 1024),
                                   (64, 520, 4096), (2560, 768, 3072), (2048, 768, 3072), (1000, 1024, 4096)])
def test_matmul_small_m_long_k(ttmi, oracle, dt, M, N, K):
    """Few output tiles, long K: the split-K path (K slices summed in a fixed order by a second kernel).
    Same bound as any other MatMul, and two runs give the same bits."""
    rng = np.random.default_rng(M + N + K)
    A, B = _ab(rng, M, N, K, 1)
    dA, dB = dev(A, dt), dev(B, dt)
    C1 = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    C2 = torch.empty_like(C1)
    for C in (C1, C2):
        ok(ttmi.ttmi_gemm(ptr(dA), ptr(dB), ptr(C), M, N, K, K, K, N, 1, 1.0, 0.0, TTMI_DTYPES[dt], stream()))
    want = oracle.matmul(rounded(A, dt), rounded(B, dt), True)
    assert max_abs(host(C1), want) <= GEMM_TOL[dt] * max(1.0, float(np.abs(want).max()))
    assert torch.equal(C1, C2)


@pytest.mark.parametrize("dt", ALL_DTYPES)
def test_fused_epilogues_small_m_long_k(ttmi, oracle, dt):
    """bias + GELU and bias + residual through the split-K reduction kernel."""
    import ctypes
    rng = np.random.default_rng(5)
    M, N, K = 96, 768, 3072
    A, W = _ab(rng, M, N, K, 1)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    dA, dW, db, dres = dev(A, dt), dev(W, dt), dev(bias, dt), dev(res, dt)
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    C = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_ACT,
                            ctypes.byref(_epi(bias=db, act=capi.ACT_GELU)), TTMI_DTYPES[dt], stream()))
    assert max_abs(host(C), oracle.add_bias_act(base, rounded(bias, dt), 0)) <= GEMM_TOL[dt] * 3
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_RESIDUAL,
                            ctypes.byref(_epi(bias=db, residual=dres)), TTMI_DTYPES[dt], stream()))
    assert max_abs(host(C), base + rounded(bias, dt) + rounded(res, dt)) <= GEMM_TOL[dt] * 3


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (33, 72, 128), (65, 200, 192), (127, 520, 768), (700, 1544, 256), (1400, 3072, 768),
                                   (2000, 768, 768), (2560, 776, 320), (2500, 3072, 192), (260, 768, 3072)])
def test_ring_kernel_epilogues_on_ragged_tiles(ttmi, oracle, dt, M, N, K):
    """The deep-ring tiles behind bias, bias + residual, bias + ReLU and fp32 output: fewer K steps than ring stages, rows and
    columns past the last whole tile of every width, whole and K-sliced products.  Rows past M stay untouched."""
    import ctypes
    if K * (4 if dt == "f32" else 2) % 128:
        pytest.skip("K is no whole number of 128-byte steps")
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    dA, dW, db, dres = dev(A, dt), dev(W, dt), dev(bias, dt), dev(res, dt)
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True) + rounded(bias, dt)
    for epi, args, want in ((capi.EPI_BIAS, _epi(bias=db), base), (capi.EPI_BIAS_ACT, _epi(bias=db, act=capi.ACT_RELU), np.maximum(base, 0)),
                            (capi.EPI_BIAS_RESIDUAL, _epi(bias=db, residual=dres), base + rounded(res, dt)),
                            (capi.EPI_F32_OUT, _epi(bias=db), base)):
        C = torch.full((M + 40, N), -7.0, dtype=torch.float32 if epi == capi.EPI_F32_OUT else dA.dtype, device="cuda")
        ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, epi, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
        assert max_abs(host(C[:M]), want) <= GEMM_TOL[dt] * 3
        assert torch.all(C[M:] == -7.0)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,K,offset", [(10, 2, 768, 0), (128, 772, 3072, 0), (300, 1541, 768, 0), (2560, 772, 3072, 0), (9000, 1002, 256, 0),
                                          (40, 768, 1536, 1), (128, 3072, 768, 1), (2000, 768, 1024, 1), (8200, 768, 256, 1)])
def test_fused_products_that_the_ring_tiles_refuse(ttmi, dt, M, N, K, offset):
    """Widths that are no multiple of eight, and biases, residuals and outputs off the 16-byte grid: few rows, the wavefront
    kernel, K slices, the DMA tiles of every size.  Rows past M stay untouched."""
    import ctypes
    g = torch.Generator(device="cuda").manual_seed(M + N)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    off = lambda t: torch.cat([t.new_full((offset,), -7.0), t.flatten()])[offset:].view(t.shape)
    A, W = rand(M, K).to(TORCH_DTYPES[dt]), (rand(N, K) / K ** 0.5).to(TORCH_DTYPES[dt])
    bias, res = off(rand(N).to(A.dtype)), off(rand(M, N).to(A.dtype))
    base = (A.double() @ W.double().T + bias.double())
    for epi, args, want in ((capi.EPI_BIAS, _epi(bias=bias), base), (capi.EPI_BIAS_ACT, _epi(bias=bias, act=capi.ACT_RELU), base.relu()),
                            (capi.EPI_BIAS_ACT, _epi(bias=bias, act=capi.ACT_GELU), torch.nn.functional.gelu(base, approximate="tanh")),
                            (capi.EPI_BIAS_RESIDUAL, _epi(bias=bias, residual=res), base + res.double()),
                            (capi.EPI_F32_OUT, _epi(bias=bias), base)):
        C = off(torch.full((M + 40, N), -7.0, dtype=torch.float32 if epi == capi.EPI_F32_OUT else A.dtype, device="cuda"))
        ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(W), ptr(C), M, N, K, K, K, N, epi, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
        assert float((C[:M].double() - want).abs().max()) <= GEMM_TOL[dt] * 3
        assert torch.all(C[M:] == -7.0)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,steps", [(1, 8, 1), (16, 24, 16), (17, 776, 17), (33, 768, 24), (32, 3072, 12), (10, 768, 33), (64, 136, 96),
                                       (160, 768, 12)])
def test_few_row_kernel_epilogues(ttmi, oracle, dt, M, N, steps):
    """The form for few rows (sixteen wavefronts divide K): shares of no, one, two and more K steps of 128 bytes, one and two blocks
    of rows, ragged rows and columns, every epilogue.  Rows past M stay untouched."""
    import ctypes
    K = steps * (32 if dt == "f32" else 64)
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    dA, dW, db, dres = dev(A, dt), dev(W, dt), dev(bias, dt), dev(res, dt)
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True) + rounded(bias, dt)
    for epi, args, want in ((capi.EPI_BIAS, _epi(bias=db), base), (capi.EPI_BIAS_ACT, _epi(bias=db, act=capi.ACT_RELU), np.maximum(base, 0)),
                            (capi.EPI_BIAS_RESIDUAL, _epi(bias=db, residual=dres), base + rounded(res, dt)),
                            (capi.EPI_F32_OUT, _epi(bias=db), base)):
        C = torch.full((M + 40, N), -7.0, dtype=torch.float32 if epi == capi.EPI_F32_OUT else dA.dtype, device="cuda")
        ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, epi, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
        assert max_abs(host(C[:M]), want) <= GEMM_TOL[dt] * 3
        assert torch.all(C[M:] == -7.0)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("B,S,h", [(1, 1, 12), (3, 5, 12), (1, 37, 16), (9, 31, 12), (7, 130, 12), (2, 387, 16)])
def test_ring_kernel_head_split(ttmi, oracle, dt, v_transposed, B, S, h):
    """The same tiles behind the QKV projection: sequences shorter than a group of rows and off its grid, V row-major and
    transposed (four or eight rows a store), hidden sizes whose V third starts inside and on a wavefront's columns."""
    import ctypes
    d, H = 64, h * 64
    rng = np.random.default_rng(S + h)
    A, W = _ab(rng, B * S, 3 * H, H, 1)
    bias = rng.standard_normal(3 * H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    pitch = (S + 7) // 8 * 8 if v_transposed else 0
    q, k = (torch.full((B, h, S, d), float("nan"), dtype=dA.dtype, device="cuda") for _ in range(2))
    v = torch.full((B, h, d, pitch) if v_transposed else (B, h, S, d), 7.0, dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, B * S, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    want = oracle.split_add_bias_transpose(oracle.matmul(rounded(A, dt), rounded(W, dt), True), rounded(bias, dt), B, S, h, d)
    got_v = host(v)
    if v_transposed:
        assert np.all(got_v[..., S:] == 7.0)
        got_v = got_v[..., :S].transpose(0, 1, 3, 2)
    for got, w in zip((host(q), host(k), got_v), want):
        assert max_abs(got, w) <= GEMM_TOL[dt] * 2


@pytest.fixture(params=["3 A stages", "2 A stages"])
def large_tile_forced(request, ttmi):
    """Switch TTMI_LARGE_TILE = 1 sends every eligible problem to the one-wavefront-per-SIMD kernel whatever its
    size (set through the C ABI: the library reads its environment variables only once).  Both forms of its K loop:
    three LDS stages for the A operand where they fit (192-wide tiles, row-major outputs), and two everywhere."""
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", 1))
    if request.param == "2 A stages":
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_W4_A_STAGES", 2))
    yield
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", -1))
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_W4_A_STAGES", -1))


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(256, 192, 128), (1, 8, 128), (300, 200, 256), (777, 776, 384), (2560, 768, 768),
                                   (515, 3072, 256), (4100, 1000, 128), (64, 2304, 768)])
def test_large_tile_kernel_against_oracle_and_small_tiles(ttmi, oracle, large_tile_forced, dt, M, N, K):
    """The 256 x 192 tile kernel (four wavefronts, accumulators in AGPRs) on whole, ragged and tiny problems: plain
    product, bias, bias + GELU.  Bound as for any MatMul against the oracle; against the 8-wavefront kernels the
    plain and the bias form may differ by the last bit of the output type and no more (the 16x16x32 matrix instruction
    sums the 32 products of a step in another order than the 32x32x16 one: fp32 rounding of the accumulator)."""
    import ctypes
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)

    def run(epilogue):
        C = torch.full((M, N), float("nan"), dtype=dA.dtype, device="cuda")
        if epilogue is None:
            ok(ttmi.ttmi_gemm(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, 1, 1.0, 0.0, TTMI_DTYPES[dt], stream()))
        elif epilogue == "bias":
            ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS, ctypes.byref(_epi(bias=db)),
                                    TTMI_DTYPES[dt], stream()))
        else:
            ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_ACT,
                                    ctypes.byref(_epi(bias=db, act=capi.ACT_GELU)), TTMI_DTYPES[dt], stream()))
        torch.cuda.synchronize()
        return C

    got = {e: run(e) for e in (None, "bias", "gelu")}
    assert max_abs(host(got[None]), base) <= GEMM_TOL[dt]
    assert max_abs(host(got["bias"]), base + rounded(bias, dt)) <= GEMM_TOL[dt] * 3
    assert max_abs(host(got["gelu"]), oracle.add_bias_act(base, rounded(bias, dt), 0)) <= GEMM_TOL[dt] * 3
    if (M, N, K) != (64, 2304, 768):  # that one is cut along K by the other path: another summation order
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", 0))
        ulp = 2.0 ** -10 if dt == "f16" else 2.0 ** -7  # one step of the output type, relative to the larger neighbour
        for form in (None, "bias"):
            a, b = host(run(form)), host(got[form])
            assert np.all(np.abs(a - b) <= ulp * np.maximum(np.abs(a), np.abs(b)) + 1e-6)
            assert np.mean(a != b) < 0.05  # and the two mostly agree exactly


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("M", [1, 300, 777, 4100])
def test_large_tile_kernel_leaves_rows_past_m_alone(ttmi, oracle, large_tile_forced, dt, M):
    """The last tile row of the 256-row tiles is ragged for every one of these M.  C lives inside a larger tensor
    with 256 sentinel rows behind row M (and 8 in front of row 0): the kernel's row-major stores, plain, bias and
    bias + GELU, must leave every sentinel as it was, and rows 0..M-1 must still be the product."""
    import ctypes
    N, K, GUARD = 776, 256, 256
    rng = np.random.default_rng(M)
    A, W = _ab(rng, M, N, K, 1)
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = {"plain": base, "bias": base + rounded(bias, dt), "gelu": oracle.add_bias_act(base, rounded(bias, dt), 0)}
    SENTINEL = -7.0
    for form in ("plain", "bias", "gelu"):
        whole = torch.full((8 + M + GUARD, N), SENTINEL, dtype=dA.dtype, device="cuda")
        C = whole[8:8 + M]
        if form == "plain":
            ok(ttmi.ttmi_gemm(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, 1, 1.0, 0.0, TTMI_DTYPES[dt], stream()))
        else:
            epi = _epi(bias=db) if form == "bias" else _epi(bias=db, act=capi.ACT_GELU)
            ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N,
                                    capi.EPI_BIAS if form == "bias" else capi.EPI_BIAS_ACT, ctypes.byref(epi),
                                    TTMI_DTYPES[dt], stream()))
        torch.cuda.synchronize()
        assert torch.all(whole[:8] == SENTINEL), form
        assert torch.all(whole[8 + M:] == SENTINEL), "%s: rows past M were written" % form
        assert max_abs(host(C), want[form]) <= GEMM_TOL[dt] * 3


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("B,S,h,d", [(2, 40, 12, 64), (16, 128, 12, 64), (3, 100, 6, 64), (2, 300, 16, 64), (64, 32, 12, 64),
                                     (20, 512, 16, 64), (7, 75, 12, 64), (6, 100, 12, 64)])
def test_large_tile_kernel_qkv_split(ttmi, oracle, large_tile_forced, dt, B, S, h, d, v_transposed):
    """The same kernel behind the QKV projection: bias + head split, V row-major or transposed (those tiles run with
    the matrix operands unswapped and leave through the strip column-wise).  Sequence lengths that are and are not
    multiples of 8 and of 32 (eight rows of one V^T store, the 32 rows of a staged group, may straddle two sequences;
    a group of eight positions inside a sequence of a length off the 8-grid is one element-aligned 16-byte store),
    hidden sizes whose V third does and does not start on a multiple of the tile width (then the tile in front of it
    is cut short and a new run of tiles starts there)."""
    import ctypes
    rng = np.random.default_rng(S + h)
    H = h * d
    A, W = _ab(rng, B * S, 3 * H, H, 1)
    bias = rng.standard_normal(3 * H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    q, k, v = (torch.full((B, h, S, d), float("nan"), dtype=dA.dtype, device="cuda") for _ in range(3))
    pitch = (S + 7) // 8 * 8 + 8 if v_transposed else 0
    if v_transposed:
        v = torch.full((B, h, d, pitch), 7.0, dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
    name = ctypes.create_string_buffer(64)
    ok(ttmi.ttmi_gemm_describe(B * S, 3 * H, H, capi.EPI_QKV_SPLIT, ctypes.byref(args), TTMI_DTYPES[dt], name, 64))
    assert name.value.decode().startswith("dma_agpr4w")
    if (B, S, h) == (20, 512, 16):  # 40 x 12 tiles of 256 x 256 beat 40 x 17 of 256 x 192: the widest tile's head split
        assert name.value.decode() == "dma_agpr4w_256x256"
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, B * S, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT,
                            ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    qkv = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.split_add_bias_transpose(qkv, rounded(bias, dt), B, S, h, d)
    got_v = host(v)
    if v_transposed:
        assert np.all(got_v[..., S:] == 7.0)
        got_v = got_v[..., :S].transpose(0, 1, 3, 2)
    for got, w in zip((host(q), host(k), got_v), want):
        assert max_abs(got, w) <= GEMM_TOL[dt] * 2


LN_TOL = {"f32": 1e-4, "f16": 4e-3, "bf16": 3e-2}  # relative to 1 + |expected|; large shapes round the product to 16 bits first


def _ln_close(got, want, dt):
    return bool(np.all(np.abs(got - want) <= LN_TOL[dt] * (1.0 + np.abs(want))))


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,K", [(128, 768, 768), (128, 768, 3072), (1, 768, 3072), (2560, 768, 3072), (300, 1024, 4096),
                                   (40, 2052, 1024), (64, 4096, 1024), (64, 520, 256), (4096, 768, 768), (50, 770, 768)])
def test_gemm_bias_layer_norm(ttmi, oracle, dt, M, N, K):
    """Dense projection + AddBiasLayerNorm as one call: shapes that take the split-K kernels (normalised by
    the kernel that sums the slices), and shapes that run the two kernels one after the other."""
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    res = rng.standard_normal((M, N)).astype(np.float32)
    bias, gamma, beta = (rng.standard_normal(N).astype(np.float32) for _ in range(3))
    dA, dW, dres = dev(A, dt), dev(W, dt), dev(res, dt)
    out = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    out2 = torch.empty_like(out)
    for o in (out, out2):
        ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(dA), ptr(dW), ptr(o), ptr(dres), None, ptr(dev(bias, dt)), ptr(dev(gamma, dt)),
                                          ptr(dev(beta, dt)), None, M, N, K, 1e-12, TTMI_DTYPES[dt], stream()))
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.add_bias_layer_norm(base, rounded(res, dt), rounded(bias, dt), rounded(gamma, dt), rounded(beta, dt))
    assert _ln_close(host(out), want, dt)
    assert torch.equal(out, out2)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(128, 768, 3072), (2560, 1024, 4096), (4096, 768, 768)])
def test_gemm_bias_layer_norm_fp32_residual(ttmi, oracle, dt, M, N, K):
    """The same with the residual stream in fp32: the 16-bit output is the rounding of the fp32 one, and
    writing the fp32 result over the residual buffer is allowed."""
    rng = np.random.default_rng(M + N + K + 1)
    A, W = _ab(rng, M, N, K, 1)
    res = rng.standard_normal((M, N)).astype(np.float32)
    bias, gamma, beta = (rng.standard_normal(N).astype(np.float32) for _ in range(3))
    dA, dW, dres = dev(A, dt), dev(W, dt), dev(res)
    out = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    out32 = torch.empty((M, N), device="cuda")
    args = (ptr(dev(bias, dt)), ptr(dev(gamma, dt)), ptr(dev(beta, dt)))
    ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(dA), ptr(dW), ptr(out), None, ptr(dres), *args, ptr(out32), M, N, K, 1e-12,
                                      TTMI_DTYPES[dt], stream()))
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.add_bias_layer_norm(base, res, rounded(bias, dt), rounded(gamma, dt), rounded(beta, dt))
    assert _ln_close(host(out32), want, dt)
    assert np.array_equal(host(out), rounded(host(out32), dt))
    # with its own fp32 output buffer nothing is rounded between the accumulators and the normalisation, on the
    # K-sliced path and on the large-problem path alike: the fp32 result is as close to the oracle as an fp32 run
    assert _ln_close(host(out32), want, "f32")
    first = out32.clone()
    ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(dA), ptr(dW), ptr(out), None, ptr(dres), *args, ptr(dres), M, N, K, 1e-12,
                                      TTMI_DTYPES[dt], stream()))
    if M <= 128:
        assert torch.equal(dres, first)  # K-sliced: the same kernels either way
    else:
        # a large problem writing over its residual has nowhere to keep an fp32 product: it passes through `out`
        # in the 16-bit type, one more rounding
        assert _ln_close(host(dres), want, dt)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,slices,fp32_residual", [(6275, 768, 3072, -1, False), (6275, 768, 3072, -1, True),
                                                        (700, 384, 768, 3, False), (1, 8, 512, 2, False),
                                                        (1300, 1000, 1024, 4, True), (520, 200, 256, 2, False)])
def test_gemm_bias_layer_norm_k_slices_on_the_large_tile_kernel(ttmi, oracle, dt, M, N, K, slices, fp32_residual):
    """The projection in front of a LayerNorm cut along K on the one-wavefront-per-SIMD kernel: (slice, tile) work
    items, fp32 partial products, summed and normalised by the reduction kernel.  Forced onto small and ragged shapes
    with 2, 3 and 4 slices (switch TTMI_W4_SPLITK: the library takes this path by itself for no size), and left to the
    library's choice for the second FFN product of a 6275-token batch, which the ring tiles hold in fp32.  Against the
    oracle, and against the same call with the path switched off: both sum fp32 partial sums of the same products, in
    another order."""
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    res = rng.standard_normal((M, N)).astype(np.float32)
    bias, gamma, beta = (rng.standard_normal(N).astype(np.float32) for _ in range(3))
    dA, dW = dev(A, dt), dev(W, dt)
    dres = dev(res) if fp32_residual else dev(res, dt)
    args = (ptr(dev(bias, dt)), ptr(dev(gamma, dt)), ptr(dev(beta, dt)))
    outs = {}
    try:
        for name, value in (("sliced", slices), ("unsliced", 0)):
            ok(ttmi.ttmi_set_kernel_switch(b"TTMI_W4_SPLITK", value))
            out = torch.full((M + 8, N), -7.0, dtype=dA.dtype, device="cuda")
            out32 = torch.full((M + 8, N), -7.0, device="cuda") if fp32_residual else None
            ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(dA), ptr(dW), ptr(out), None if fp32_residual else ptr(dres),
                                              ptr(dres) if fp32_residual else None, *args,
                                              ptr(out32) if fp32_residual else None, M, N, K, 1e-12, TTMI_DTYPES[dt], stream()))
            torch.cuda.synchronize()
            assert torch.all(out[M:] == -7.0), "rows past M were written"
            outs[name] = (out[:M], out32[:M] if fp32_residual else None)
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_W4_SPLITK", -1))
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.add_bias_layer_norm(base, res if fp32_residual else rounded(res, dt), rounded(bias, dt), rounded(gamma, dt),
                                      rounded(beta, dt))
    got, got32 = outs["sliced"]
    assert _ln_close(host(got), want, dt)
    if fp32_residual:
        assert _ln_close(host(got32), want, "f32")  # nothing rounded between the accumulators and the normalisation
        assert np.array_equal(host(got), rounded(host(got32), dt))
        assert max_abs(host(got32), host(outs["unsliced"][1])) < 1e-3
    else:
        assert _ln_close(host(got), host(outs["unsliced"][0]).astype(np.float32), dt)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("static", [False, True])
@pytest.mark.parametrize("M,N,K,most", [(384, 768, 768, 7), (512, 512, 512, 9), (385, 1024, 1024, 7), (2048, 1024, 1024, 7), (6827, 768, 3072, 3),
                                        (10752, 768, 3072, 3), (5121, 1024, 4096, 3), (8192, 1024, 4096, 3)])
def test_product_in_front_of_a_layer_norm_is_held_in_fp32(ttmi, dt, static, M, N, K, most):
    """The product reaches AddBiasLayerNorm unrounded up to the sizes of fp32_product_expected in gemm_typed.h: the residual is minus
    the product rounded to 16 bits, so that what is normalised is that rounding, which a 16-bit product would not have.
    Whole numbers throughout (products below 2^16 and 2^24): the sum in front of the LayerNorm is exact."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, W = (torch.randint(0, most + 1, shape, generator=g, device="cuda").to(TORCH_DTYPES[dt]) for shape in ((M, K), (N, K)))
    product = A.float() @ W.float().T
    assert float(product.max()) < 65504 and torch.equal(product, product.round())
    residual = (-product).to(TORCH_DTYPES[dt])
    zero, one = torch.zeros(N, dtype=A.dtype, device="cuda"), torch.ones(N, dtype=A.dtype, device="cuda")
    out = torch.full((M + 8, N), -7.0, dtype=A.dtype, device="cuda")
    fn = ttmi.ttmi_gemm_bias_layer_norm_static if static else ttmi.ttmi_gemm_bias_layer_norm
    ok(fn(ptr(A), ptr(W), ptr(out), ptr(residual), None, ptr(zero), ptr(one), ptr(zero), None, M, N, K, 1e-12, TTMI_DTYPES[dt], stream()))
    x = (product + residual.float()).double()
    want = (x - x.mean(1, keepdim=True)) / (x.var(1, unbiased=False, keepdim=True) + 1e-12).sqrt()
    assert float(x.abs().max()) >= 1
    # one rounding to 16 bits of values of up to about 4, and fp32 sums of squares of numbers of one or two digits
    assert float((out[:M].double() - want).abs().max()) <= GEMM_TOL[dt]
    assert torch.all(out[M:] == -7.0)


def test_captured_product_survives_larger_ones_on_its_stream(ttmi):
    """The workspace of a stream does not move: a product in K slices is captured, then the same stream runs the largest
    product that is held in fp32 (32 MiB of workspace), and every replay still equals the eager result."""
    M, N, K = 128, 768, 3072
    g = torch.Generator(device="cuda").manual_seed(0)
    new = lambda *shape: torch.randn(shape, generator=g, device="cuda").half()
    A, W, res, bias, gamma, beta = new(M, K), new(N, K) / 55, new(M, N), new(N), new(N), new(N)
    big = [new(8192, 4096), new(1024, 4096) / 64, new(8192, 1024), new(1024), new(1024), new(1024)]
    out, want, big_out = torch.zeros_like(res), torch.zeros_like(res), torch.zeros_like(big[2])
    side = torch.cuda.Stream()

    def call(dst, ops, m, n, k):
        a, w, r, b, ga, be = ops
        ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(a), ptr(w), ptr(dst), ptr(r), None, ptr(b), ptr(ga), ptr(be), None, m, n, k, 1e-12,
                                          TTMI_DTYPES["f16"], stream()))

    small = (A, W, res, bias, gamma, beta)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(out, small, M, N, K)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(out, small, M, N, K)
    for turn in range(3):
        A.copy_(new(M, K))
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            call(big_out, big, 8192, 1024, 4096)
            call(want, small, M, N, K)
        torch.cuda.synchronize()
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert not torch.isnan(want).any() and torch.equal(out, want), "replay %d" % turn


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("forced", [False, True])
@pytest.mark.parametrize("M,N,K,with_bias", [(300, 200, 256, True), (4100, 1024, 1024, False), (2560, 768, 3072, True),
                                             (8192, 768, 768, True), (777, 776, 384, False), (128, 768, 3072, True)])
def test_gemm_with_fp32_output(ttmi, oracle, dt, forced, M, N, K, with_bias):
    """TTMI_EPI_F32_OUT: 16-bit operands, the accumulators (plus an optional bias) stored as fp32.  Tile kernels of
    every family (small tiles, K slices, the 8-wavefront DMA tiles, the one-wavefront-per-SIMD kernel with whole and
    ragged tiles, also forced onto small shapes): the result is the fp32 product of the rounded operands, to fp32
    accumulation error, and rows past M stay untouched."""
    import ctypes
    rng = np.random.default_rng(M + N + K)
    A, W = _ab(rng, M, N, K, 1)
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    whole = torch.full((M + 64, N), -7.0, device="cuda")
    C = whole[:M]
    if forced:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", 1))
    try:
        ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_F32_OUT,
                                ctypes.byref(_epi(bias=db) if with_bias else _epi()), TTMI_DTYPES[dt], stream()))
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", -1))
    want = oracle.matmul(rounded(A, dt), rounded(W, dt), True) + (rounded(bias, dt) if with_bias else 0.0)
    assert max_abs(host(C), want) <= GEMM_TOL["f32"] * max(1.0, float(np.abs(want).max()))
    assert torch.all(whole[M:] == -7.0)


def test_gemm_bias_layer_norm_rejects_bad_arguments(ttmi):
    x = torch.zeros((8, 8), device="cuda")
    v = torch.zeros(8, device="cuda")
    # no residual at all; fp32 residual without its output
    assert ttmi.ttmi_gemm_bias_layer_norm(ptr(x), ptr(x), ptr(x), None, None, ptr(v), ptr(v), ptr(v), None, 8, 8, 8, 1e-12,
                                          TTMI_DTYPES["f32"], stream()) != 0
    assert ttmi.ttmi_gemm_bias_layer_norm(ptr(x), ptr(x), ptr(x), None, ptr(x), ptr(v), ptr(v), ptr(v), None, 8, 8, 8, 1e-12,
                                          TTMI_DTYPES["f32"], stream()) != 0


@pytest.mark.parametrize("dt", ALL_DTYPES)
def test_matmul_alpha_beta_and_ld(ttmi, oracle, dt):
    rng = np.random.default_rng(5)
    M, N, K, lda, ldb, ldc = 70, 90, 64, 80, 72, 96
    A = rng.standard_normal((M, lda), np.float32)
    B = (rng.standard_normal((N, ldb), np.float32) / 8).astype(np.float32)
    C0 = rng.standard_normal((M, ldc), np.float32)
    dC = dev(C0, dt)
    ok(ttmi.ttmi_gemm(ptr(dev(A, dt)), ptr(dev(B, dt)), ptr(dC), M, N, K, lda, ldb, ldc, 1, 0.5, 2.0, TTMI_DTYPES[dt],
                      stream()))
    want = rounded(C0, dt).copy()
    want[:, :N] = 0.5 * (rounded(A, dt)[:, :K].astype(np.float64) @ rounded(B, dt)[:, :K].T.astype(np.float64)) + 2.0 * want[:, :N]
    got = host(dC)
    assert max_abs(got[:, :N], want[:, :N]) <= GEMM_TOL[dt] * 3
    assert np.array_equal(got[:, N:], rounded(C0, dt)[:, N:])  # columns beyond N untouched


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("batch,S,d", [(24, 100, 64), (6, 500, 64), (4, 128, 64), (3, 37, 20)])
def test_batch_matmul_attention_shapes(ttmi, oracle, dt, batch, S, d):
    """batch_gemm3 (Q K^T, alpha = 1/sqrt(d)) and batch_gemm4 (P V) of
    layers/multi_headed_attention.cpp:328-346."""
    rng = np.random.default_rng(S)
    Q, Kt, V = (rng.standard_normal((batch, S, d), np.float32) for _ in range(3))
    alpha = 1.0 / np.sqrt(d)
    dQ, dK, dV = dev(Q, dt), dev(Kt, dt), dev(V, dt)
    score = torch.empty((batch, S, S), dtype=dQ.dtype, device="cuda")
    ok(ttmi.ttmi_gemm_strided_batched(ptr(dQ), ptr(dK), ptr(score), S, S, d, d, d, S, S * d, S * d, S * S, batch, 1,
                                      alpha, 0.0, TTMI_DTYPES[dt], stream()))
    want = oracle.batch_matmul(rounded(Q, dt), rounded(Kt, dt), True, alpha)
    assert max_abs(host(score), want) <= GEMM_TOL[dt] * 4
    P = (rng.random((batch, S, S), np.float32) / S * 2).astype(np.float32)
    dP = dev(P, dt)
    ctx = torch.empty((batch, S, d), dtype=dQ.dtype, device="cuda")
    ok(ttmi.ttmi_gemm_strided_batched(ptr(dP), ptr(dV), ptr(ctx), S, d, S, S, d, d, S * S, S * d, S * d, batch, 0, 1.0,
                                      0.0, TTMI_DTYPES[dt], stream()))
    want = oracle.batch_matmul(rounded(P, dt), rounded(V, dt), False)
    assert max_abs(host(ctx), want) <= GEMM_TOL[dt]


@pytest.mark.parametrize("dt", ALL_DTYPES)
def test_batched_heads_writes_merged_layout(ttmi, oracle, dt):
    """P V with the [B,h,S,d] -> [B,S,h,d] transpose folded into the store."""
    rng = np.random.default_rng(9)
    B, h, S, d = 2, 3, 50, 64
    P = (rng.random((B, h, S, S), np.float32) / S * 2).astype(np.float32)
    V = rng.standard_normal((B, h, S, d), np.float32)
    dP, dV = dev(P, dt), dev(V, dt)
    out = torch.empty((B, S, h, d), dtype=dP.dtype, device="cuda")
    ok(ttmi.ttmi_gemm_batched_heads(ptr(dP), ptr(dV), ptr(out), S, d, S, S, d, h * d, h, h * S * S, S * S, h * S * d,
                                    S * d, S * h * d, d, B, 0, 1.0, 0.0, TTMI_DTYPES[dt], stream()))
    want = oracle.transpose_for_score(oracle.batch_matmul(rounded(P, dt), rounded(V, dt), False))
    assert max_abs(host(out), want) <= GEMM_TOL[dt]


def _epi(**kw):
    a = capi.EpilogueArgs()
    for k, v in kw.items():
        setattr(a, k, v.data_ptr() if isinstance(v, torch.Tensor) else v)
    return a


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,N,K", [(100, 3072, 768), (4096, 3072, 768), (77, 768, 3072)])
def test_fused_bias_gelu(ttmi, oracle, dt, M, N, K):
    import ctypes
    rng = np.random.default_rng(M)
    A, W = _ab(rng, M, N, K, 1)
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    C = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, act=capi.ACT_GELU)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_ACT, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    want = oracle.add_bias_act(oracle.matmul(rounded(A, dt), rounded(W, dt), True), rounded(bias, dt), 0)
    assert max_abs(host(C), want) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("dt", ALL_DTYPES)
def test_fused_bias_and_bias_residual(ttmi, oracle, dt):
    import ctypes
    rng = np.random.default_rng(11)
    M, N, K = 300, 768, 768
    A, W = _ab(rng, M, N, K, 1)
    bias = rng.standard_normal(N).astype(np.float32)
    res = rng.standard_normal((M, N), np.float32)
    dA, dW, db, dres = dev(A, dt), dev(W, dt), dev(bias, dt), dev(res, dt)
    C = torch.empty((M, N), dtype=dA.dtype, device="cuda")
    base = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    args = _epi(bias=db)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    assert max_abs(host(C), base + rounded(bias, dt)) <= GEMM_TOL[dt] * 2
    args = _epi(bias=db, residual=dres)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_RESIDUAL, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    assert max_abs(host(C), base + rounded(bias, dt) + rounded(res, dt)) <= GEMM_TOL[dt] * 3


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("B,S,h,d", [(2, 40, 12, 64), (16, 128, 12, 64), (3, 7, 2, 32), (2, 300, 16, 64), (5, 13, 3, 64),
                                     (20, 100, 12, 64), (6, 60, 12, 64), (4, 27, 2, 64), (300, 5, 12, 64)])  # the last four: lengths off the 8-grid
def test_fused_qkv_split(ttmi, oracle, dt, B, S, h, d, v_transposed):
    """QKV GEMM + SplitAddBiasTransposeForScore; with v_seq_pitch the V third lands transposed,
    [B,h,d,pitch] (pad columns untouched), everything else as before."""
    import ctypes
    rng = np.random.default_rng(S)
    H = h * d
    A, W = _ab(rng, B * S, 3 * H, H, 1)
    bias = rng.standard_normal(3 * H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    q, k, v = (torch.empty((B, h, S, d), dtype=dA.dtype, device="cuda") for _ in range(3))
    pitch = (S + 7) // 8 * 8 + 8 if v_transposed else 0
    if v_transposed:
        v = torch.full((B, h, d, pitch), 7.0, dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, B * S, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT,
                            ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    qkv = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.split_add_bias_transpose(qkv, rounded(bias, dt), B, S, h, d)
    got_v = host(v)
    if v_transposed:
        assert np.all(got_v[..., S:] == 7.0)
        got_v = got_v[..., :S].transpose(0, 1, 3, 2)
    for got, w in zip((host(q), host(k), got_v), want):
        assert max_abs(got, w) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("B,S,h,d", [(2, 11, 4, 64), (3, 128, 12, 64), (2, 5, 3, 20)])
def test_fused_single_projection_to_heads(ttmi, oracle, dt, B, S, h, d):
    """MatMul + AddBiasTransposeForScore of one projection (context attention, multi_headed_attention.cpp:73-88)
    as the one-output case of the QKV epilogue: N = h*d, only q is written."""
    import ctypes
    rng = np.random.default_rng(S * 7)
    H = h * d
    A, W = _ab(rng, B * S, H, H, 1)
    bias = rng.standard_normal(H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    q = torch.empty((B, h, S, d), dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, q=q, seq=S, heads=h, head_dim=d)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, B * S, H, H, H, H, H, capi.EPI_QKV_SPLIT, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    proj = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.add_bias_transpose_for_score(proj, rounded(bias, dt), B, S, h, d)
    assert max_abs(host(q), want) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("B,S,h,d", [(1, 1, 2, 64), (2, 11, 3, 64), (8, 100, 12, 64), (33, 200, 12, 64), (2, 5, 3, 20)])
def test_fused_two_projections_to_heads(ttmi, oracle, dt, B, S, h, d):
    """Keys and values of one memory: N = 2*h*d, q and k are written, nothing past them."""
    import ctypes
    rng = np.random.default_rng(S * 7 + h)
    H = h * d
    A, W = _ab(rng, B * S, 2 * H, H, 1)
    bias = rng.standard_normal(2 * H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    q, k = (torch.full((B + 1, h, S, d), -7.0, dtype=dA.dtype, device="cuda") for _ in range(2))
    args = _epi(bias=db, q=q, k=k, seq=S, heads=h, head_dim=d)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, B * S, 2 * H, H, H, H, 2 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args),
                            TTMI_DTYPES[dt], stream()))
    proj = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    for got, part in ((q, slice(0, H)), (k, slice(H, 2 * H))):
        want = oracle.add_bias_transpose_for_score(np.ascontiguousarray(proj[:, part]), rounded(bias, dt)[part], B, S, h, d)
        assert max_abs(host(got[:B]), want) <= GEMM_TOL[dt] * 2
        assert torch.all(got[B] == -7.0)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("lens", [[9, 30, 1, 17], [64, 8, 200, 16, 33]])
def test_fused_qkv_split_pad(ttmi, oracle, dt, lens, v_transposed):
    import ctypes
    rng = np.random.default_rng(21)
    lens = np.array(lens, np.int64)
    h, d = 4, 64
    H, B, maxS, total = h * d, len(lens), int(lens.max()), int(lens.sum())
    A, W = _ab(rng, total, 3 * H, H, 1)
    bias = rng.standard_normal(3 * H).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    cu = np.zeros(B + 1, np.int32)
    cu[1:] = np.cumsum(lens)
    rows = torch.empty(total, dtype=torch.int32, device="cuda")
    ok(ttmi.ttmi_build_token_rows(ptr(dev(cu)), B, maxS, total, ptr(rows), stream()))
    q, k, v = (torch.zeros((B, h, maxS, d), dtype=dA.dtype, device="cuda") for _ in range(3))
    pitch = (maxS + 7) // 8 * 8 if v_transposed else 0
    if v_transposed:
        v = torch.zeros((B, h, d, pitch), dtype=dA.dtype, device="cuda")
    args = _epi(bias=db, q=q, k=k, v=v, seq=maxS, heads=h, head_dim=d, token_rows=rows, batch=B, v_seq_pitch=pitch)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, total, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT_PAD,
                            ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    qkv = oracle.matmul(rounded(A, dt), rounded(W, dt), True)
    want = oracle.split_add_bias_transpose_pad(qkv, rounded(bias, dt), lens, h, d)
    got_v = host(v)
    if v_transposed:
        got_v = got_v[..., :maxS].transpose(0, 1, 3, 2)
    for got, w in zip((host(q), host(k), got_v), want):
        assert max_abs(got, w) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("M,N,K", [(20, 768, 768), (2560, 3072, 768), (2560, 768, 3072), (33, 48, 80), (300, 1000, 130)])
def test_gemm_i8_accumulators_bit_exact(ttmi, oracle, M, N, K):
    rng = np.random.default_rng(K)
    A = rng.integers(-127, 128, (M, K)).astype(np.int8)
    B = rng.integers(-127, 128, (N, K)).astype(np.int8)
    C = torch.empty((M, N), dtype=torch.int32, device="cuda")
    ok(ttmi.ttmi_gemm_i8(ptr(dev(A)), ptr(dev(B)), ptr(C), M, N, K, K, K, N, stream()))
    want = A.astype(np.int32) @ B.astype(np.int32).T  # exact integer arithmetic
    assert np.array_equal(host(C), want)
    if M * N * K < 5e7:
        assert np.array_equal(want, oracle.gemm_i8(A, B))


@pytest.mark.parametrize("M,N,K,with_bias", [(2560, 768, 768, False), (2560, 3072, 768, True), (37, 100, 48, True), (300, 1000, 130, False)])
def test_gemm_i8_dequant_equals_unfused(ttmi, oracle, M, N, K, with_bias):
    """The dequantisation folded into the int8 GEMM gives the bits of gemm_i8 + dequant_bias, and those
    are the oracle's scheme: float(acc) * s_x * s_w[n] (+ b[n])."""
    rng = np.random.default_rng(M + N)
    a = rng.integers(-127, 128, (M, K), dtype=np.int8)
    b = rng.integers(-127, 128, (N, K), dtype=np.int8)
    sx = np.array([0.0123, 0.0], np.float32)
    sw = (rng.random(N, np.float32) + 0.5) * 1e-3
    bias = rng.standard_normal(N).astype(np.float32) if with_bias else None
    dA, dB, dsx, dsw = dev(a), dev(b), dev(sx), dev(sw)
    dbias = dev(bias) if with_bias else None
    acc = torch.empty((M, N), dtype=torch.int32, device="cuda")
    two_step, fused = torch.empty((M, N), device="cuda"), torch.empty((M, N), device="cuda")
    ok(ttmi.ttmi_gemm_i8(ptr(dA), ptr(dB), ptr(acc), M, N, K, K, K, N, stream()))
    ok(ttmi.ttmi_dequant_bias(ptr(acc), ptr(dsx), ptr(dsw), ptr(dbias) if with_bias else None, ptr(two_step), M, N, stream()))
    ok(ttmi.ttmi_gemm_i8_dequant(ptr(dA), ptr(dB), ptr(fused), ptr(dsx), ptr(dsw), ptr(dbias) if with_bias else None, -1, M, N,
                                 K, K, K, N, stream()))
    assert np.array_equal(host(fused), host(two_step))
    want = oracle.dequant_bias(oracle.gemm_i8(a, b), sx[0], sw, bias if with_bias else np.zeros(N, np.float32))
    assert max_abs(host(fused), want) <= 1e-5 * max(1.0, float(np.abs(want).max()))
    # with the activation folded in as well: the bits of the stand-alone bias + GELU kernel on the unbiased product
    if with_bias:
        ok(ttmi.ttmi_dequant_bias(ptr(acc), ptr(dsx), ptr(dsw), None, ptr(two_step), M, N, stream()))
        ok(ttmi.ttmi_add_bias_act(ptr(two_step), ptr(dbias), M, N, capi.ACT_GELU, TTMI_DTYPES["f32"], stream()))
        ok(ttmi.ttmi_gemm_i8_dequant(ptr(dA), ptr(dB), ptr(fused), ptr(dsx), ptr(dsw), ptr(dbias), capi.ACT_GELU, M, N, K, K, K,
                                     N, stream()))
        assert max_abs(host(fused), host(two_step)) <= 1e-6 * max(1.0, float(np.abs(want).max()))
        assert max_abs(host(fused), oracle.add_bias_act(want, np.zeros(N, np.float32), 0)) <= 2e-5 * max(1.0, float(np.abs(want).max()))


@pytest.mark.parametrize("B,S,h,d", [(20, 128, 12, 64), (3, 17, 2, 8), (2, 9, 3, 20)])
def test_gemm_i8_dequant_qkv_split_equals_the_two_kernels(ttmi, oracle, B, S, h, d):
    """int8 QKV projection with dequantisation, bias and head split in its store: the bits of
    ttmi_gemm_i8_dequant (no bias) followed by ttmi_split_add_bias_transpose_for_score, and the oracle's values."""
    rng = np.random.default_rng(B + S)
    H = h * d
    M, N, K = B * S, 3 * H, H if H % 16 == 0 else 48
    a = rng.integers(-127, 128, (M, K), dtype=np.int8)
    b = rng.integers(-127, 128, (N, K), dtype=np.int8)
    sx = np.array([0.0123, 0.0], np.float32)
    sw = (rng.random(N, np.float32) + 0.5) * 1e-3
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dB, dsx, dsw, dbias = dev(a), dev(b), dev(sx), dev(sw), dev(bias)
    flat = torch.empty((M, N), device="cuda")
    ok(ttmi.ttmi_gemm_i8_dequant(ptr(dA), ptr(dB), ptr(flat), ptr(dsx), ptr(dsw), None, -1, M, N, K, K, K, N, stream()))
    two = [torch.empty((B, h, S, d), device="cuda") for _ in range(3)]
    ok(ttmi.ttmi_split_add_bias_transpose_for_score(ptr(flat), ptr(dbias), ptr(two[0]), ptr(two[1]), ptr(two[2]), B, S, h, d,
                                                    TTMI_DTYPES["f32"], stream()))
    one = [torch.full((B, h, S, d), 7.0, device="cuda") for _ in range(3)]
    ok(ttmi.ttmi_gemm_i8_dequant_qkv_split(ptr(dA), ptr(dB), ptr(dsx), ptr(dsw), ptr(dbias), ptr(one[0]), ptr(one[1]), ptr(one[2]),
                                           M, N, K, K, K, S, h, d, stream()))
    for x, y in zip(one, two):
        assert torch.equal(x, y)
    want = oracle.split_add_bias_transpose(oracle.dequant_bias(oracle.gemm_i8(a, b), sx[0], sw, np.zeros(N, np.float32)), bias,
                                           B, S, h, d)
    for x, y in zip(one, want):
        assert max_abs(host(x), y) <= 1e-5 * max(1.0, float(np.abs(y).max()))


@pytest.mark.parametrize("M,N,K,act", [(2560, 3072, 768, capi.ACT_GELU), (2560, 768, 3072, -1), (200, 384, 256, capi.ACT_GELU),
                                       (777, 100, 64, -1), (40000, 64, 64, -1)])
def test_gemm_i8_dequant_leaves_the_maxima_for_the_next_quantisation(ttmi, M, N, K, act):
    """ttmi_gemm_i8_dequant_absmax: the bits of ttmi_gemm_i8_dequant in c, and, when the launch filled the slots, every
    slot written (they start as NaN here: nothing needs clearing), their maximum exactly max|c|; quantising c from the
    slots gives the bits and the scale of the two-launch quantisation.  A launch with more workgroups than slots
    says so and leaves the slots alone (see the LayerNorm form of this test for a case that does)."""
    import ctypes
    rng = np.random.default_rng(M + N)
    a = rng.integers(-127, 128, (M, K), dtype=np.int8)
    b = rng.integers(-127, 128, (N, K), dtype=np.int8)
    sx, sw = np.array([0.0123, 0.0], np.float32), (rng.random(N, np.float32) + 0.5) * 1e-3
    bias = rng.standard_normal(N).astype(np.float32)
    dA, dB, dsx, dsw, dbias = dev(a), dev(b), dev(sx), dev(sw), dev(bias)
    plain, fused = torch.empty((M, N), device="cuda"), torch.empty((M, N), device="cuda")
    slots = torch.full((capi.ABSMAX_SLOTS, ), float("nan"), device="cuda")
    written = ctypes.c_int(-1)
    ok(ttmi.ttmi_gemm_i8_dequant(ptr(dA), ptr(dB), ptr(plain), ptr(dsx), ptr(dsw), ptr(dbias), act, M, N, K, K, K, N, stream()))
    ok(ttmi.ttmi_gemm_i8_dequant_absmax(ptr(dA), ptr(dB), ptr(fused), ptr(dsx), ptr(dsw), ptr(dbias), act, M, N, K, K, K, N,
                                        ptr(slots), ctypes.byref(written), stream()))
    assert torch.equal(fused, plain)
    if written.value == 0:  # (whether a shape's launch fits the slots is the tile picker's business)
        assert torch.isnan(slots).all()
        return
    assert written.value == capi.ABSMAX_SLOTS
    assert not torch.isnan(slots).any() and float(slots.min()) >= 0.0
    assert float(slots.max()) == float(plain.abs().max())
    q1, q2 = (torch.empty((M, N), dtype=torch.int8, device="cuda") for _ in range(2))
    s1, s2 = (torch.full((capi.QUANT_SCALE_FLOATS, ), float("nan"), device="cuda") for _ in range(2))
    ok(ttmi.ttmi_quantize_rows_i8(ptr(plain), ptr(q1), ptr(s1), M, N, stream()))
    ok(ttmi.ttmi_quantize_rows_i8_from_absmax(ptr(plain), ptr(q2), ptr(s2), ptr(slots), M, N, stream()))
    assert torch.equal(q1, q2) and torch.equal(s1[:2], s2[:2])


@pytest.mark.parametrize("exponent", [-125, -119, -110, -104, -96, -95, 0, 100])
def test_quantisation_rounds_as_the_division_does(ttmi, exponent):
    """rint(x / scale) at the floats around every half-integer, for scales next to powers of two of all sizes: the shared
    reciprocal must not be used where its remainder would be a subnormal number."""
    halves = np.arange(127, dtype=np.float32) + np.float32(0.5)
    for mantissa in (1, 2, 3, 4096, (1 << 23) - 1):
        scale = np.array([((127 + exponent) << 23) | mantissa], np.uint32).view(np.float32)
        near = (halves * scale).view(np.uint32)[:, None] + np.arange(-2, 3).astype(np.uint32)
        x = np.concatenate([np.float32(127) * scale, near.reshape(-1).view(np.float32), -near.reshape(-1).view(np.float32)])
        scale = x[0] / np.float32(127)
        want = np.clip(np.rint(x / scale), -127, 127).astype(np.int8)
        q, found = torch.zeros(x.size, dtype=torch.int8, device="cuda"), torch.zeros(capi.QUANT_SCALE_FLOATS, device="cuda")
        ok(ttmi.ttmi_quantize_rows_i8(ptr(dev(x)), ptr(q), ptr(found), 1, x.size, stream()))
        assert host(found)[0] == scale
        assert np.array_equal(host(q), want)


@pytest.mark.parametrize("beside", [-3, 0, 5])
@pytest.mark.parametrize("x_off,q_off", [(0, 0), (0, 4), (1, 0), (0, 1)])
def test_quantisation_on_both_sides_of_the_write_through_line(ttmi, oracle, beside, x_off, q_off):
    """From 2 MiB of output on its stores go through L2: counts around that, tensors that start off the vector alignment, guard bytes behind."""
    n = (2 << 20) + beside
    whole_x = torch.from_numpy(np.random.default_rng(n).standard_normal(n + 8).astype(np.float32)).cuda()
    x = whole_x[x_off:x_off + n]
    whole_q = torch.full((n + 32, ), 99, dtype=torch.int8, device="cuda")
    q, scale = whole_q[q_off:q_off + n], torch.full((capi.QUANT_SCALE_FLOATS, ), float("nan"), device="cuda")
    ok(ttmi.ttmi_quantize_rows_i8(ptr(x), ptr(q), ptr(scale), 1, n, stream()))
    want, want_scale = oracle.quantize_tensor_i8(host(x).reshape(1, n))
    assert np.array_equal(host(q), want.reshape(-1)) and host(scale)[0] == np.float32(want_scale)
    assert bool((whole_q[:q_off] == 99).all()) and bool((whole_q[q_off + n:] == 99).all())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [512 * 1024, 512 * 1024 + 1, 512 * 1024 + 2044, 512 * 1024 + 2048, 513 * 1024 + 1027, (2 << 20) - 2045])
@pytest.mark.parametrize("x_off", [0, 1])
def test_quantisation_with_two_loads_a_lane(ttmi, oracle, n, x_off):
    """From 512 Ki to 2 Mi values a workgroup takes 2048 of them: counts next to the line and to whole workgroups, guard bytes behind."""
    x = torch.from_numpy(np.random.default_rng(n).standard_normal(n + 8).astype(np.float32)).cuda()[x_off:x_off + n]
    whole_q = torch.full((n + 32, ), 99, dtype=torch.int8, device="cuda")
    scale = torch.full((capi.QUANT_SCALE_FLOATS, ), float("nan"), device="cuda")
    ok(ttmi.ttmi_quantize_rows_i8(ptr(x), ptr(whole_q), ptr(scale), 1, n, stream()))
    want, want_scale = oracle.quantize_tensor_i8(host(x).reshape(1, n))
    assert np.array_equal(host(whole_q[:n]), want.reshape(-1)) and host(scale)[0] == np.float32(want_scale)
    assert bool((whole_q[n:] == 99).all())


def test_int8_linear_pipeline(ttmi, oracle):
    """quantize -> int8 GEMM -> dequant+bias, against the oracle's statement of the same scheme."""
    rng = np.random.default_rng(3)
    M, N, K = 200, 384, 256
    x = rng.standard_normal((M, K), np.float32)
    w = (rng.standard_normal((N, K), np.float32) * 0.02).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    qw, sw = oracle.quantize_weight_i8(w)
    qx_want, sx_want = oracle.quantize_tensor_i8(x)
    dq = torch.empty((M, K), dtype=torch.int8, device="cuda")
    scale = torch.full((capi.QUANT_SCALE_FLOATS, ), float("nan"), device="cuda")  # scratch needs no clearing
    ok(ttmi.ttmi_quantize_rows_i8(ptr(dev(x)), ptr(dq), ptr(scale), M, K, stream()))
    assert np.array_equal(host(dq), qx_want)
    assert host(scale)[0] == np.float32(sx_want)
    acc = torch.empty((M, N), dtype=torch.int32, device="cuda")
    ok(ttmi.ttmi_gemm_i8(ptr(dq), ptr(dev(qw)), ptr(acc), M, N, K, K, K, N, stream()))
    acc_want = oracle.gemm_i8(qx_want, qw)
    assert np.array_equal(host(acc), acc_want)
    out = torch.empty((M, N), device="cuda")
    ok(ttmi.ttmi_dequant_bias(ptr(acc), ptr(scale), ptr(dev(sw)), ptr(dev(bias)), ptr(out), M, N, stream()))
    want = oracle.dequant_bias(acc_want, sx_want, sw, bias)
    assert max_abs(host(out), want) <= 1e-5
    assert max_abs(want, x @ w.T + bias) < 0.05  # and the scheme itself approximates the fp32 Linear


def _v_operand(V, dt, v_transposed, poison=True):
    """-> (device tensor, v_seq_pitch).  The transposed form is [B,h,d,pitch]; its pad columns hold
    NaN so that a kernel that lets them reach the output fails the comparison."""
    if not v_transposed:
        return dev(V, dt), 0
    B, h, S, d = V.shape
    pitch = (S + 7) // 8 * 8
    vt = np.full((B, h, d, pitch), np.nan if poison else 0.0, np.float32)
    vt[..., :S] = V.transpose(0, 1, 3, 2)
    return dev(vt, dt), pitch


@pytest.fixture(params=["auto", "8"])
def attention_waves(request, ttmi):
    """Wavefronts per workgroup of the fused attention kernel: its own choice (eight only for long sequences with a workgroup
    per compute unit, which none of these small shapes has), and eight forced through the switch TTMI_ATTENTION_WAVES."""
    if request.param != "auto":
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", int(request.param)))
    yield request.param
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("B,h,S,masked", [(2, 3, 128, True), (1, 2, 512, False), (3, 2, 100, True), (2, 1, 37, True),
                                         (1, 1, 500, True), (2, 12, 64, False), (1, 2, 1, False), (1, 1, 700, True)])
def test_fused_attention_vs_unfused_oracle(ttmi, oracle, attention_waves, dt, B, h, S, masked, v_transposed):
    """One-kernel softmax(scale QK^T + mask) V against the oracle's four-step chain
    (BatchMatMul, ApplyMaskAndSoftmax, BatchMatMul, TransposeForScore)."""
    rng = np.random.default_rng(S + B)
    d = 64
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    mask = None
    if masked:
        mask = np.zeros((B, 1, 1, S), np.float32)
        mask[0, ..., S // 2 + 1:] = -10000.0
        mask[-1, ..., :S // 3] = -10000.0
    dQ, dK = dev(Q, dt), dev(K, dt)
    dV, pitch = _v_operand(V, dt, v_transposed)
    out = torch.full((B, S, h * d), 9.0, dtype=dQ.dtype, device="cuda")
    ok(ttmi.ttmi_fused_attention(ptr(dQ), ptr(dK), ptr(dV), ptr(dev(mask)) if masked else None, ptr(out), None, B, h, S, d,
                                 pitch, 0.125, TTMI_DTYPES[dt], stream()))
    score = oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask, 1.0, True)
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, rounded(V, dt), False)).reshape(B, S, h * d)
    # P is rounded to 16 bits before the second MFMA, as the unfused path stores it
    assert max_abs(host(out), want) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("B,h,S,masked", [(2, 3, 128, True), (1, 2, 512, False), (3, 2, 100, True), (2, 1, 37, True),
                                         (1, 1, 500, True), (2, 12, 64, False), (1, 2, 1, False), (1, 1, 700, True),
                                         (3, 2, 260, True), (2, 2, 63, False)])
@pytest.mark.parametrize("v_transposed", [False, True])
def test_fused_attention_fp32_vs_unfused_oracle(ttmi, oracle, attention_waves, B, h, S, masked, v_transposed):
    """The fp32 form of the one-kernel attention (32x32x2 fp32 matrix instructions; V row-major, or transposed with NaN
    in its pad columns) against the oracle's four-step chain, to fp32 accuracy: nothing is rounded to 16 bits on the way."""
    rng = np.random.default_rng(S + 3 * B)
    d = 64
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    mask = None
    if masked:
        mask = np.zeros((B, 1, 1, S), np.float32)
        mask[0, ..., S // 2 + 1:] = -10000.0
        mask[-1, ..., :S // 3] = -10000.0
    dQ, dK = dev(Q, "f32"), dev(K, "f32")
    dV, pitch = _v_operand(V, "f32", v_transposed)
    out = torch.full((B, S, h * d), 9.0, dtype=torch.float32, device="cuda")
    ok(ttmi.ttmi_fused_attention(ptr(dQ), ptr(dK), ptr(dV), ptr(dev(mask)) if masked else None, ptr(out), None, B, h, S, d,
                                 pitch, 0.125, TTMI_DTYPES["f32"], stream()))
    score = oracle.batch_matmul(Q, K, True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask, 1.0, True)
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, V, False)).reshape(B, S, h * d)
    assert max_abs(host(out), want) <= 5e-5
    # the form that also leaves the per-workgroup maxima of its output (for the int8 Linear that quantises it next):
    # the same bits, every slot written, their maximum is max|out|
    import ctypes
    out2 = torch.full((B, S, h * d), 9.0, dtype=torch.float32, device="cuda")
    slots = torch.full((capi.ABSMAX_SLOTS, ), float("nan"), device="cuda")
    written = ctypes.c_int(-1)
    ok(ttmi.ttmi_fused_attention_absmax(ptr(dQ), ptr(dK), ptr(dV), ptr(dev(mask)) if masked else None, ptr(out2), None, B, h, S,
                                        d, pitch, 0.125, TTMI_DTYPES["f32"], ptr(slots), ctypes.byref(written), stream()))
    assert torch.equal(out, out2)
    assert written.value == capi.ABSMAX_SLOTS and not torch.isnan(slots).any()
    assert float(slots.max()) == float(out.abs().max())


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("S", [1, 31, 33, 129, 256, 257, 545])
def test_attention_with_split_keys(ttmi, oracle, dt, S):
    """The form whose wavefronts share the keys of a head (forced): fewer blocks of keys than wavefronts, the change from four
    to eight of them past 256 keys, ragged last blocks with NaN in the pad columns of V^T."""
    rng = np.random.default_rng(S)
    B, h, d = 2, 2, 64
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    mask = np.zeros((B, 1, 1, S), np.float32)
    mask[0, ..., S // 2 + 1:] = -10000.0
    dV, pitch = _v_operand(V, dt, True)
    out = torch.full((B, S, h * d), 9.0, dtype=dV.dtype, device="cuda")
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", 1))
    try:
        ok(ttmi.ttmi_fused_attention(ptr(dev(Q, dt)), ptr(dev(K, dt)), ptr(dV), ptr(dev(mask)), ptr(out), None, B, h, S, d, pitch,
                                     0.125, TTMI_DTYPES[dt], stream()))
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
    prob = oracle.apply_mask_and_softmax(oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125), mask, 1.0, True)
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, rounded(V, dt), False)).reshape(B, S, h * d)
    assert max_abs(host(out), want) <= (5e-5 if dt == "f32" else GEMM_TOL[dt] * 2)


LOWEST = float(np.finfo(np.float32).min)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("form,v_transposed", [(-1, False), (-1, True), (8, False), (8, True), (1, True)])
@pytest.mark.parametrize("S", [1, 33, 70, 200, 300])
def test_attention_masks_far_from_zero(ttmi, oracle, dt, form, v_transposed, S):
    """Additive masks of the lowest float, of -inf and of ordinary large sizes: a wholly masked sequence is the mean of V
    (its scores vanish against the mask), a partly masked one is not changed by its masked keys, wherever the first
    unmasked key lies.  Every form of the one-kernel attention."""
    rng = np.random.default_rng(S)
    h, d = 2, 64
    rows = [np.full(S, x) for x in (LOWEST, -1e9, -1e11, -1e20, -1e37)]   # wholly masked
    rows += [np.where(np.arange(S) < S - 1, x, 0.0) for x in (LOWEST, -np.inf, -1e11)]      # only the last key is seen
    rows += [np.where(np.arange(S) >= (S + 1) // 2, x, 0.0) for x in (LOWEST, -np.inf)]
    rows += [np.where(np.arange(S) % 2 == 1, -np.inf, LOWEST), np.where(np.arange(S) == S // 2, 1e12, 0.0)]
    mask = np.stack(rows).astype(np.float32)
    B = len(rows)
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    dV, pitch = _v_operand(V, dt, v_transposed)
    out = torch.full((B, S, h * d), 9.0, dtype=dV.dtype, device="cuda")
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", form))
    try:
        ok(ttmi.ttmi_fused_attention(ptr(dev(Q, dt)), ptr(dev(K, dt)), ptr(dV), ptr(dev(mask)), ptr(out), None, B, h, S, d, pitch,
                                     0.125, TTMI_DTYPES[dt], stream()))
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
    score = oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask.reshape(B, 1, 1, S), 1.0, True)
    assert max_abs(prob[0], np.full_like(prob[0], 1.0 / S)) < 1e-6
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, rounded(V, dt), False)).reshape(B, S, h * d)
    assert max_abs(host(out), want) <= (5e-5 if dt == "f32" else GEMM_TOL[dt] * 2)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("form,v_transposed", [(-1, False), (-1, True), (8, True), (1, True)])
@pytest.mark.parametrize("S", [33, 200])
def test_attention_keeps_nans_where_they_belong(ttmi, dt, form, v_transposed, S):
    """A NaN in a query makes the row of that query and head NaN, one in a key or in the mask of a key the head or the sequence,
    and nothing else, on every form of the one-kernel attention."""
    rng = np.random.default_rng(S)
    B, h, d = 3, 2, 64
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    mask = np.zeros((B, S), np.float32)
    Q[0, 0, S // 2, 7] = np.nan
    K[1, 1, S - 1, 50] = np.nan
    mask[2, 3] = np.nan
    dV, pitch = _v_operand(V, dt, v_transposed)
    out = torch.full((B, S, h * d), 9.0, dtype=dV.dtype, device="cuda")
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", form))
    try:
        ok(ttmi.ttmi_fused_attention(ptr(dev(Q, dt)), ptr(dev(K, dt)), ptr(dV), ptr(dev(mask)), ptr(out), None, B, h, S, d, pitch,
                                     0.125, TTMI_DTYPES[dt], stream()))
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
    q, k, v = (rounded(x, dt).astype(np.float64) for x in (Q, K, V))
    p = np.exp(q @ k.transpose(0, 1, 3, 2) * 0.125 + mask[:, None, None, :])
    want = ((p / p.sum(-1, keepdims=True)) @ v).transpose(0, 2, 1, 3).reshape(B, S, h * d)
    got = host(out)
    assert np.isnan(want).sum() == d + S * d + S * h * d
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert max_abs(got[~np.isnan(want)], want[~np.isnan(want)]) <= (5e-5 if dt == "f32" else GEMM_TOL[dt] * 2)


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("F,past,fresh,per_query", [(1, 0, 1, False), (33, 0, 33, True), (1, 40, 1, False), (1, 127, 1, True),
                                                    (5, 124, 5, True), (64, 0, 256, False), (2, 255, 2, True), (31, 300, 212, False)])
def test_attention_with_probs(ttmi, oracle, dt, F, past, fresh, per_query):
    """Attention that returns its probabilities and grows the cache: [past | new] keys around the block of 32 and the limits
    of its three forms (128, 256, 512 keys), masks per key and per query, against the oracle's chain."""
    rng = np.random.default_rng(F + past + fresh)
    B, h, d, T = 2, 3, 64, past + fresh
    Q = rng.standard_normal((B, h, F, d), np.float32)
    K, V = (rng.standard_normal((B, h, T, d), np.float32) for _ in range(2))
    mask = np.where(rng.random((B, F if per_query else 1, T)) < 0.3, -1e18, 0.0).astype(np.float32)
    mask[..., 0] = 0.0
    dQ, dK, dV = dev(Q, dt), dev(K, dt), dev(V, dt)
    split = lambda x: (x[:, :, :past].contiguous(), x[:, :, past:].contiguous())
    (kp, kn), (vp, vn) = split(dK), split(dV)
    probs = torch.full((B, h, F, T), 9.0, dtype=dQ.dtype, device="cuda")
    out = torch.full((B, F, h * d), 9.0, dtype=dQ.dtype, device="cuda")
    kg, vg = torch.zeros_like(dK), torch.zeros_like(dV)
    ok(ttmi.ttmi_attention_with_probs(ptr(dQ), ptr(kp) if past else None, ptr(vp) if past else None, past, ptr(kn), ptr(vn), ptr(kg),
                                      ptr(vg), ptr(dev(mask)), int(per_query), ptr(probs), ptr(out), B, h, F, T, d, 0.125,
                                      TTMI_DTYPES[dt], stream()))
    assert torch.equal(kg, dK) and torch.equal(vg, dV)
    score = oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask.reshape(B, 1, -1, T), 1.0, not per_query)
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, rounded(V, dt), False)).reshape(B, F, h * d)
    assert max_abs(host(probs), prob) <= (2e-6 if dt == "f32" else GEMM_TOL[dt])
    assert max_abs(host(out), want) <= (5e-5 if dt == "f32" else GEMM_TOL[dt] * 2)


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("F,past,fresh,per_query", [(1, 40, 1, False), (33, 0, 70, True), (5, 195, 5, True), (2, 298, 2, False)])
def test_attention_with_probs_masks_far_from_zero(ttmi, oracle, dt, F, past, fresh, per_query):
    """The lowest float over a whole row (uniform probabilities), over all keys but one, and -inf: the three forms of the kernel."""
    rng = np.random.default_rng(F + past + fresh)
    h, d, T = 2, 64, past + fresh
    rows = [np.full(T, LOWEST), np.full(T, -1e11), np.where(np.arange(T) == T - 1, 0.0, LOWEST), np.where(np.arange(T) < T // 2, -np.inf, 0.0)]
    B = len(rows)
    mask = np.repeat(np.stack(rows).astype(np.float32)[:, None], F if per_query else 1, axis=1)
    Q = rng.standard_normal((B, h, F, d), np.float32)
    K, V = (rng.standard_normal((B, h, T, d), np.float32) for _ in range(2))
    dQ, dK, dV = dev(Q, dt), dev(K, dt), dev(V, dt)
    (kp, kn), (vp, vn) = ((x[:, :, :past].contiguous(), x[:, :, past:].contiguous()) for x in (dK, dV))
    probs = torch.full((B, h, F, T), 9.0, dtype=dQ.dtype, device="cuda")
    out = torch.full((B, F, h * d), 9.0, dtype=dQ.dtype, device="cuda")
    ok(ttmi.ttmi_attention_with_probs(ptr(dQ), ptr(kp) if past else None, ptr(vp) if past else None, past, ptr(kn), ptr(vn), None, None,
                                      ptr(dev(mask)), int(per_query), ptr(probs), ptr(out), B, h, F, T, d, 0.125, TTMI_DTYPES[dt], stream()))
    score = oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask.reshape(B, 1, -1, T), 1.0, not per_query)
    want = oracle.transpose_for_score(oracle.batch_matmul(prob, rounded(V, dt), False)).reshape(B, F, h * d)
    assert max_abs(host(probs), prob) <= (2e-6 if dt == "f32" else GEMM_TOL[dt])
    assert max_abs(host(out), want) <= (5e-5 if dt == "f32" else GEMM_TOL[dt] * 2)


def test_fused_attention_absmax_reports_no_slots_where_it_leaves_none(ttmi):
    """16-bit types, packed batches and launches with more workgroups than slots: the output as always, 0 slots
    reported, the slots untouched."""
    import ctypes
    d = 64
    for dt, B, h, S, packed in (("f16", 2, 2, 64, False), ("f32", 2, 2, 64, True), ("f32", 90, 12, 32, False)):
        g = torch.Generator(device="cuda").manual_seed(S + B)
        q, k, v = (torch.randn((B, h, S, d), device="cuda", generator=g).to(TORCH_DTYPES[dt]) for _ in range(3))
        cu = torch.arange(0, (B + 1) * S, S, dtype=torch.int32, device="cuda") if packed else None
        outs = []
        for with_slots in (False, True):
            out = torch.zeros((B, S, h * d), dtype=q.dtype, device="cuda")
            slots = torch.full((capi.ABSMAX_SLOTS, ), float("nan"), device="cuda")
            written = ctypes.c_int(-1)
            args = (ptr(q), ptr(k), ptr(v), None, ptr(out), ptr(cu) if packed else None, B, h, S, d, 0, 0.125, TTMI_DTYPES[dt])
            if with_slots:
                ok(ttmi.ttmi_fused_attention_absmax(*args, ptr(slots), ctypes.byref(written), stream()))
                assert written.value == 0 and torch.isnan(slots).all()
            else:
                ok(ttmi.ttmi_fused_attention(*args, stream()))
            outs.append(out)
        assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("lens", [[70, 5, 129, 33], [300, 5, 257, 256]])
def test_fused_attention_packed_batch(ttmi, oracle, attention_waves, dt, v_transposed, lens):
    """Packed batch: pad rows of q,k,v hold NaN on the device -- the kernel must never let a row
    past a sequence's length reach the output -- and zeros in the oracle's padded chain."""
    rng = np.random.default_rng(17)
    h, d = 2, 64
    B, maxS, total = len(lens), max(lens), sum(lens)
    Q, K, V = (rng.standard_normal((B, h, maxS, d), np.float32) for _ in range(3))
    Qp, Kp, Vp = Q.copy(), K.copy(), V.copy()
    for b, L in enumerate(lens):
        Q[b, :, L:], K[b, :, L:], V[b, :, L:] = 0, 0, 0
        Qp[b, :, L:], Kp[b, :, L:], Vp[b, :, L:] = np.nan, np.nan, np.nan
    cu = np.zeros(B + 1, np.int32)
    cu[1:] = np.cumsum(lens)
    mask = np.where(np.arange(maxS)[None, :] < np.array(lens)[:, None], 0.0, -1e9).astype(np.float32)
    out = torch.full((total, h * d), 9.0, dtype=dev(Q, dt).dtype, device="cuda")
    dV, pitch = _v_operand(Vp, dt, v_transposed)
    ok(ttmi.ttmi_fused_attention(ptr(dev(Qp, dt)), ptr(dev(Kp, dt)), ptr(dV), ptr(dev(mask)), ptr(out), ptr(dev(cu)), B, h,
                                 maxS, d, pitch, 0.125, TTMI_DTYPES[dt], stream()))
    score = oracle.batch_matmul(rounded(Q, dt), rounded(K, dt), True, 0.125)
    prob = oracle.apply_mask_and_softmax(score, mask.reshape(B, 1, 1, maxS), 1.0, True)
    ctx = oracle.batch_matmul(prob, rounded(V, dt), False)
    want = oracle.transpose_for_score_pad(ctx, lens).reshape(total, h * d)
    assert max_abs(host(out), want) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("lens", [[70, 5, 129, 33], [300, 5, 257, 256], [512] + [40, 100, 270] * 7])
def test_fused_attention_packed_batch_has_the_same_bits_whatever_the_pad_rows_hold(ttmi, attention_waves, dt, v_transposed, lens):
    rng = np.random.default_rng(18)
    h, d = 3, 64
    B, longest = len(lens), max(lens)
    tensors = [rng.standard_normal((B, h, longest, d), np.float32) for _ in range(3)]
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    results = []
    for pad in (0.0, 1.0, 30.0, np.inf, np.nan):
        Q, K, V = (t.copy() for t in tensors)
        for b, n in enumerate(lens):
            for t in (Q, K, V):
                t[b, :, n:] = t[b, :, n:] * pad if np.isfinite(pad) else pad
        dV, pitch = _v_operand(V, dt, v_transposed)
        out = torch.full((sum(lens), h * d), 9.0, dtype=dev(Q, dt).dtype, device="cuda")
        dQ, dK = dev(Q, dt), dev(K, dt)
        ok(ttmi.ttmi_fused_attention(ptr(dQ), ptr(dK), ptr(dV), None, ptr(out), ptr(cu), B, h, longest, d, pitch, 0.125, TTMI_DTYPES[dt], stream()))
        torch.cuda.synchronize()
        results.append(out)
    assert bool(torch.isfinite(results[0].float()).all()) and all(torch.equal(r, results[0]) for r in results)


@pytest.mark.parametrize("dt", ["f16", "f32"])
@pytest.mark.parametrize("B,h,longest", [(64, 5, 140), (65, 4, 300), (130, 3, 129), (22, 12, 260), (90, 4, 128)])
def test_packed_attention_of_many_sequences(ttmi, dt, B, h, longest):
    """More workgroups than CUs start in the order of the lengths: equal lengths, empty sequences, one more than the 64 that are
    ordered together, one and several blocks of queries.  Every sequence against fp64."""
    rng = np.random.default_rng(B)
    d, lens = 64, rng.integers(0, longest + 1, B)
    lens[rng.integers(B)] = longest
    lens[:5] = lens[5]
    Q, K, V = (rng.standard_normal((B, h, longest, d), np.float32) for _ in range(3))
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    out = torch.full((int(cu[-1]), h * d), 9.0, dtype=dev(Q[:1], dt).dtype, device="cuda")
    dQ, dK, dV, dcu = dev(Q, dt), dev(K, dt), dev(V, dt), dev(cu)
    ok(ttmi.ttmi_fused_attention(ptr(dQ), ptr(dK), ptr(dV), None, ptr(out), ptr(dcu), B, h, longest, d, 0, 0.125, TTMI_DTYPES[dt],
                                 stream()))
    got = host(out)
    Q, K, V = (rounded(x, dt).astype(np.float64) for x in (Q, K, V))
    for b, n in enumerate(lens):
        if n == 0:
            continue
        score = Q[b, :, :n] @ K[b, :, :n].transpose(0, 2, 1) * 0.125
        prob = np.exp(score - score.max(-1, keepdims=True))
        want = (prob / prob.sum(-1, keepdims=True)) @ V[b, :, :n]
        assert max_abs(got[cu[b]:cu[b + 1]], want.transpose(1, 0, 2).reshape(n, h * d)) <= GEMM_TOL[dt] * 2


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("B,S,v_transposed,packed", [(1, 100, True, False), (1, 20, True, False), (2, 200, False, False), (22, 130, True, False),
                                                     (2, 60, True, True)])
def test_attention_that_reads_ahead(ttmi, dt, B, S, v_transposed, packed):
    """The same bits with ranges to read ahead, on forms that read them and forms that do not (fp32 with V row-major, fp32 packed); ranges of nothing, of one word, ragged, and larger than a round of the reading workgroups.  What is no whole word is refused."""
    import ctypes
    rng = np.random.default_rng(S)
    h, d = 12, 64
    Q, K, V = (dev(rng.standard_normal((B, h, S, d), np.float32), dt) for _ in range(3))
    V, pitch = _v_operand(host(V), dt, v_transposed)
    cu = torch.arange(B + 1, dtype=torch.int32, device="cuda") * S
    ranges = [torch.ones(n, dtype=torch.int32, device="cuda") for n in (1, 1, 300001, 8 << 20)]
    data = (ctypes.c_void_p * 4)(*[r.data_ptr() for r in ranges])

    def run(sizes):
        out = torch.full((B * S, h * d), 9.0, dtype=Q.dtype, device="cuda")
        rc = ttmi.ttmi_fused_attention_ahead(ptr(Q), ptr(K), ptr(V), None, ptr(out), ptr(cu) if packed else None, B, h, S, d, pitch,
                                             0.125, TTMI_DTYPES[dt], data, (ctypes.c_int64 * 4)(*sizes), len(sizes), stream())
        return rc, out

    (rc, want), (rc2, got) = run([]), run([0, 4, 4 * 300001, 32 << 20])
    ok(rc)
    ok(rc2)
    assert torch.equal(got, want) and bool(torch.isfinite(want.float()).all())
    assert run([4, 2])[0] != 0 and run([-4])[0] != 0


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("B,longest,packed,v_transposed", [(20, 500, True, False), (20, 500, True, True), (3, 300, True, False), (64, 500, True, False),
                                                           (64, 130, False, True), (64, 130, False, False)])
def test_attention_that_reads_ahead_beside_many_workgroups(ttmi, dt, B, longest, packed, v_transposed):
    """The same where the workgroups nearly fill the chip: ragged packed batches of more than 256 (whose sequences the kernel orders by
    their lengths, for which it has to know the rows that only read), and, of 64 sequences, more than the chip holds at a time, which
    read nothing.  NaN in the ranges and behind the sequences reaches no result."""
    import ctypes
    rng = np.random.default_rng(B + longest)
    h, d = 12, 64
    lens = [longest] + rng.integers(5, longest, B - 1).tolist() if packed else [longest] * B
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    Q, K, V = (rng.standard_normal((B, h, longest, d), np.float32) for _ in range(3))
    for b, n in enumerate(lens):
        Q[b, :, n:], K[b, :, n:], V[b, :, n:] = np.nan, np.nan, np.nan
    Q, K, (V, pitch) = dev(Q, dt), dev(K, dt), _v_operand(V, dt, v_transposed)
    ranges = [torch.full((n, ), float("nan"), device="cuda") for n in (300001, 4 << 20)]
    data = (ctypes.c_void_p * 2)(*[r.data_ptr() for r in ranges])

    def run(sizes):
        out = torch.full((sum(lens) + 1, h * d), 9.0, dtype=Q.dtype, device="cuda")
        ok(ttmi.ttmi_fused_attention_ahead(ptr(Q), ptr(K), ptr(V), None, ptr(out), ptr(cu) if packed else None, B, h, longest, d, pitch,
                                           0.125, TTMI_DTYPES[dt], data, (ctypes.c_int64 * 2)(*sizes), len(sizes), stream()))
        return out

    want, got = run([]), run([4 * 300001, 16 << 20])
    assert torch.equal(got, want) and bool(torch.isfinite(want.float()).all()) and bool((want[-1] == 9.0).all())


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("B,h", [(3, 2), (45, 2), (60, 12)])
@pytest.mark.parametrize("S", [9, 34, 36, 37, 39])
def test_transposed_v_of_sequences_off_the_grid(ttmi, dt, B, h, S):
    """Groups of eight and of four rows of the QKV product that two sequences share, divided at every place: V^T holds what a row-major V
    does, and its pad columns nothing."""
    import ctypes
    rng = np.random.default_rng(S)
    H, pitch, M = 64 * h, (S + 7) // 8 * 8 + 8, B * S
    dA, dW = dev(rng.standard_normal((M, H), np.float32), dt), dev((rng.standard_normal((3 * H, H)) / np.sqrt(H)).astype(np.float32), dt)
    db = dev(rng.standard_normal(3 * H).astype(np.float32), dt)
    q, k, v = (torch.empty((B, h, S, 64), dtype=dA.dtype, device="cuda") for _ in range(3))
    vt = torch.full((B, h, 64, pitch), 7.0, dtype=dA.dtype, device="cuda")
    for out, v_pitch in ((v, 0), (vt, pitch)):
        args = _epi(bias=db, q=q, k=k, v=out, seq=S, heads=h, head_dim=64, v_seq_pitch=v_pitch)
        ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(dW), None, M, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    # (values of size 2, summed in the same or another order and rounded once)
    assert max_abs(host(vt[..., :S]), host(v.transpose(2, 3))) <= GEMM_TOL[dt]
    assert bool((vt[..., S:] == 7.0).all())


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("B,h,S", [(1, 1, 1), (1, 12, 10), (3, 3, 32), (1, 5, 33), (2, 12, 60), (1, 16, 300)])
def test_attention_with_its_projection(ttmi, dt, B, h, S):
    """Attention and the output projection in one launch, a slice per head, against fp64; one and several blocks of queries and keys, a
    last group of columns with idle wavefronts, four and eight wavefronts.  The slices' sum through the LayerNorm behind them, with
    either residual, against ttmi_gemm_bias_layer_norm; more slices than one round of loads.  Ranges read ahead change nothing."""
    import ctypes
    rng = np.random.default_rng(B * S + h)
    d, H, M = 64, 64 * h, B * S
    Q, K, V = (rng.standard_normal((B, h, S, d), np.float32) for _ in range(3))
    W = (rng.standard_normal((H, H)) / np.sqrt(H)).astype(np.float32)
    mask = np.where(rng.random((B, S)) < 0.3, -1e4, 0).astype(np.float32)
    mask[:, 0] = 0
    dV, pitch = _v_operand(V, dt, True)
    dQ, dK, dW, dmask = dev(Q, dt), dev(K, dt), dev(W, dt), dev(mask)
    buffer = torch.full((h * M + 8, H), 9.0, device="cuda")
    packed = buffer[:h * M].view(h, M, H)
    words = torch.ones(1000, dtype=torch.int32, device="cuda")
    for ranges in (0, 1):
        ok(ttmi.ttmi_attention_projection(ptr(dQ), ptr(dK), ptr(dV), ptr(dmask), ptr(dW), ptr(packed), B, h, S, d, pitch, 0.125, TTMI_DTYPES[dt],
                                          (ctypes.c_void_p * 1)(words.data_ptr()), (ctypes.c_int64 * 1)(4000), ranges, stream()))
        first = packed.clone() if ranges == 0 else first
        assert torch.equal(first, packed) and bool((buffer[h * M:] == 9.0).all())
    q, k, v, w = (rounded(x, dt).astype(np.float64) for x in (Q, K, V, W))
    p = np.exp(q @ k.transpose(0, 1, 3, 2) * 0.125 + mask[:, None, None, :])
    ctx = ((p / p.sum(-1, keepdims=True)) @ v).transpose(0, 2, 1, 3).reshape(M, h, d)
    want = np.stack([ctx[:, i] @ w[:, i * d:(i + 1) * d].T for i in range(h)])
    # (probabilities and context are rounded to the type, both sums of products of size 1 / sqrt(H))
    assert max_abs(host(packed), want) <= GEMM_TOL[dt] * 2
    # the LayerNorm over the slices' sum: the same as over the rounded context's product, but for the order of the sums
    R, bias, gamma, beta = (rng.standard_normal(n).astype(np.float32) for n in ((M, H), H, H, H))
    dR, db, dg, dbeta = dev(R, dt), dev(bias, dt), dev(gamma, dt), dev(beta, dt)
    r32 = dev(R)
    for residual, residual32 in ((dR, None), (None, r32)):
        out, out2 = torch.empty_like(dR), torch.empty_like(dR)
        o32, o322 = torch.empty_like(r32), torch.empty_like(r32)
        pp = lambda t: None if t is None else ptr(t)
        ok(ttmi.ttmi_add_slices_layer_norm(ptr(packed), h, ptr(out), pp(residual), pp(residual32), ptr(db), ptr(dg), ptr(dbeta),
                                           ptr(o32) if residual32 is not None else None, M, H, ctypes.c_float(1e-12), TTMI_DTYPES[dt], stream()))
        x = want.sum(0) + rounded(bias, dt) + (R if residual is None else rounded(R, dt))
        ref = (x - x.mean(1, keepdims=True)) / x.std(1, keepdims=True) * rounded(gamma, dt) + rounded(beta, dt)
        assert max_abs(host(out), ref) <= GEMM_TOL[dt] * 6
        if residual32 is not None:
            assert max_abs(host(o32), ref) <= GEMM_TOL[dt] * 6
    assert ttmi.ttmi_add_slices_layer_norm(ptr(packed), 0, ptr(out), None, ptr(r32), ptr(db), ptr(dg), ptr(dbeta), ptr(o32), M, H,
                                           ctypes.c_float(1e-12), TTMI_DTYPES[dt], stream()) != 0


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M,h,steps", [(1, 1, 1), (16, 1, 16), (17, 12, 12), (33, 3, 17), (8, 12, 24), (31, 4, 32), (40, 2, 33)])
def test_layer_norm_in_front_of_a_few_row_product(ttmi, oracle, dt, M, h, steps):
    """LayerNorm on the rows' way into the form for few rows (and, past its sizes, in a launch of its own): one and two steps of K
    per wavefront, one and two blocks of rows, ragged tiles; ReLU and head-split epilogues; a row of equal values."""
    import ctypes
    N, K = 64 * h, steps * (32 if dt == "f32" else 64)
    rng = np.random.default_rng(M + N + K)
    X, W = rng.standard_normal((M, K)).astype(np.float32), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    X[M // 2] = 3.0
    gamma, beta = 1 + 0.1 * rng.standard_normal(K).astype(np.float32), 0.1 * rng.standard_normal(K).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    dX, dW, dg, dbeta, db = dev(X, dt), dev(W, dt), dev(gamma, dt), dev(beta, dt), dev(bias, dt)
    x = rounded(X, dt).astype(np.float64)
    ln = (x - x.mean(1, keepdims=True)) / np.sqrt(x.var(1, keepdims=True) + 1e-6) * rounded(gamma, dt) + rounded(beta, dt)
    base = ln @ rounded(W, dt).astype(np.float64).T + rounded(bias, dt)
    normed = torch.empty_like(dX)
    C = torch.full((M + 40, N), -7.0, dtype=dX.dtype, device="cuda")
    args = _epi(bias=db, act=capi.ACT_RELU)
    ok(ttmi.ttmi_layer_norm_gemm_fused(ptr(dX), ptr(dg), ptr(dbeta), ctypes.c_float(1e-6), ptr(normed), ptr(dW), ptr(C), M, N, K, N, capi.EPI_BIAS_ACT,
                                       ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    # |LN| and the rows of W are of size 1, so the rounding of LN to the type is one more rounding of the kind GEMM_TOL holds
    assert max_abs(host(C[:M]), np.maximum(base, 0)) <= GEMM_TOL[dt] * 3
    assert torch.all(C[M:] == -7.0)
    q = torch.full((M + 1, h, 1, 64), -7.0, dtype=dX.dtype, device="cuda")
    args = _epi(bias=db, q=q, seq=1, heads=h, head_dim=64)
    ok(ttmi.ttmi_layer_norm_gemm_fused(ptr(dX), ptr(dg), ptr(dbeta), ctypes.c_float(1e-6), ptr(normed), ptr(dW), None, M, N, K, N, capi.EPI_QKV_SPLIT,
                                       ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    assert max_abs(host(q[:M]).reshape(M, N), base) <= GEMM_TOL[dt] * 3
    assert torch.all(q[M:] == -7.0)


def _attention64(Q, K, V, mask, scale=0.125):
    s = Q.double() @ K.double().transpose(2, 3) * scale
    return torch.softmax(s if mask is None else s + mask.double()[:, None, None, :], -1) @ V.double()


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("lens", [[1], [63, 64, 65, 3], [129, 100], [40, 300, 7], [545]])
@pytest.mark.parametrize("form", ["dense", "packed", "packed, V transposed"])
def test_fused_attention_fp32_in_halves(ttmi, waves, lens, form):
    """fp32 attention on the 16-bit matrix instructions, against 64 bits: lengths around the tiles of 64 keys, masks, both layouts of V
    (NaN behind the last key).  No further off than the fp32 instruction, which a dense batch with row-major V runs on."""
    B, h, S, d = len(lens), 2, max(lens), 64
    g = torch.Generator(device="cuda").manual_seed(S + waves)
    Q, K, V = (torch.randn(B, h, S, d, generator=g, device="cuda") for _ in range(3))
    pitch, packed = (S + 7) // 8 * 8, form != "dense"
    Vt = torch.full((B, h, d, pitch), float("nan"), device="cuda")
    Vt[..., :S] = V.transpose(2, 3)
    if packed:
        for b, n in enumerate(lens):
            K[b, :, n:], V[b, :, n:], Vt[b, :, :, n:] = float("nan"), float("nan"), float("nan")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    mask = torch.where(torch.rand(B, S, generator=g, device="cuda") < 0.2, -1e4, 0.0)

    def run(v, v_pitch, cu):
        out = torch.full((sum(lens) if cu is not None else B * S, h * d), 9.0, device="cuda")
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", waves))
        ok(ttmi.ttmi_fused_attention(ptr(Q), ptr(K), ptr(v), ptr(mask), ptr(out), ptr(cu), B, h, S, d, v_pitch, 0.125, capi.F32, stream()))
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
        if cu is None:
            return list(out.view(B, S, h, d).permute(0, 2, 1, 3).double())
        return [out[cu[b]:cu[b + 1]].view(-1, h, d).permute(1, 0, 2).double() for b in range(B)]

    lengths = lens if packed else [S] * B
    want = [_attention64(Q[b:b + 1, :, :n], K[b:b + 1, :, :n], V[b:b + 1, :, :n], mask[b:b + 1, :n])[0] for b, n in enumerate(lengths)]
    got = run(V if form == "packed" else Vt, 0 if form == "packed" else pitch, cu if packed else None)
    # scores up to 8 of 64 products each (3 * 2^-22 of sum |q k| / 8 <= 20), as a relative error of a probability, and as much again
    # for sums and exp2: 2^-16 of the largest value
    for a, w in zip(got, want):
        assert float((a - w).abs().max()) <= 2.0**-16 * float(w.abs().max())
    if not packed and S > 32:
        fp32 = run(V, 0, None)
        error = lambda x: sum(float(((a - w)**2).sum()) for a, w in zip(x, want))**0.5
        assert error(got) <= error(fp32), (error(got), error(fp32))


@pytest.mark.parametrize("what", ["large Q", "large K", "infinite K", "large V", "infinite V", "tiny column of V", "zero column of V", "NaN"])
@pytest.mark.parametrize("v_transposed,packed", [(True, False), (False, True), (True, True)])
def test_fused_attention_fp32_outside_the_window(ttmi, what, v_transposed, packed):
    """Values that fp16 halves do not hold: the workgroups that meet one compute on the fp32 instruction, the others as before."""
    B, h, S, d = 2, 2, 150, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    Q, K, V = (torch.randn(B, h, S, d, generator=g, device="cuda") for _ in range(3))
    if what == "large Q":
        Q[0, 0, 140] *= 1e5
    elif what == "large K":
        K[0, 1, 70] *= 3e3
    elif what == "infinite K":
        K[0, 1, 70, 5] = float("inf")
    elif what == "large V":
        V[1, 0] *= 1e6
    elif what == "infinite V":
        V[1, 0, 149, 7] = float("-inf")
    elif what == "tiny column of V":
        V[1, 1, :, 9] *= 1e-9
    elif what == "zero column of V":
        V[1, 1, :, 9] = 0
    else:
        V[0, 0, 3, 3] = float("nan")
    pitch = (S + 7) // 8 * 8
    v = V
    if v_transposed:
        v = torch.full((B, h, d, pitch), float("nan"), device="cuda")
        v[..., :S] = V.transpose(2, 3)
    cu = torch.tensor([0, S, 2 * S], dtype=torch.int32, device="cuda") if packed else None
    out = torch.full((B * S, h * d), 9.0, device="cuda")
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", 4))
    ok(ttmi.ttmi_fused_attention(ptr(Q), ptr(K), ptr(v), None, ptr(out), ptr(cu), B, h, S, d, pitch if v_transposed else 0, 0.125, capi.F32, stream()))
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
    got, want = out.view(B, S, h, d).permute(0, 2, 1, 3).double(), _attention64(Q, K, V, None)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), finite) and torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    # relative to the column that a value averages; scores of up to 1e5 are themselves rounded by 2^-8
    column = torch.where(torch.isfinite(V), V.abs(), 0).amax(2, keepdim=True).double()
    bound = 2.0**-6 if what in ("large Q", "large K") else 2.0**-15
    assert bool(((got - want).abs() <= bound * column + 1e-30)[finite].all())


@pytest.mark.parametrize("a,b", [(1e-8, 1e-8), (1e-6, 1e-6), (1e-8, 1.0), (1.0, 1e-7), (1e-15, 1e-15), (1e-3, 1e-3), (0.3, 0.3), (30.0, 30.0), (300.0, 1 / 300)])
@pytest.mark.parametrize("v_transposed,packed", [(True, False), (False, True), (True, True)])
def test_fused_attention_fp32_of_any_scale(ttmi, v_transposed, packed, a, b):
    """|q| of size a, |k| of size b and the scale that brings the scores to size 1: no further from 64 bits than the fp32 instruction,
    which a dense batch with row-major V runs on."""
    B, h, S, d = 2, 3, 150, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    Q, K, V = (torch.randn(B, h, S, d, generator=g, device="cuda") for _ in range(3))
    Q, K, scale, pitch = Q * a, K * b, 0.125 / (a * b), 152
    v = V
    if v_transposed:
        v = torch.full((B, h, d, pitch), float("nan"), device="cuda")
        v[..., :S] = V.transpose(2, 3)
    cu = torch.tensor([0, S, 2 * S], dtype=torch.int32, device="cuda") if packed else None

    def run(v, v_pitch, cu):
        out = torch.full((B * S, h * d), 9.0, device="cuda")
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", 4))
        ok(ttmi.ttmi_fused_attention(ptr(Q), ptr(K), ptr(v), None, ptr(out), ptr(cu), B, h, S, d, v_pitch, scale, capi.F32, stream()))
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
        return out.view(B, S, h, d).permute(0, 2, 1, 3).double()

    want = _attention64(Q, K, V, None, float(np.float32(scale)))
    got, fp32 = run(v, pitch if v_transposed else 0, cu), run(V, 0, None)
    # as in test_fused_attention_fp32_in_halves
    assert float((got - want).abs().max()) <= 2.0**-16 * float(want.abs().max())
    assert float((got - want).norm()) <= float((fp32 - want).norm())


@pytest.mark.parametrize("waves", [-1, 4, 8])
@pytest.mark.parametrize("form", ["V transposed", "packed", "packed, V transposed"])
@pytest.mark.parametrize("keys", [1, 2, 7, 16, 31, 32, 33])
def test_fused_attention_fp32_of_few_keys(ttmi, waves, form, keys):
    """Sums of a few products are hardly rounded: no further from 64 bits than the fp32 instruction, which a dense batch with row-major V
    runs on, whether the scores are small or not; beside a long sequence of a packed batch too."""
    B, h, d, packed = 40, 3, 64, "packed" in form
    lens = [keys] * B + ([150] if packed else [])
    S, pitch = max(lens), (max(lens) + 7) // 8 * 8
    g = torch.Generator(device="cuda").manual_seed(keys)
    for size in (0.3, 1.0):
        Q, K, V = (torch.randn(len(lens), h, S, d, generator=g, device="cuda") for _ in range(3))
        Q, K = Q * size, K * size
        Vt = torch.full((len(lens), h, d, pitch), float("nan"), device="cuda")
        Vt[..., :S] = V.transpose(2, 3)
        cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda") if packed else None

        def run(Q, K, v, B, S, v_pitch, cu, waves):
            out = torch.full((sum(lens) if cu is not None else B * S, h * d), 9.0, device="cuda")
            ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", waves))
            ok(ttmi.ttmi_fused_attention(ptr(Q), ptr(K), ptr(v), None, ptr(out), ptr(cu), B, h, S, d, v_pitch, 0.125, capi.F32, stream()))
            ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
            return out[:40 * keys].view(40, keys, h, d).permute(0, 2, 1, 3).double()

        few = [x[:40, :, :keys].contiguous() for x in (Q, K, V)]
        want = _attention64(*few, None)
        got = run(Q, K, V if form == "packed" else Vt, len(lens), S, 0 if form == "packed" else pitch, cu, waves)
        fp32 = run(*few, 40, keys, 0, None, 4)
        error, before = float((got - want).norm()), float((fp32 - want).norm())
        # (the split over the wavefronts of a workgroup adds the shares in another order: as many roundings, not the same ones)
        assert error <= before * 1.02, (error, before)


def _packed(ttmi, W):
    """fp32 weights [N, K] as ttmi_split_weights lays them out."""
    N, K = W.shape
    p = torch.full((2 * N * K + N, ), float("nan"), device="cuda")
    p[:N * K] = W.flatten()
    ok(ttmi.ttmi_split_weights(ptr(p), N, K, stream()))
    return p


def _split_error_bound(A, W):
    """Per element.  Halves of 11 bits leave 2^-22 of a value and drop the product of the low ones (2^-22): 3 * 2^-22 of sum |a b|.
    The sums: one rounding (2^-24) per 32 products of each kind, of partial sums no larger than sum |a b|."""
    absolute = A.double().abs() @ W.double().abs().T
    return absolute * (3 * 2.0**-22 + (A.shape[1] / 32 + 8) * 2.0**-23)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 8, 32), (40, 72, 64), (100, 776, 96), (100, 776, 416), (129, 2304, 544), (300, 1024, 1056), (129, 2304, 768), (264, 768, 3072), (387, 3072, 768),
                                   (1000, 1536, 160), (1999, 768, 768), (2000, 3072, 128), (2500, 2304, 768), (8200, 520, 256)])
def test_packed_weights(ttmi, M, N, K):
    """fp32 products on the 16-bit matrix instructions: every tile, ragged rows and columns, one to many K steps, shares
    of them that differ by group of wavefronts, K slices, every epilogue; rows past M stay untouched.  No further from 64 bits than the fp32 instruction is."""
    import ctypes
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    A, W, bias, res = rand(M, K), rand(N, K) * 0.02, rand(N), rand(M, N)
    P, base = _packed(ttmi, W), A.double() @ W.double().T
    bound = _split_error_bound(A, W) + 2.0**-22 * (1 + bias.abs() + res.abs()).double()
    error = {}
    for name, epi, args, want in (("bias", capi.EPI_BIAS, _epi(bias=bias), base + bias.double()),
                                  ("relu", capi.EPI_BIAS_ACT, _epi(bias=bias, act=capi.ACT_RELU), (base + bias.double()).relu()),
                                  ("residual", capi.EPI_BIAS_RESIDUAL, _epi(bias=bias, residual=res), base + bias.double() + res.double()),
                                  ("f32", capi.EPI_F32_OUT, _epi(), base)):
        for weight, dt in ((P, capi.F32_PACKED), (W, capi.F32)):
            C = torch.full((M + 40, N), -7.0, device="cuda")
            ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(weight), ptr(C), M, N, K, K, K, N, epi, ctypes.byref(args), dt, stream()))
            assert torch.all(C[M:] == -7.0)
            error[name, dt] = (C[:M].double() - want).norm()
            if dt == capi.F32_PACKED:
                assert bool(((C[:M].double() - want).abs() <= bound).all()), name
    if K >= 96:
        assert float(error["f32", capi.F32_PACKED]) <= float(error["f32", capi.F32])
    if N <= 4096:
        one, zero, out, out2 = torch.ones(N, device="cuda"), torch.zeros(N, device="cuda"), torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
        x = base + res.double() + bias.double()
        want = torch.nn.functional.layer_norm(x, (N, ), eps=1e-5)
        for fn, dst in ((ttmi.ttmi_gemm_bias_layer_norm, out), (ttmi.ttmi_gemm_bias_layer_norm_static, out2)):
            ok(fn(ptr(A), ptr(P), ptr(dst), ptr(res), None, ptr(bias), ptr(one), ptr(zero), None, M, N, K, 1e-5, capi.F32_PACKED, stream()))
        assert torch.equal(out, out2)
        assert float((out.double() - want).abs().max()) <= LN_TOL["f32"]


@pytest.mark.gpu
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("B,S,h", [(7, 5, 12), (1, 37, 16), (9, 31, 12), (7, 130, 12), (2, 387, 16), (20, 100, 12)])
def test_packed_weights_head_split(ttmi, v_transposed, B, S, h):
    """The QKV projection: row by row and through the column pass of a transposed V (sequences off every grid)."""
    import ctypes
    d, H = 64, h * 64
    g = torch.Generator(device="cuda").manual_seed(S + h)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    A, W, bias = rand(B * S, H), rand(3 * H, H) * 0.02, rand(3 * H)
    pitch = (S + 7) // 8 * 8 if v_transposed else 0
    q, k = (torch.full((B, h, S, d), float("nan"), device="cuda") for _ in range(2))
    v = torch.full((B, h, d, pitch) if v_transposed else (B, h, S, d), 7.0, device="cuda")
    args = _epi(bias=bias, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
    ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, W)), None, B * S, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args),
                            capi.F32_PACKED, stream()))
    split = lambda x: x.view(B, S, 3, h, d).permute(2, 0, 3, 1, 4)
    want = split(A.double() @ W.double().T + bias.double())
    bound = split(_split_error_bound(A, W) + 2.0**-22 * (1 + bias.abs()).double())
    if v_transposed:
        assert torch.all(v[..., S:] == 7.0)
        v = v[..., :S].transpose(2, 3)
    for i, got in enumerate((q, k, v)):
        assert bool(((got.double() - want[i]).abs() <= bound[i]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(70, 136, 96), (300, 768, 768), (2000, 768, 768)])
def test_packed_weights_outside_the_window(ttmi, M, N, K):
    """Rows of either operand whose largest value the halves do not hold (tiny, huge, zero, infinite, NaN) come out as the fp32
    instruction gives them: to fp32 accuracy of the row, infinities and NaNs where they belong."""
    import ctypes
    g = torch.Generator(device="cuda").manual_seed(M)
    A, W = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * 0.02
    A[3] *= 1e-9
    A[17] *= 1e6
    A[18] = 0
    A[40] *= 2.0**-12
    A[33, :5] = torch.tensor([5e4, -3e5, 1.0, 1e-6, 0.0], device="cuda")
    W[7] *= 1e-12
    W[8] = 0
    W[50] *= 1e8
    want = A.double() @ W.double().T
    bound = (A.double().abs() @ W.double().abs().T) * (K + 8) * 2.0**-24 + 1e-37
    C = torch.empty(M, N, device="cuda")

    def run(A, W):
        C.fill_(7.0)
        ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, W)), ptr(C), M, N, K, K, K, N, capi.EPI_F32_OUT, ctypes.byref(_epi()), capi.F32_PACKED, stream()))
        return C.double()

    assert bool(((run(A, W) - want).abs() <= bound).all())
    A[20, 2], A[21, 3], A[60, 9], W[70, 4] = float("inf"), float("-inf"), float("nan"), float("inf")
    want = A.double() @ W.double().T
    got = run(A, W)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    assert bool(((got - want).abs() <= bound)[finite].all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 8, 32), (100, 776, 96), (129, 2304, 544), (129, 2304, 768), (264, 768, 3072), (387, 3072, 768), (1000, 1536, 160), (1999, 768, 768),
                                   (2000, 3072, 128), (2500, 2304, 768)])
def test_packed_weights_outside_the_window_beside_others(ttmi, M, N, K):
    """What a row of either operand holds changes no other row's results, whatever tile they share: rows and columns outside the window
    are right to fp32 accuracy, and all others keep their bits."""
    import ctypes
    g = torch.Generator(device="cuda").manual_seed(M + K)
    A, W = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * 0.02

    def run(A, W):
        C = torch.full((M, N), 7.0, device="cuda")
        ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, W)), ptr(C), M, N, K, K, K, N, capi.EPI_F32_OUT, ctypes.byref(_epi()), capi.F32_PACKED, stream()))
        return C

    alone = run(A, W)
    rows, cols = torch.zeros(M, dtype=torch.bool, device="cuda"), torch.zeros(N, dtype=torch.bool, device="cuda")
    rows[torch.tensor([0, 17, M // 2, M - 1])] = True
    cols[torch.tensor([1, 2, 5, N - 2])] = True
    A2, W2 = A.clone(), W.clone()
    A2[rows] *= torch.tensor([1e-9, 1e5, 1e-6, 1e4], device="cuda")[:, None]
    W2[cols] *= torch.tensor([1e-38, 1e30, 1e-7, 1e8], device="cuda")[:, None]  # (the first are subnormal)
    got = run(A2, W2)
    other = ~rows[:, None] & ~cols[None, :]
    assert torch.equal(got[other], alone[other])
    want = A2.double() @ W2.double().T
    bound = (A2.double().abs() @ W2.double().abs().T) * (K + 8) * 2.0**-24 + 1e-37
    assert bool(((got.double() - want).abs() <= bound)[~other].all())
    A2[17, 3], W2[5, 1] = float("inf"), float("nan")
    assert torch.equal(run(A2, W2)[other], alone[other])


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,h", [(1, 37, 16), (7, 130, 12), (2, 387, 16), (20, 100, 12)])
def test_packed_weights_head_split_outside_the_window(ttmi, B, S, h):
    """The same through the head split and the column pass of a transposed V."""
    import ctypes
    d, H = 64, h * 64
    g = torch.Generator(device="cuda").manual_seed(S + h)
    A, W, bias = torch.randn(B * S, H, generator=g, device="cuda"), torch.randn(3 * H, H, generator=g, device="cuda") * 0.02, torch.randn(3 * H, generator=g, device="cuda")
    pitch = (S + 7) // 8 * 8

    def run(A, W):
        q, k = (torch.empty(B, h, S, d, device="cuda") for _ in range(2))
        v = torch.zeros(B, h, d, pitch, device="cuda")
        args = _epi(bias=bias, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
        ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, W)), None, B * S, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args), capi.F32_PACKED, stream()))
        return torch.stack([q, k, v[..., :S].transpose(2, 3)]).permute(1, 3, 0, 2, 4).reshape(B * S, 3 * H)

    alone = run(A, W)
    A2, W2 = A.clone(), W.clone()
    A2[11] *= 1e-8
    A2[B * S - 1] *= 1e5
    W2[H + 7] *= 1e-6
    W2[3 * H - 3] *= 1e-6
    got, other = run(A2, W2), torch.ones(B * S, 3 * H, dtype=torch.bool, device="cuda")
    other[11] = other[B * S - 1] = other[:, H + 7] = other[:, 3 * H - 3] = False
    assert torch.equal(got[other], alone[other])
    want = A2.double() @ W2.double().T + bias.double()
    bound = (A2.double().abs() @ W2.double().abs().T + bias.double().abs()) * (H + 8) * 2.0**-24
    assert bool(((got.double() - want).abs() <= bound)[~other].all())


def _held(x):
    """The size at which the halves hold a value: as if none but zero were smaller than 2^-14."""
    return torch.where(x == 0, 0.0, x.double().abs().clamp(min=2.0**-14))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [100, 2000])
@pytest.mark.parametrize("rest", [1e-2, 1e-4, 1e-6, 1e-7, 1e-10, 1e-13])
@pytest.mark.parametrize("operand", ["A", "W"])
def test_packed_weights_small_values_beside_large(ttmi, M, rest, operand):
    """Rows whose largest value is in the window while the others are not, the large one beside a zero: 3 * 2^-22 max(|a|, 2^-14)
    max(|b|, 2^-14) of each product, and the rounding of the sums as in _split_error_bound."""
    import ctypes
    N, K = 776, 416
    g = torch.Generator(device="cuda").manual_seed(M)
    A, W = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda") * 0.02
    small, other = (A, W) if operand == "A" else (W, A)
    small *= rest / (1.0 if operand == "A" else 0.02)
    small[:, 7], other[:, 7] = 1000.0, 0.0
    C = torch.empty(M, N, device="cuda")
    ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, W)), ptr(C), M, N, K, K, K, N, capi.EPI_F32_OUT, ctypes.byref(_epi()), capi.F32_PACKED, stream()))
    want, absolute = A.double() @ W.double().T, A.double().abs() @ W.double().abs().T
    bound = 3 * 2.0**-22 * (_held(A) @ _held(W).T) + absolute * (K / 32 + 8) * 2.0**-23
    assert bool(((C.double() - want).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("K", [96, 768])
def test_packed_weights_hold_single_values(ttmi, K):
    """A unit matrix as the weight: values come out to within 2^-22 max(|x|, 2^-14), of any magnitude (rows outside the window as they are)."""
    import ctypes
    M = 500
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randn(M, K, generator=g, device="cuda") * 2.0**torch.randint(-40, 9, (M, K), generator=g, device="cuda")
    A[::50] *= 2.0**-30
    A[::70] *= 2.0**20
    C = torch.empty(M, K, device="cuda")
    ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(_packed(ttmi, torch.eye(K, device="cuda"))), ptr(C), M, K, K, K, K, K, capi.EPI_F32_OUT, ctypes.byref(_epi()),
                            capi.F32_PACKED, stream()))
    largest = A.abs().amax(1, keepdim=True)
    outside = (largest < 2.0**-13) | (largest >= 2.0**11)
    assert 5 < int(outside.sum()) < 50
    # (a row that is cut along K has parts that may be outside by themselves: then they are exact)
    assert bool(((C.double() - A.double()).abs() <= torch.where(outside, 0.0, 2.0**-22 * _held(A))).all())


@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 64])
@pytest.mark.parametrize("M", [40, 500, 2000])
def test_packed_weights_of_short_sums(ttmi, M, K):
    """Sums of a few products too are no further from 64 bits than the fp32 instruction leaves them."""
    import ctypes
    N = 768
    g = torch.Generator(device="cuda").manual_seed(M + K)
    for make in (lambda *s: torch.randn(s, generator=g, device="cuda"), lambda *s: torch.rand(s, generator=g, device="cuda"),
                 lambda *s: torch.nn.functional.gelu(torch.randn(s, generator=g, device="cuda"))):
        A, W = make(M, K), make(N, K) * 0.02
        want, error = A.double() @ W.double().T, []
        for weight, dt in ((_packed(ttmi, W), capi.F32_PACKED), (W, capi.F32)):
            C = torch.empty(M, N, device="cuda")
            ok(ttmi.ttmi_gemm_fused(ptr(A), ptr(weight), ptr(C), M, N, K, K, K, N, capi.EPI_F32_OUT, ctypes.byref(_epi()), dt, stream()))
            error.append(float((C.double() - want).norm()))
        assert error[0] <= error[1], (error, K)


@pytest.mark.parametrize("v_transposed,packed", [(True, False), (False, True)])
@pytest.mark.parametrize("rest", [1e-2, 1e-4, 1e-6, 1e-9])
def test_fused_attention_fp32_large_values_at_masked_keys(ttmi, v_transposed, packed, rest):
    """Columns of V whose largest value sits at a masked key, the others far below: 3 * 2^-22 of each probability times max(|v|, 2^-14), a
    probability counting 2^-14 of the row's largest at least (and not more than 1), beside what the scores leave."""
    B, h, S, d = 2, 3, 150, 64
    g = torch.Generator(device="cuda").manual_seed(7)
    Q, K, V = (torch.randn(B, h, S, d, generator=g, device="cuda") for _ in range(3))
    V *= rest
    V[:, :, 70:80] = 1000.0
    mask = torch.zeros(B, S, device="cuda")
    mask[:, 70:80] = -1e9
    pitch, v = 152, V
    if v_transposed:
        v = torch.full((B, h, d, pitch), float("nan"), device="cuda")
        v[..., :S] = V.transpose(2, 3)
    cu = torch.tensor([0, S, 2 * S], dtype=torch.int32, device="cuda") if packed else None
    out = torch.full((B * S, h * d), 9.0, device="cuda")
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", 4))
    ok(ttmi.ttmi_fused_attention(ptr(Q), ptr(K), ptr(v), ptr(mask), ptr(out), ptr(cu), B, h, S, d, pitch if v_transposed else 0, 0.125, capi.F32, stream()))
    ok(ttmi.ttmi_set_kernel_switch(b"TTMI_ATTENTION_WAVES", -1))
    got = out.view(B, S, h, d).permute(0, 2, 1, 3).double()
    P = torch.softmax(Q.double() @ K.double().transpose(2, 3) * 0.125 + mask.double()[:, None, None, :], -1)
    P2 = torch.where(P == 0, 0.0, P + 2.0**-14 * P.amax(-1, keepdim=True))
    bound = 2.0**-16 * (P @ V.double().abs()) + 3 * 2.0**-22 * (P2 @ _held(V))
    assert bool(((got - P @ V.double()).abs() <= bound).all())


def _guarded(rows, cols, dtype):
    """A matrix with eight rows behind it that nothing may write."""
    whole = torch.full((rows + 8, cols), 7.0, dtype=dtype, device="cuda")
    return whole, whole[:rows]


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("N,K", [(3072, 128), (776, 256)])
@pytest.mark.parametrize("beside", [-1, 0, 1])
def test_products_on_both_sides_of_the_write_through_line(ttmi, dt, N, K, beside):
    """From 2 MiB of output on a launch writes its stores through L2; the row counts around that line, the last ones of a ragged tile, into a
    matrix with guard rows."""
    import ctypes
    M = -(-(2 << 20) // (N * torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size())) + beside
    rng = np.random.default_rng(M)
    A, W, bias = rng.standard_normal((M, K), np.float32), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    want = np.maximum(rounded(A, dt).astype(np.float64) @ rounded(W, dt).T.astype(np.float64) + rounded(bias, dt), 0)
    weights = [(dW, TTMI_DTYPES[dt])] + ([(_packed(ttmi, dW), capi.F32_PACKED)] if dt == "f32" else [])
    for w, kind in weights:
        whole, C = _guarded(M, N, dA.dtype)
        ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(w), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_ACT, ctypes.byref(_epi(bias=db, act=capi.ACT_RELU)), kind, stream()))
        # values of size up to 8, rounded once; fp32: sums of 256 products
        assert max_abs(host(C), want) <= 2 * GEMM_TOL[dt]
        assert bool((whole[M:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("beside", [0, 1])
def test_products_on_both_sides_of_the_line_where_stores_stay_again(ttmi, dt, beside):
    """Outputs of 144 MiB (16-bit, the 256-row tiles) and 90 MiB (fp32, the split ring) are the largest that are written through."""
    import ctypes
    N, K = 3072, 128
    M = ((90 << 20) // (4 * N) if dt == "f32" else (144 << 20) // (2 * N)) + beside
    torch.manual_seed(M)
    A, W, bias = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda") / K**0.5, torch.randn(N, device="cuda")
    dA, dW, db = (x.to(TORCH_DTYPES[dt]) for x in (A, W, bias))
    want = (dA.double() @ dW.double().t() + db.double()).relu_()
    w, kind = (_packed(ttmi, dW), capi.F32_PACKED) if dt == "f32" else (dW, TTMI_DTYPES[dt])
    whole, C = _guarded(M, N, dA.dtype)
    ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(w), ptr(C), M, N, K, K, K, N, capi.EPI_BIAS_ACT, ctypes.byref(_epi(bias=db, act=capi.ACT_RELU)), kind, stream()))
    # values of size up to 8, rounded once; fp32: sums of 128 products
    assert float((C.double() - want).abs().max()) <= 2 * GEMM_TOL[dt]
    assert bool((whole[M:] == 7.0).all())


def _layer_norm_operands(dt, m, n, shadow):
    """-> residual (fp32 if `shadow`) and the three row vectors as the kernel sees them, want(base in 64 bits), the operands on the device."""
    rng = np.random.default_rng(m)
    res, bias, gamma, beta = (rng.standard_normal(s).astype(np.float32) for s in ((m, n), (n,), (n,), (n,)))
    residual = res if shadow else rounded(res, dt)

    def want(base):
        s = base + residual + rounded(bias, dt).astype(np.float64)
        return rounded(beta, dt) + rounded(gamma, dt) * (s - s.mean(1, keepdims=True)) / np.sqrt(s.var(1, keepdims=True) + 1e-12)

    return rng, want, dev(res, dt), dev(res), [dev(v, dt) for v in (bias, gamma, beta)]


LAYER_NORM_TOL = {"f32": 1e-4, "f16": 2e-2, "bf16": 1.2e-1}  # values of size up to 16, rounded once; in front of it the product may be


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("shadow", [False, True])
@pytest.mark.parametrize("beside", [-1, 0, 1])
@pytest.mark.parametrize("n", [776, 768, 1024])
def test_layer_norm_on_both_sides_of_the_write_through_line(ttmi, dt, shadow, beside, n):
    """AddBiasLayerNorm by itself, row counts around 2 MiB of output (fp32: 6 MB); of 16-bit rows of 768 and 776 values it also leaves the
    workgroups of one wavefront there."""
    m = -(-(6000000 if dt == "f32" else 2 << 20) // (n * torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size())) + beside
    rng, want, res, res32, row = _layer_norm_operands(dt, m, n, shadow)
    x = rng.standard_normal((m, n)).astype(np.float32)
    whole, out = _guarded(m, n, TORCH_DTYPES[dt])
    out.copy_(dev(x, dt))
    whole32, out32 = _guarded(m, n, torch.float32)
    if shadow:
        ok(ttmi.ttmi_add_bias_layer_norm_residual32(ptr(out), ptr(res32), *[ptr(v) for v in row], ptr(out32), m, n, 1e-12, TTMI_DTYPES[dt], stream()))
        assert torch.equal(out, out32.to(out.dtype))
    else:
        ok(ttmi.ttmi_add_bias_layer_norm(ptr(out), ptr(res), *[ptr(v) for v in row], m, n, 1e-12, TTMI_DTYPES[dt], stream()))
    assert max_abs(host(out), want(rounded(x, dt).astype(np.float64))) <= LAYER_NORM_TOL[dt]
    for w in (whole, whole32):
        assert bool((w[m:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("shadow", [False, True])
@pytest.mark.parametrize("beside", [-1, 0, 1])
@pytest.mark.parametrize("n", [776, 260])
def test_summing_layer_norm_on_both_sides_of_the_write_through_line(ttmi, dt, shadow, beside, n):
    """The LayerNorm that sums the slices of a product with K of twice its columns and more: row counts around 2 MiB of what it stores, the
    unrounded rows among it, of widths that leave its workgroups partly idle."""
    K = 1664
    stored = torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size() + (4 if shadow else 0)
    m = -(-(2 << 20) // (n * stored)) + beside
    rng, want, res, res32, row = _layer_norm_operands(dt, m, n, shadow)
    A, W = rng.standard_normal((m, K), np.float32), (rng.standard_normal((n, K)) / np.sqrt(K)).astype(np.float32)
    exact = want(rounded(A, dt).astype(np.float64) @ rounded(W, dt).T.astype(np.float64))
    for w, kind in [(dev(W, dt), TTMI_DTYPES[dt])] + ([(_packed(ttmi, dev(W)), capi.F32_PACKED)] if dt == "f32" else []):
        whole, out = _guarded(m, n, TORCH_DTYPES[dt])
        whole32, out32 = _guarded(m, n, torch.float32)
        ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(dev(A, dt)), ptr(w), ptr(out), None if shadow else ptr(res), ptr(res32) if shadow else None, *[ptr(v) for v in row],
                                          ptr(out32) if shadow else None, m, n, K, 1e-12, kind, stream()))
        assert max_abs(host(out), exact) <= LAYER_NORM_TOL[dt]
        if shadow:
            assert torch.equal(out, out32.to(out.dtype))
        for guarded in (whole, whole32):
            assert bool((guarded[m:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024])
def test_layer_norm_of_few_rows_takes_one_wavefront_a_workgroup(ttmi, dt, n):
    """Row counts on both sides of 255 workgroups of four wavefronts, of widths that do not write through there, and ones that leave a wavefront
    partly idle."""
    element = torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size()
    vectors = n * element // 16
    per = 16 if vectors <= 16 else 8 if vectors <= 32 else 4  # rows of four wavefronts
    assert 255 * per * n * element < (6000000 if dt == "f32" else 2 << 20)
    for m in (1, 3, 2 * per + 1, 255 * per - 1, 255 * per, 255 * per + 1):
        rng, want, res, _, row = _layer_norm_operands(dt, m, n, False)
        x = rng.standard_normal((m, n), np.float32)
        whole, out = _guarded(m, n, TORCH_DTYPES[dt])
        out.copy_(dev(x, dt))
        ok(ttmi.ttmi_add_bias_layer_norm(ptr(out), ptr(res), *[ptr(v) for v in row], m, n, 1e-12, TTMI_DTYPES[dt], stream()))
        assert max_abs(host(out), want(rounded(x, dt).astype(np.float64))) <= LAYER_NORM_TOL[dt]
        assert bool((whole[m:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("M", [1, 64, 65, 97, 128, 129])
@pytest.mark.parametrize("N,K", [(3072, 768), (776, 96), (130, 64)])
def test_gemm_bias_act_has_no_named_form(ttmi, dt, M, N, K):
    """The layers' product with bias and activation, around the rows for which ttmi_gemm_fused keeps the form that ttmi_gemm_describe names."""
    rng = np.random.default_rng(M + N)
    A, W, bias = rng.standard_normal((M, K), np.float32), (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    dA, dW, db = dev(A, dt), dev(W, dt), dev(bias, dt)
    x = torch.from_numpy(rounded(A, dt)).double() @ torch.from_numpy(rounded(W, dt)).double().T + torch.from_numpy(rounded(bias, dt)).double()
    want = torch.nn.functional.gelu(x, approximate="tanh").numpy()
    for w, kind in [(dW, TTMI_DTYPES[dt])] + ([(_packed(ttmi, dW), capi.F32_PACKED)] if dt == "f32" else []):
        whole, C = _guarded(M, N, dA.dtype)
        ok(ttmi.ttmi_gemm_bias_act(ptr(dA), ptr(w), ptr(db), ptr(C), M, N, K, capi.ACT_GELU, kind, stream()))
        assert max_abs(host(C), want) <= 2 * GEMM_TOL[dt]  # values of size up to 8, rounded once
        assert bool((whole[M:] == 7.0).all())


def _guarded_heads(B, h, S, d, dtype):
    """A head-split tensor with eight sequences' worth of one head behind it that nothing may write."""
    whole = torch.full((B * h * S * d + 8 * S * d, ), 7.0, dtype=dtype, device="cuda")
    return whole, whole[:B * h * S * d].view(B, h, S, d)


@pytest.mark.parametrize("dt,forced", [("f32", False), ("f16", False), ("f16", True), ("bf16", False), ("bf16", True)])
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("S", [100, 112, 75])
@pytest.mark.parametrize("mib", [2, 120])
def test_head_split_on_both_sides_of_the_write_through_lines(ttmi, dt, forced, v_transposed, S, mib):
    """From 2 MiB of output on the head split writes Q, K and a row-major V through L2, up to 120 MiB on the large tiles (90 MiB in fp32, which
    two sequence counts on each side of the other types' line are past): by direct stores where sequences are multiples of 16 and from
    the strips where not, on tiles of the launcher's choice and on the large ones."""
    import ctypes
    h, d = 2, 64
    H = h * d
    element = torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size()
    below = (mib << 20) // (3 * H * element * S)
    torch.manual_seed(S)
    if forced:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", 1))
    try:
        for B in (below, below + 1):
            M = B * S
            A, W, bias = torch.randn(M, H, device="cuda"), torch.randn(3 * H, H, device="cuda") / H**0.5, torch.randn(3 * H, device="cuda")
            dA, dW, db = (x.to(TORCH_DTYPES[dt]) for x in (A, W, bias))
            want = (dA.double() @ dW.double().t() + db.double()).view(B, S, 3, h, d).permute(2, 0, 3, 1, 4)
            pitch = (S + 7) // 8 * 8 + 8 if v_transposed else 0
            for w, kind in [(dW, TTMI_DTYPES[dt])] + ([(_packed(ttmi, dW), capi.F32_PACKED)] if dt == "f32" else []):
                held = [_guarded_heads(B, h, S, d, dA.dtype) for _ in range(3)]
                (_, q), (_, k), (_, v) = held
                if v_transposed:
                    whole_v = torch.full((B * h * d * pitch + 8 * pitch, ), 7.0, dtype=dA.dtype, device="cuda")
                    v = whole_v[:B * h * d * pitch].view(B, h, d, pitch)
                args = _epi(bias=db, q=q, k=k, v=v, seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
                ok(ttmi.ttmi_gemm_fused(ptr(dA), ptr(w), None, M, 3 * H, H, H, H, 3 * H, capi.EPI_QKV_SPLIT, ctypes.byref(args), kind, stream()))
                if v_transposed:
                    assert bool((v[..., S:] == 7.0).all()) and bool((whole_v[v.numel():] == 7.0).all())
                    v = v[..., :S].transpose(2, 3)
                for got, exact in zip((q, k, v), want):
                    # values of size up to 8, rounded once; fp32: sums of 128 products
                    assert float((got.double() - exact).abs().max()) <= 2 * GEMM_TOL[dt]
                for whole, part in held:
                    assert bool((whole[part.numel():] == 7.0).all())
    finally:
        ok(ttmi.ttmi_set_kernel_switch(b"TTMI_LARGE_TILE", -1))


@pytest.mark.parametrize("beside", [-1, 0, 1])
@pytest.mark.parametrize("N,K", [(768, 128), (520, 256), (64, 128)])
@pytest.mark.parametrize("absmax", [False, True])
def test_int8_products_on_both_sides_of_the_write_through_line(ttmi, N, K, beside, absmax):
    """From 2 MiB of fp32 output on the dequantising stores go through L2: row counts around that line, guard rows, the bits of the product
    and its dequantisation one after the other; with the maxima that the next quantisation takes."""
    import ctypes
    M = -(-(2 << 20) // (4 * N)) + beside
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = (torch.randint(-127, 128, s, generator=g, device="cuda", dtype=torch.int8) for s in ((M, K), (N, K)))
    sx, sw, bias = torch.tensor([0.0123, 0.0], device="cuda"), (torch.rand(N, generator=g, device="cuda") + 0.5) * 1e-3, torch.randn(N, generator=g, device="cuda")
    acc, two_step = torch.empty((M, N), dtype=torch.int32, device="cuda"), torch.empty((M, N), device="cuda")
    ok(ttmi.ttmi_gemm_i8(ptr(a), ptr(b), ptr(acc), M, N, K, K, K, N, stream()))
    ok(ttmi.ttmi_dequant_bias(ptr(acc), ptr(sx), ptr(sw), ptr(bias), ptr(two_step), M, N, stream()))
    whole, fused = _guarded(M, N, torch.float32)
    if absmax:
        slots, written = torch.full((capi.ABSMAX_SLOTS, ), float("nan"), device="cuda"), ctypes.c_int(-1)
        ok(ttmi.ttmi_gemm_i8_dequant_absmax(ptr(a), ptr(b), ptr(fused), ptr(sx), ptr(sw), ptr(bias), -1, M, N, K, K, K, N, ptr(slots), ctypes.byref(written), stream()))
        assert written.value == 0 or float(slots.max()) == float(two_step.abs().max())
    else:
        ok(ttmi.ttmi_gemm_i8_dequant(ptr(a), ptr(b), ptr(fused), ptr(sx), ptr(sw), ptr(bias), -1, M, N, K, K, K, N, stream()))
    assert torch.equal(fused, two_step) and bool((whole[M:] == 7.0).all())


@pytest.mark.parametrize("mib", [2, 12, 90])
@pytest.mark.parametrize("S", [64, 75])
def test_int8_head_split_on_both_sides_of_the_write_through_lines(ttmi, S, mib):
    """The int8 head split writes through from 12 to 90 MiB of output: sequence counts around those lines and around 2 MiB, where other products begin."""
    h, d = 2, 64
    H = h * d
    below = (mib << 20) // (3 * H * 4 * S)
    for B in (below, below + 1):
        M = B * S
        g = torch.Generator(device="cuda").manual_seed(M)
        a, b = (torch.randint(-127, 128, s, generator=g, device="cuda", dtype=torch.int8) for s in ((M, H), (3 * H, H)))
        sx, sw, bias = torch.tensor([0.0123, 0.0], device="cuda"), (torch.rand(3 * H, generator=g, device="cuda") + 0.5) * 1e-3, torch.randn(3 * H, generator=g, device="cuda")
        flat, two = torch.empty((M, 3 * H), device="cuda"), [torch.empty((B, h, S, d), device="cuda") for _ in range(3)]
        ok(ttmi.ttmi_gemm_i8_dequant(ptr(a), ptr(b), ptr(flat), ptr(sx), ptr(sw), None, -1, M, 3 * H, H, H, H, 3 * H, stream()))
        ok(ttmi.ttmi_split_add_bias_transpose_for_score(ptr(flat), ptr(bias), *[ptr(t) for t in two], B, S, h, d, TTMI_DTYPES["f32"], stream()))
        held = [_guarded_heads(B, h, S, d, torch.float32) for _ in range(3)]
        ok(ttmi.ttmi_gemm_i8_dequant_qkv_split(ptr(a), ptr(b), ptr(sx), ptr(sw), ptr(bias), *[ptr(t) for _, t in held], M, 3 * H, H, H, H, S, h, d, stream()))
        for (whole, one), want in zip(held, two):
            assert torch.equal(one, want) and bool((whole[one.numel():] == 7.0).all())


@pytest.mark.parametrize("rows", [12287, 12288, 12289])
@pytest.mark.parametrize("k", [171, 192])
def test_quantisation_on_both_sides_of_the_rows_that_write_through(ttmi, oracle, rows, k):
    """Passes of 2 MiB and more write through L2 up to 12288 rows; ragged and whole workgroups, guard bytes behind."""
    n = rows * k
    x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    whole_q = torch.full((n + 32, ), 99, dtype=torch.int8, device="cuda")
    scale = torch.full((capi.QUANT_SCALE_FLOATS, ), float("nan"), device="cuda")
    ok(ttmi.ttmi_quantize_rows_i8(ptr(x), ptr(whole_q), ptr(scale), rows, k, stream()))
    want, want_scale = oracle.quantize_tensor_i8(host(x).reshape(rows, k))
    assert np.array_equal(host(whole_q[:n]), want.reshape(-1)) and host(scale)[0] == np.float32(want_scale)
    assert bool((whole_q[n:] == 99).all())


@pytest.mark.parametrize("dt", ALL_DTYPES)
@pytest.mark.parametrize("v_transposed", [False, True])
@pytest.mark.parametrize("S", [128, 100, 300])
@pytest.mark.parametrize("packed", [False, True])
def test_fused_attention_on_both_sides_of_the_write_through_line(ttmi, dt, v_transposed, S, packed):
    """From 2 MiB of context on (of packed batches half of the padded size) it is written through L2: sequence counts on both sides, each
    sequence's own softmax in 64 bits, guard rows behind."""
    h, d = 2, 64
    element = torch.empty(0, dtype=TORCH_DTYPES[dt]).element_size()
    at_line = -(-(2 << 20) * (2 if packed else 1) // (h * S * d * element))
    rng = np.random.default_rng(S)
    for B in (at_line - 1, at_line):
        lens = [S] + [int(n) for n in rng.integers(1, S + 1, B - 1)] if packed else [S] * B
        g = torch.Generator(device="cuda").manual_seed(B)
        q, k, v = (torch.randn(B, h, S, d, generator=g, device="cuda").to(TORCH_DTYPES[dt]) for _ in range(3))
        pitch, given = (S + 7) // 8 * 8, v
        if v_transposed:
            given = torch.full((B, h, d, pitch), float("nan"), dtype=v.dtype, device="cuda")
            given[..., :S] = v.transpose(2, 3)
        cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda") if packed else None
        keys = (torch.arange(S, device="cuda")[None] < torch.tensor(lens, device="cuda")[:, None])
        whole, out = _guarded(sum(lens), h * d, q.dtype)
        ok(ttmi.ttmi_fused_attention(ptr(q), ptr(k), ptr(given), None, ptr(out), ptr(cu), B, h, S, d, pitch if v_transposed else 0, 0.125, TTMI_DTYPES[dt], stream()))
        scores = (q.double() @ k.double().transpose(2, 3).contiguous() * 0.125).masked_fill(~keys[:, None, None, :], float("-inf"))
        want = (torch.softmax(scores, -1) @ v.double()).transpose(1, 2).reshape(B * S, h * d)[keys.reshape(-1)]
        # P is rounded to 16 bits before the second product
        assert float((out.double() - want).abs().max()) <= (5e-5 if dt == "f32" else 2 * GEMM_TOL[dt])
        assert bool((whole[sum(lens):] == 7.0).all())


@pytest.mark.parametrize("B,S", [(20, 100), (17, 113)])
def test_fp32_head_split_just_short_of_a_round(ttmi, B, S):
    """96 x 192 tiles, rows that end inside one, V transposed.  An fp32 product to 3 * 2^-22 of its operands (at least 2^-14), 768 of them summed."""
    h, d, k, m = 12, 64, 768, B * S
    pitch = (S + 7) // 8 * 8
    gen = torch.Generator(device="cuda").manual_seed(S)
    a, w, b = (torch.randn(shape, generator=gen, device="cuda").mul_(scale) for shape, scale in [((m, k), 1.0), ((3 * h * d, k), k ** -0.5), ((3 * h * d,), 0.1)])
    q, kk = torch.empty(B, h, S, d, device="cuda"), torch.empty(B, h, S, d, device="cuda")
    v = torch.full((B, h, d, pitch), 7.0, device="cuda")
    args = capi.EpilogueArgs(bias=b.data_ptr(), q=q.data_ptr(), k=kk.data_ptr(), v=v.data_ptr(), seq=S, heads=h, head_dim=d, v_seq_pitch=pitch)
    name = ctypes.create_string_buffer(64)
    ok(ttmi.ttmi_gemm_describe(m, 3 * h * d, k, capi.EPI_QKV_SPLIT, ctypes.byref(args), capi.F32_PACKED, name, 64))
    assert "96x192" in name.value.decode(), name.value
    ok(ttmi.ttmi_gemm_fused(ptr(a), ptr(_packed(ttmi, w)), None, m, 3 * h * d, k, k, k, 3 * h * d, capi.EPI_QKV_SPLIT, ctypes.byref(args), capi.F32_PACKED, stream()))
    want = (a.double() @ w.double().T + b.double()).view(B, S, 3, h, d).permute(2, 0, 3, 1, 4)
    room = (a.abs().double() @ w.abs().double().T + b.abs().double()).view(B, S, 3, h, d).permute(2, 0, 3, 1, 4) * (3 * 2.0 ** -22 + 2.0 ** -20)
    for got, i in [(q, 0), (kk, 1), (v[..., :S].transpose(2, 3), 2)]:
        assert bool(((got.double() - want[i]).abs() <= room[i]).all()), i


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("tile,m,n,k", [("160x64", 800, 3072, 768), ("160x64", 797, 3080, 768), ("160x128", 1600, 3072, 768),
                                        ("160x128", 1589, 3064, 768), ("256x160", 6275, 3072, 768), ("256x160", 6145, 3048, 896)])
def test_tiles_between_powers_of_two(ttmi, dt, tile, m, n, k):
    """Whole tiles, and rows and columns that end inside one.  Against 64 bits: the result's own rounding (half of its last place), and 2^-12
    of an O(1) value for sums of k products in fp32 and the GELU of them."""
    name = ctypes.create_string_buffer(64)
    ok(ttmi.ttmi_gemm_bias_act_describe(m, n, k, capi.ACT_GELU, TTMI_DTYPES[dt], name, 64))
    assert tile in name.value.decode(), name.value
    gen = torch.Generator(device="cuda").manual_seed(m)
    a, w, b = (torch.randn(shape, generator=gen, device="cuda").mul_(scale).to(TORCH_DTYPES[dt])
               for shape, scale in [((m, k), 1.0), ((n, k), k ** -0.5), ((n,), 0.1)])
    c = torch.full((m + 1, n), 7.0, device="cuda", dtype=TORCH_DTYPES[dt])
    ok(ttmi.ttmi_gemm_bias_act(ptr(a), ptr(w), ptr(b), ptr(c), m, n, k, capi.ACT_GELU, TTMI_DTYPES[dt], stream()))
    want = torch.nn.functional.gelu(a.double() @ w.double().T + b.double(), approximate="tanh")
    half = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt]
    assert bool(((c[:m].double() - want).abs() <= half * want.abs() + 2.0 ** -12).all())
    assert bool((c[m] == 7.0).all())


def _tile_operands(m, n, k, dt):
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    return [torch.randn(shape, generator=gen, device="cuda").mul_(scale).to(TORCH_DTYPES[dt]) for shape, scale in [((m, k), 1.0), ((n, k), k ** -0.5), ((n,), 0.1)]]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("fp32_out", [False, True])
@pytest.mark.parametrize("tile,m,n,k", [("160x64", 2800, 768, 768), ("160x64", 2797, 776, 768), ("160x64", 2400, 1024, 4096), ("160x128", 6000, 768, 3072),
                                        ("160x128", 5989, 760, 768), ("256x160", 11500, 768, 768), ("256x160", 11490, 776, 832)])
def test_tiles_between_powers_of_two_store_products(ttmi, dt, fp32_out, tile, m, n, k):
    """With a bias alone, in the operands' type and in fp32.  Against 64 bits: k products by sixteen at a time are k / 16 roundings of at most 2^-24 of the
    sum of their magnitudes; then the result's own rounding, half of its last place."""
    epilogue = capi.EPI_F32_OUT if fp32_out else capi.EPI_BIAS
    a, w, b = _tile_operands(m, n, k, dt)
    args = _epi(bias=b)
    name = ctypes.create_string_buffer(64)
    ok(ttmi.ttmi_gemm_describe(m, n, k, epilogue, ctypes.byref(args), TTMI_DTYPES[dt], name, 64))
    assert tile in name.value.decode(), name.value
    c = torch.full((m + 1, n), 7.0, device="cuda", dtype=torch.float32 if fp32_out else TORCH_DTYPES[dt])
    ok(ttmi.ttmi_gemm_fused(ptr(a), ptr(w), ptr(c), m, n, k, k, k, n, epilogue, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    want = a.double() @ w.double().T + b.double()
    room = (a.abs().double() @ w.abs().double().T + b.abs().double()) * (k // 16 + 2) * 2.0 ** -24
    if not fp32_out:
        room += {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt] * want.abs()
    assert bool(((c[:m].double() - want).abs() <= room).all())
    assert bool((c[m] == 7.0).all())


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("tile,heads,lens", [("160x64", 12, [160] + [90] * 8 + [120]), ("160x64", 16, [200, 3, 97, 150, 50, 111, 89]),
                                             ("160x128", 12, [200, 1, 7] + [100] * 17 + [95]), ("160x128", 16, [113] * 13 + [31])])
def test_tiles_between_powers_of_two_split_the_heads_of_a_packed_batch(ttmi, dt, tile, heads, lens):
    """Rows that end inside a tile, requests that begin and end inside one; what lies past a request's rows stays as it was.  Tolerance as above."""
    d, B, S, total = 64, len(lens), max(lens), sum(lens)
    h = heads * d
    a, w, b = _tile_operands(total, 3 * h, h, dt)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    rows = torch.empty(total, dtype=torch.int32, device="cuda")
    ok(ttmi.ttmi_build_token_rows(ptr(cu), B, S, total, ptr(rows), stream()))
    q, k, v = (torch.full((B, heads, S, d), 7.0, dtype=a.dtype, device="cuda") for _ in range(3))
    args = _epi(bias=b, q=q, k=k, v=v, seq=S, heads=heads, head_dim=d, token_rows=rows, batch=B)
    name = ctypes.create_string_buffer(64)
    ok(ttmi.ttmi_gemm_describe(total, 3 * h, h, capi.EPI_QKV_SPLIT_PAD, ctypes.byref(args), TTMI_DTYPES[dt], name, 64))
    assert tile in name.value.decode(), name.value
    ok(ttmi.ttmi_gemm_fused(ptr(a), ptr(w), None, total, 3 * h, h, h, h, 3 * h, capi.EPI_QKV_SPLIT_PAD, ctypes.byref(args), TTMI_DTYPES[dt], stream()))
    want = a.double() @ w.double().T + b.double()
    room = (a.abs().double() @ w.abs().double().T + b.abs().double()) * (h // 16 + 2) * 2.0 ** -24 + {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt] * want.abs()
    want, room = (t.view(total, 3, heads, d) for t in (want, room))
    at = 0
    for i, n in enumerate(lens):
        for part, got in enumerate((q, k, v)):
            assert bool(((got[i, :, :n].double() - want[at:at + n, part].transpose(0, 1)).abs() <= room[at:at + n, part].transpose(0, 1)).all()), (i, part)
            assert bool((got[i, :, n:] == 7.0).all())
        at += n


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("fp32_residual", [False, True])
@pytest.mark.parametrize("m,n,k", [(2400, 1024, 1024), (3000, 768, 3072), (6000, 768, 768), (6275, 768, 3072), (9001, 1024, 1024), (11490, 768, 768)])
def test_projections_of_the_sizes_between_powers_of_two_with_layer_norm(ttmi, dt, fp32_residual, m, n, k):
    """Products that a LayerNorm follows, whole and in slices, at the row counts that tiles of 160 rows and columns are for.  Against 64 bits: with the residual in
    fp32 the sums' roundings alone, k / 16 + 20 of 2^-24 of the sum of magnitudes, through a LayerNorm that divides by no less than one; else the roundings of the
    product and of the result to the stored type, half of the last place of values up to 6 each."""
    a, w, b = _tile_operands(m, n, k, dt)
    gen = torch.Generator(device="cuda").manual_seed(k)
    res = torch.randn(m, n, generator=gen, device="cuda")
    gamma, beta = (torch.randn(n, generator=gen, device="cuda").mul_(0.1).add_(x).to(a.dtype) for x in (1.0, 0.0))
    stored = res if fp32_residual else res.to(a.dtype)
    out, out32 = torch.full((m + 1, n), 7.0, dtype=a.dtype, device="cuda"), torch.full((m + 1, n), 7.0, device="cuda") if fp32_residual else None
    ok(ttmi.ttmi_gemm_bias_layer_norm(ptr(a), ptr(w), ptr(out), None if fp32_residual else ptr(stored), ptr(stored) if fp32_residual else None, ptr(b), ptr(gamma),
                                      ptr(beta), ptr(out32), m, n, k, 1e-12, TTMI_DTYPES[dt], stream()))
    x = a.double() @ w.double().T + b.double() + stored.double()
    want = torch.nn.functional.layer_norm(x, (n, ), gamma.double(), beta.double(), 1e-12)
    sums = float((a.abs().double() @ w.abs().double().T + b.abs().double() + stored.abs().double()).max()) * (k // 16 + 20) * 2.0 ** -24
    gain = float(gamma.abs().max())
    half = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt]
    if fp32_residual:
        assert float((out32[:m].double() - want).abs().max()) <= 2 * gain * sums
        assert torch.equal(out[:m], out32[:m].to(a.dtype)) and bool((out32[m] == 7.0).all())
    else:
        assert float((out[:m].double() - want).abs().max()) <= 2 * gain * (sums + 6 * half) + 6 * half
    assert bool((out[m] == 7.0).all())
