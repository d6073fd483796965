"""GPU parity of the affine quantized matmul (ema_quantized_matmul, MLX quantized_matmul
with transpose=true as called by crates/ops/src/quant.rs:57-76) against the oracle's f64
restatement (oracle.qmatmul), through the C ABI.

Bars. For up to 32 rows of x the kernels multiply exactly and accumulate in f32, so every
output is within one rounding of the exact sum: |y - ref| <= 2^-8 |ref| (bf16; 2^-10 for
f16) plus 4e-5 * sum_k |x_k w_k| for the f32 accumulation. For more rows (K a multiple of
64) the weights are dequantised into the activation type first, as MLX's qmm kernels do
(oracle.dequantize_act), and the same bar holds against x times those weights; against the
exact sum they add at most half an ulp of the type per weight (2^-8 sum |x w| for bf16;
2^-11 for f16, plus 2^-25 sum |x| below f16's normal range); at the Qwen3-8B decode shape also the
bf16 bar of the other parity tests (max-abs 2e-2, mean-abs 2e-3). Separate q, k and v
calls into one q|k|v row (ldy > N) and the fused call are each within one rounding of the
oracle, so within two of each other: the property the reference checks at 1e-3
(crates/serve/tests/forward_separate.rs:80-91); repeated calls are bit-identical.
"""
import numpy as np
import pytest

from gpu_util import MAX_ABS, MEAN_ABS, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ema():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    import ema_attn

    ema_attn.lib()
    return ema_attn


def make(ora, seed, M, N, K, gs, bits, dtype="bf16", wstd=0.02):
    """Host inputs: x [M, K] (activation values as f32), packed w, scales/biases as f32
    values of the activation type, and the matching device tensors."""
    import torch

    td = torch.bfloat16 if dtype == "bf16" else torch.float16
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(td)
    w = (rng.standard_normal((N, K)) * wstd).astype(np.float32)
    wq, sb, bb = ora.minmax_quantize(w, gs, bits)
    s = torch.from_numpy(ora.f32_from_bf16(sb)).to(td)  # bf16 values, exact in f16 at this range
    b = torch.from_numpy(ora.f32_from_bf16(bb)).to(td)
    hx, hs, hb = x.float().numpy(), s.float().numpy(), b.float().numpy()
    d = (x.cuda(), torch.from_numpy(wq.view(np.int32)).cuda(), s.cuda(), b.cuda())
    return d, (hx, wq, hs, hb)


def dq_path(M, K):
    """Whether ema_quantized_matmul takes the dequantising GEMM (more than 32 rows, K a
    multiple of its 64-wide chunks)."""
    return M > 32 and K % 64 == 0


def check(ora, y, h, gs, bits, what, dtype="bf16", bar=False):
    hx, wq, hs, hb = h
    W = ora.dequantize(wq, hs, hb, gs, bits)
    mag = np.abs(hx).astype(np.float64) @ np.abs(W).T
    if dq_path(*hx.shape):
        Wt = ora.dequantize_act(wq, hs, hb, gs, bits, dtype).astype(np.float64)
        ref = hx.astype(np.float64) @ Wt.T
        exact = ora.qmatmul(hx, wq, hs, hb, gs, bits)
        half_ulp, floor = (2.0**-8, 0.0) if dtype == "bf16" else (2.0**-11, 2.0**-25)
        xs = np.abs(hx).astype(np.float64).sum(axis=1, keepdims=True)
        assert np.all(np.abs(ref - exact) <= (half_ulp * mag + floor * xs) * (1 + 1e-6)), f"{what}: dequantised weights"
    else:
        ref = ora.qmatmul(hx, wq, hs, hb, gs, bits)
    got = y.float().cpu().numpy().astype(np.float64)
    assert got.shape == ref.shape and np.all(np.isfinite(got)), what
    rel = 2.0**-8 if dtype == "bf16" else 2.0**-10
    err = np.abs(got - ref)
    over = err - (rel * np.abs(ref) + 4e-5 * mag)
    say(f"  {what}: max_abs={err.max():.3e} mean_abs={err.mean():.3e} worst margin={over.max():.3e} "
        f"(|y| max {np.abs(ref).max():.2f})")
    assert np.all(over <= 0), f"{what}: {int((over > 0).sum())} outputs beyond one rounding"
    if bar:
        assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS, what


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
def test_qmatmul_matches_oracle(ema, ora, dtype, bits, gs):
    for M, N, K in ((1, 96, 512), (5, 100, 1024), (16, 48, 256), (17, 64, 768), (32, 80, 2048)):
        say(f"qmatmul {dtype} bits={bits} gs={gs} M={M} N={N} K={K}")
        d, h = make(ora, M * 7 + N + K + gs + bits, M, N, K, gs, bits, dtype)
        y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
        check(ora, y, h, gs, bits, f"M={M} N={N} K={K}", dtype)


@pytest.mark.parametrize("M,N,bits", [(1, 6144, 4), (8, 6144, 4), (32, 6144, 4), (32, 4096, 4), (1, 6144, 8),
                                      (16, 6144, 8), (32, 6144, 8), (32, 4096, 8)])
def test_qmatmul_qwen3_8b_qkv_decode_shape(ema, ora, M, N, bits):
    # x [M, 4096] -> q|k|v [M, 6144] or o_proj [M, 4096], group 64: the one-row kernel (M = 1)
    # and the K-split kernel with one or two column tiles
    K, gs = 4096, 64
    say(f"qmatmul Qwen3-8B decode shape M={M} N={N} K={K} bits={bits}")
    d, h = make(ora, 1, M, N, K, gs, bits)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, "8B qkv", bar=True)


@pytest.mark.parametrize("M,N,bits", [(1, 7168, 4), (32, 7168, 4), (32, 5120, 4), (1, 5120, 8), (32, 7168, 8)])
def test_qmatmul_qwen3_14b_decode_shape(ema, ora, M, N, bits):
    # Qwen3-14B: hidden 5120, 40 query / 8 kv heads of 128, so x [M, 5120] -> q|k|v
    # [M, 7168] or o_proj [M, 5120], group 64 (K / 64 = 80 groups per row)
    K, gs = 5120, 64
    say(f"qmatmul Qwen3-14B decode shape M={M} N={N} K={K} bits={bits}")
    d, h = make(ora, 2, M, N, K, gs, bits)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, "14B qkv", bar=True)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_qmatmul_one_row_8bit_group_128_many_rows(ema, ora, dtype):
    # one row of x over 6144 weight rows at 8 bits, group 128: enough rows that the one-row
    # kernel gives each lane its most rows (two for this format, whose 32-dword groups
    # would not fit four to a lane)
    M, N, K, gs, bits = 1, 6144, 2048, 128, 8
    say(f"qmatmul one-row {dtype} bits={bits} gs={gs} N={N} K={K}")
    d, h = make(ora, 11, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, "one row, 8-bit group 128", dtype)


@pytest.mark.parametrize("M,gs,dtype", [(20, 128, "bf16"), (12, 64, "f16")])
def test_qmatmul_8bit_wide_rows(ema, ora, M, gs, dtype):
    # 8-bit weights, more column tiles than CUs: the K-split kernel, two column tiles; ragged
    # rows of x (test_qmatmul_scales_off_alignment runs the staged kernels at these sizes)
    N, K, bits = 6144, 4096, 8
    say(f"qmatmul 8-bit M={M} N={N} K={K} gs={gs} {dtype}")
    d, h = make(ora, 60 + M, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)


@pytest.mark.parametrize("M,N,K,gs,bits,dtype", [
    (64, 256, 1024, 64, 4, "bf16"),     # tiled GEMM: one 128-row tile, several column tiles
    (300, 256, 1024, 64, 4, "bf16"),    # ragged last row tile
    (130, 100, 2048, 128, 4, "bf16"),   # group 128: 128-wide chunks; ragged columns
    (500, 70, 1024, 128, 8, "f16"),
    (96, 80, 512, 32, 8, "bf16"),
    (2048, 256, 2048, 64, 4, "bf16"),   # a prefill chunk's rows
    (40, 48, 320, 32, 4, "bf16"),       # K / gs = 10
    (70, 64, 320, 32, 8, "f16"),
    (40, 48, 288, 32, 4, "bf16"),       # K not a multiple of 64: the streaming kernel
    (70, 64, 288, 32, 8, "f16"),
    (257, 129, 512, 32, 4, "f16"),      # ragged tiles in both directions
])
def test_qmatmul_prefill_rows(ema, ora, M, N, K, gs, bits, dtype):
    say(f"qmatmul prefill rows M={M} N={N} K={K} gs={gs} bits={bits} {dtype}")
    d, h = make(ora, M + N, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)


# The last column is the kernel and its tiles on 256 CUs, which tests/test_qmm_route.py checks on
# the CPU against the rules that the launches use.
KSPLIT_TILES = [
    # the K-split GEMM: each of its tiles (row x column tiles of 16), ragged last rows and
    # columns, at most one unit of 128 k per wave
    (33, 100, 128, 32, 4, "bf16", "qgemm_ks 3 2"),      # one unit
    (48, 30, 384, 32, 8, "f16", "qgemm_ks 3 2"),        # three units
    (64, 5100, 256, 64, 4, "f16", "qgemm_ks 4 2"),
    (157, 4093, 256, 64, 4, "bf16", "qgemm_ks 5 2"),
    (157, 4090, 512, 128, 8, "bf16", "qgemm_ks 5 2"),
    (96, 6140, 256, 64, 8, "bf16", "qgemm_ks 3 3"),
    (101, 6144, 256, 32, 4, "bf16", "qgemm_ks 4 3"),
    (127, 6143, 256, 32, 8, "f16", "qgemm_ks 4 3"),
    (159, 6142, 512, 128, 4, "f16", "qgemm_ks 5 3"),
    (140, 5437, 256, 64, 4, "bf16", "qgemm_ks 3 4"),
    (140, 5440, 256, 64, 8, "f16", "qgemm_ks 3 4"),
    (190, 5439, 256, 32, 4, "bf16", "qgemm_ks 4 4"),
    # each tile again with several units per wave (the refill of the next unit, the walk's wrap
    # at the end of K, slots written again), equal and unequal shares of the waves
    (80, 64, 1152, 32, 4, "bf16", "qgemm_ks 3 2"),      # nine units: one wave takes two
    (50, 70, 2560, 64, 8, "bf16", "qgemm_ks 3 2"),      # twenty units
    (64, 5100, 1152, 32, 4, "bf16", "qgemm_ks 4 2"),
    (61, 5437, 2176, 32, 8, "bf16", "qgemm_ks 4 2"),
    (157, 4096, 4096, 64, 4, "bf16", "qgemm_ks 5 2"),
    (157, 4093, 2304, 64, 8, "f16", "qgemm_ks 5 2"),
    (96, 5437, 2304, 64, 4, "f16", "qgemm_ks 3 3"),
    (93, 6140, 1152, 32, 8, "bf16", "qgemm_ks 3 3"),
    (127, 6140, 2176, 32, 4, "bf16", "qgemm_ks 4 3"),
    (125, 6144, 2304, 64, 8, "bf16", "qgemm_ks 4 3"),
    (157, 6144, 4096, 64, 4, "bf16", "qgemm_ks 5 3"),
    (140, 5437, 2304, 64, 4, "f16", "qgemm_ks 3 4"),
    (139, 5440, 1152, 32, 8, "bf16", "qgemm_ks 3 4"),
    (190, 5437, 2176, 32, 4, "bf16", "qgemm_ks 4 4"),
    (40, 64, 9728, 32, 4, "bf16", "qgemm_ks 3 2"),      # 304 groups: scales staged in two passes
    (40, 70, 9728, 32, 8, "f16", "qgemm_ks 3 2"),
]

KSPLIT_DECODE = [
    # exact products split over K (K >= 2048; 8 bits and up to 16 rows K >= 4096): 8, 16 and 32
    # rows, one and two column tiles, ragged columns, units that do not divide among the eight
    # waves
    (2, 70, 2048, 64, 4, "bf16", "qmv_ks 1 1"),
    (8, 33, 2176, 32, 4, "f16", "qmv_ks 1 1"),          # 17 units
    (9, 100, 4096, 128, 8, "bf16", "qmv_ks 1 1"),
    (16, 4099, 2048, 64, 4, "bf16", "qmv_ks 1 2"),      # ragged
    (17, 48, 2560, 64, 8, "f16", "qmv_ks 2 1"),         # 20 units
    (31, 4110, 2304, 32, 4, "bf16", "qmv_ks 2 2"),      # 18 units
    (32, 8200, 2048, 64, 4, "bf16", "qmv_ks 2 1"),      # more than two rounds: one column tile
    (5, 4097, 4608, 64, 8, "bf16", "qmv_ks 1 2"),       # 36 units: a fifth turn for four waves
    (4, 40, 9728, 32, 4, "f16", "qmv_ks 1 1"),          # 304 groups: scales staged in two passes
    # calls that stay with the staged kernels: short K with one and two column tiles, 8 bits and
    # up to 16 rows below K = 4096, 384 groups (past the LDS bound of the K-split kernel)
    (16, 4112, 1024, 64, 4, "bf16", "qmv 16 2"),
    (32, 4109, 1024, 64, 4, "f16", "qmv 32 2"),
    (8, 4100, 1024, 32, 4, "bf16", "qmv 8 2"),
    (9, 100, 3072, 64, 8, "bf16", "qmv 16 1"),
    (16, 6144, 2560, 64, 8, "bf16", "qmv 16 2"),
    (3, 40, 12288, 32, 4, "bf16", "qmv 4 1"),
    (17, 40, 14848, 32, 4, "bf16", "qmvx 32 1"),
    (2, 8213, 2048, 64, 4, "bf16", "qmv 2 1"),          # more columns than one round holds
    (6, 16390, 2048, 64, 4, "f16", "qmv 8 2"),
    (24, 8209, 2048, 64, 8, "bf16", "qmv 32 2"),
    (9, 100, 3968, 128, 8, "bf16", "qmm 1 1"),          # 31 groups: the streaming kernel
]

DQ_TILES = [
    # tiles of 128, 192 and 256 rows of the dequantising GEMM (chosen by the rounds on 256 CUs),
    # ragged in both directions, scales loaded per chunk and, from 32 groups on, staged in LDS
    (1020, 4093, 128, 32, 4, "bf16", "qgemm_dq 2 1"),   # 256 tiles of 128 rows
    (1000, 4096, 192, 64, 8, "f16", "qgemm_dq 2 1"),    # the same, three groups
    (1530, 4090, 256, 32, 8, "bf16", "qgemm_dq 3 1"),   # 256 tiles of 192 rows
    (1531, 4096, 192, 64, 4, "f16", "qgemm_dq 3 1"),
    (2040, 4091, 128, 32, 4, "f16", "qgemm_dq 4 1"),    # 256 tiles of 256 rows
    (2047, 4096, 64, 64, 8, "bf16", "qgemm_dq 4 1"),    # one chunk
    (80, 64, 1152, 64, 4, "bf16", "qgemm_dq 2 1"),      # 18 groups: not the K-split kernel
    (1020, 4093, 1024, 32, 4, "bf16", "qgemm_dq_staged 2 1"),
    (1530, 4090, 1024, 32, 8, "bf16", "qgemm_dq_staged 3 1"),
    (1531, 4096, 2048, 64, 4, "f16", "qgemm_dq_staged 3 1"),
    (2040, 4091, 1024, 32, 4, "f16", "qgemm_dq_staged 4 1"),
    (2047, 4096, 2048, 64, 8, "bf16", "qgemm_dq_staged 4 1"),
]

# Scales and biases that start 4 or 2 bytes past a 16-byte boundary (the entry asks for their
# element's alignment only): the K-split kernels and the staged scales of the dequantising GEMM
# need 8 bytes.
OFF_ALIGNMENT = [
    (20, 6144, 4096, 128, 8, "bf16", 4, "qmvx 32 2"),
    (12, 6144, 4096, 64, 8, "f16", 4, "qmv 16 2"),
    (32, 4096, 4096, 64, 8, "bf16", 4, "qmv 32 1"),
    (157, 4093, 2048, 64, 4, "bf16", 4, "qgemm_dq 2 1"),
    (157, 300, 2048, 64, 8, "f16", 2, "qgemm_dq 2 1"),
]


def same_bits_elsewhere(ema, d, y, gs, bits):
    """The call again into a view with an odd row stride (2-byte stores) and from rows of x that
    lie further apart: the same bits, nothing written beside the view."""
    import torch

    M, N, K = y.shape[0], y.shape[1], d[0].shape[1]
    wide = torch.full((M, N + 3), 7.0, dtype=y.dtype, device="cuda")
    ema.quantized_matmul(*d, group_size=gs, bits=bits, out=wide[:, 1:N + 1])
    wx = torch.full((M, K + 72), float("nan"), dtype=y.dtype, device="cuda")
    wx[:, :K] = d[0]
    strided = ema.quantized_matmul(wx[:, :K], *d[1:], group_size=gs, bits=bits)
    torch.cuda.synchronize()
    assert torch.equal(wide[:, 1:N + 1].contiguous().view(torch.int16), y.view(torch.int16))
    assert torch.all(wide[:, :1] == 7.0) and torch.all(wide[:, N + 1:] == 7.0)
    assert torch.equal(strided.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("M,N,K,gs,bits,dtype,route", KSPLIT_TILES)
def test_qmatmul_ksplit_tiles(ema, ora, M, N, K, gs, bits, dtype, route):
    say(f"qmatmul K-split M={M} N={N} K={K} gs={gs} bits={bits} {dtype} ({route})")
    d, h = make(ora, M + N + K, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)
    same_bits_elsewhere(ema, d, y, gs, bits)


@pytest.mark.parametrize("M,N,K,gs,bits,dtype,route", KSPLIT_DECODE)
def test_qmatmul_ksplit_decode_rows(ema, ora, M, N, K, gs, bits, dtype, route):
    say(f"qmatmul K-split decode M={M} N={N} K={K} gs={gs} bits={bits} {dtype} ({route})")
    d, h = make(ora, M + N + K, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)
    same_bits_elsewhere(ema, d, y, gs, bits)


@pytest.mark.parametrize("M,N,K,gs,bits,dtype,route", DQ_TILES)
def test_qmatmul_dequantising_tiles(ema, ora, M, N, K, gs, bits, dtype, route):
    say(f"qmatmul dequantising tiles M={M} N={N} K={K} gs={gs} bits={bits} {dtype} ({route})")
    d, h = make(ora, M + N + K, M, N, K, gs, bits, dtype)
    y = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)
    same_bits_elsewhere(ema, d, y, gs, bits)


@pytest.mark.parametrize("M,N,K,gs,bits,dtype,past,route", OFF_ALIGNMENT)
def test_qmatmul_scales_off_alignment(ema, ora, M, N, K, gs, bits, dtype, past, route):
    import torch

    say(f"qmatmul scales {past} bytes past 16 M={M} N={N} K={K} gs={gs} bits={bits} {dtype} ({route})")
    d, h = make(ora, M + N + K + past, M, N, K, gs, bits, dtype)

    def shifted(t):
        flat = torch.empty(t.numel() + past // 2, dtype=t.dtype, device="cuda")
        v = flat[past // 2:].view(t.shape)
        v.copy_(t)
        assert v.data_ptr() % 16 == past
        return v

    y = ema.quantized_matmul(d[0], d[1], shifted(d[2]), shifted(d[3]), group_size=gs, bits=bits)
    check(ora, y, h, gs, bits, f"M={M}", dtype)


@pytest.mark.parametrize("M,N,K", [(1, 192, 1024), (32, 192, 1024), (256, 192, 1024), (1000, 4096, 192),
                                   (16, 4099, 4096), (32, 4096, 4096), (157, 4096, 2304)])
def test_qmatmul_graph_replay(ema, ora, M, N, K):
    # captured in a HIP graph and replayed several times with eager work between the
    # replays: every replay equals the eager call (no memsets or host state in the call)
    import torch

    gs, bits = 64, 4
    say(f"qmatmul graph replay M={M} N={N} K={K}")
    d, _ = make(ora, 5 + M, M, N, K, gs, bits)
    y_eager = ema.quantized_matmul(*d, group_size=gs, bits=bits)
    torch.cuda.synchronize()
    y = torch.empty_like(y_eager)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            ema.quantized_matmul(*d, group_size=gs, bits=bits, out=y, stream=s)
    torch.cuda.synchronize()
    for i in range(3):
        y.fill_(float(i + 3))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), y_eager.view(torch.int16)), f"replay {i}"


def test_qmatmul_separate_pieces_equal_fused(ema, ora):
    # run_qkv's separate branch (projection.rs:119-125) writing its three pieces straight
    # into one q|k|v row (ldy = 6144): columns of other pieces untouched, every piece and the
    # fused call within one rounding of the oracle, hence of each other (the reference checks
    # max-abs 1e-3, forward_separate.rs:80-91; the 4096-column piece and the fused call may be
    # tiled differently, which reorders the f32 sums)
    import torch

    M, K, gs, bits = 8, 4096, 64, 4
    sizes = (4096, 1024, 1024)
    say(f"qmatmul separate vs fused M={M} pieces={sizes}")
    made = [make(ora, 50 + i, M, n, K, gs, bits) for i, n in enumerate(sizes)]
    parts = [m[0] for m in made]
    x = parts[0][0]
    fused = ema.quantized_matmul(x, torch.cat([p[1] for p in parts]), torch.cat([p[2] for p in parts]),
                                 torch.cat([p[3] for p in parts]), group_size=gs, bits=bits)
    qkv = torch.full((M, sum(sizes)), 7.0, dtype=torch.bfloat16, device="cuda")
    col = 0
    for (_, w, s, b), n in zip(parts, sizes):
        if col == 0:
            assert torch.all(qkv[:, n:] == 7.0)
        ema.quantized_matmul(x, w, s, b, group_size=gs, bits=bits, out=qkv[:, col:col + n])
        if col + n < qkv.shape[1]:
            assert torch.all(qkv[:, col + n:] == 7.0), "wrote past its piece"
        col += n
    torch.cuda.synchronize()
    col = 0
    for (_, h), n in zip(made, sizes):
        h = (made[0][1][0],) + h[1:]  # every piece reads the same x
        check(ora, qkv[:, col:col + n], h, gs, bits, f"piece at column {col}")
        col += n
    hx = made[0][1][0]
    fused_h = (hx, np.concatenate([m[1][1] for m in made]), np.concatenate([m[1][2] for m in made]),
               np.concatenate([m[1][3] for m in made]))
    check(ora, fused, fused_h, gs, bits, "fused")
    # the two results are each within one rounding (plus the f32 accumulation allowance)
    # of the exact product, so within the sum of both allowances of each other
    a, b = qkv.float().cpu().numpy().astype(np.float64), fused.float().cpu().numpy().astype(np.float64)
    W = ora.dequantize(fused_h[1], fused_h[2], fused_h[3], gs, bits)
    mag = np.abs(hx).astype(np.float64) @ np.abs(W).T
    assert np.all(np.abs(a - b) <= 2.0**-7 * np.maximum(np.abs(a), np.abs(b)) + 8e-5 * mag)
    say(f"  separate vs fused: {int((a != b).sum())} of {a.size} outputs differ, max {np.abs(a - b).max():.3e}")


def test_qmatmul_strided_rows_and_determinism(ema, ora):
    import torch

    M, N, K, gs, bits = 9, 128, 1024, 64, 8
    say("qmatmul strided x rows, repeat determinism")
    d, h = make(ora, 3, M, N, K, gs, bits)
    x, w, s, b = d
    wide = torch.zeros((M, K + 64), dtype=x.dtype, device="cuda")
    wide[:, :K] = x
    y1 = ema.quantized_matmul(wide[:, :K], w, s, b, group_size=gs, bits=bits)
    y2 = ema.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    torch.cuda.synchronize()
    assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
    check(ora, y1, h, gs, bits, "strided")


@pytest.mark.parametrize("M", [4, 64])
def test_qmatmul_extreme_fields_and_groups(ema, ora, M):
    # all-zero and all-max fields, zero and negative scales, large biases: the C + q
    # offset and the bias term cancel exactly (4 rows); dequantised into bf16 (64 rows)
    import torch

    N, K, gs = 32, 512, 64
    for bits in (4, 8):
        say(f"qmatmul extreme fields bits={bits} M={M}")
        rng = np.random.default_rng(bits)
        q = np.where(rng.random((N, K)) < 0.5, 0, (1 << bits) - 1).astype(np.uint32)
        wq = ora.pack_bits(q, bits)
        s = rng.choice([0.0, -0.015625, 0.03125, 1.0], (N, K // gs)).astype(np.float32)
        b = rng.choice([0.0, -3.0, 2.5, 100.0], (N, K // gs)).astype(np.float32)
        x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(torch.bfloat16)
        args = (x.cuda(), torch.from_numpy(wq.view(np.int32)).cuda(), torch.from_numpy(s).to(torch.bfloat16).cuda(),
                torch.from_numpy(b).to(torch.bfloat16).cuda())
        y = ema.quantized_matmul(*args, group_size=gs, bits=bits)
        check(ora, y, (x.float().numpy(), wq, s, b), gs, bits, f"extreme bits={bits}")
