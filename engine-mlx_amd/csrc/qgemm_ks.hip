// Dequantising GEMM for some tens to some hundreds of rows of x (a chat turn, a short
// prompt): y = x W^T over MLX-packed weights, each weight rounded once into the activation
// type, w = round(fma(s, q, b)), as qgemm_dq_kernel does.
//
// At 157 rows the 256 x 128 tiles of qgemm_dq_kernel are 48 workgroups for 6144 columns: a
// fifth of the chip. Small tiles fill it, but a small tile shared by several waves through
// LDS spends its time on operand reads and barriers. Here the eight waves of a workgroup
// split K instead: each multiplies the whole 16 MT x 16 NT tile over its own units of 128 k
// (wave, wave + 8, ... of a walk that starts elsewhere in each workgroup), with no barrier
// until the eight partial tiles are added in f32 at the end, in a fixed order (repeated
// calls are bit-identical).
//
// Loads. Consecutive lanes read consecutive 16-byte pieces of a row (8 lanes a 128-byte line
// of x): a quarter wave of a buffer load touches two lines. Straight loads in MFMA layout
// (lane = row + 16 * piece) touch 16 lines per quarter wave and took 54 to 67 cycles per
// load, whatever their size. The registers then pass through a few KB of LDS that belong to
// the wave (write by rows, read in MFMA layout; wave_lds_fence in between, which emits nothing:
// a wave's LDS operations execute in order, and the fence has the compiler keep that order)
// while the next unit's loads are in flight behind them. Scales and biases are staged once per
// workgroup as {scale, bias} pairs.
// MFMA step i (32 k) needs fields 8 j .. 8 j + 7 of the step in lane row j:
// - 4 bits: dword i of lane row j holds fields 32 j + 8 i ..; a 4 x 4 transpose between lane
//   rows and registers (v_permlane16_swap, v_permlane32_swap: four instructions per 16
//   bytes) gives register i, lane row j fields 32 i + 8 j ..;
// - 8 bits: v_permlane32_swap alone gives lane row j of step i the 8 bytes at k
//   32 i + 16 (j % 2) + 8 (j / 2); x is read in that order (any order of k within a step
//   gives the same products).
//
// Measured (4 bits, group 64, K = 4096, M = 157): N = 6144 18.3 us (5 x 3 tiles), N = 4096
// 15.8 us (5 x 2), against 55.6 and 54.4 us of qgemm_dq_kernel; with MFMA-layout loads 26.0
// and 24.1. What bounds it: the dequantisation's VALU (23 per 8 weights), LDS traffic (every
// byte written and read once) and MFMA, which add up rather than overlap; staging the next
// line before the current one's MFMAs, or other wave priorities, changed nothing.
#include "qmatmul_common.hpp"

#include <type_traits>

namespace ema {
namespace {

constexpr uint32_t kSlots = 4, kSlot = 2048;
static_assert(kKsWaves * kSlots * kSlot == kKsSlotBytes, "the plan counts these slots");

__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Scales and biases of the tile's weight rows, in LDS as {scale, bias} pairs, rows of
// group_stride pairs (an odd number of 16-byte pieces, so that the 16 rows of a tile are read
// without bank conflicts): staged once per workgroup, since a wave's own loads of a few bytes
// per row and unit would each cost a whole cache line. A lane takes four groups of a row, a
// wave as many rows as its lanes cover; groups past 256 (long K) follow in a loop. Staged
// before the first weights and x are requested: requesting those in between, ahead of the LDS
// writes, took 0.2 to 0.3 us more at up to 16 rows.
template <int NT>
struct GroupStage {
  static constexpr int kRows = 16 * NT, kPer = kRows / kKsWaves;
  u32x2 sv[kPer], bv[kPer];
  uint32_t rows, row0, g0;  // rows per wave and pass, this lane's first row and groups

  __device__ __forceinline__ GroupStage(uint32_t G, uint32_t wave, uint32_t lane) {
    const uint32_t pieces = G / 4;
    const uint32_t sh = pieces >= 64 ? 6u : pieces <= 1 ? 0u : 32u - __builtin_clz(pieces - 1);
    rows = 64u >> sh;
    row0 = wave * rows + (lane >> sh);
    g0 = 4 * (lane & ((1u << sh) - 1));
  }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t S, __amdgpu_buffer_rsrc_t B, uint32_t G, int rows_n,
                                       uint32_t g) {
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      if (r * kKsWaves * rows >= kRows) break;
      const uint32_t row = row0 + r * kKsWaves * rows;
      const uint32_t off = row < (uint32_t)rows_n && g < G ? (row * G + g) * 2 : kOffRow;
      sv[r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(S, off, 0, 0));
      bv[r] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(B, off, 0, 0));
    }
  }
  __device__ __forceinline__ void store(uint32_t* groups, uint32_t G, uint32_t g) const {
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      if (r * kKsWaves * rows >= kRows) break;
      const uint32_t row = row0 + r * kKsWaves * rows;
      if (row >= kRows || g >= G) continue;
      *reinterpret_cast<u32x4*>(groups + row * group_stride(G) + g) =
          u32x4{pair(sv[r][0], bv[r][0], kSelLo), pair(sv[r][0], bv[r][0], kSelHi),
                pair(sv[r][1], bv[r][1], kSelLo), pair(sv[r][1], bv[r][1], kSelHi)};
    }
  }
};

template <int BITS, int GS, bool F16, int MT, int NT>
__global__ __launch_bounds__(64 * kKsWaves) void qgemm_ks_kernel(QmmArgs a, uint32_t slot_off) {
  constexpr int kWL = BITS / 4;  // 16-byte weight loads per unit and column tile
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const KsTile tile = ks_tile_of((int)blockIdx.x, (int)gridDim.x, a.mtiles);
  const int nt = tile.nt, mt = tile.mt;
  const int n0 = nt * 16 * NT, m0 = mt * 16 * MT;
  const int rows_n = min(16 * NT, a.N - n0), rows_m = min(16 * MT, a.M - m0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;

  const uint32_t wrow = (uint32_t)a.K * BITS / 8, xrow = (uint32_t)a.ldx * 2, G2 = (uint32_t)a.G * 2;
  const auto X = rsrc(a.x + (int64_t)m0 * xrow, (rows_m - 1) * xrow + (uint32_t)a.K * 2);
  const auto W = rsrc(a.w + (int64_t)n0 * wrow, rows_n * wrow);
  const auto S = rsrc(a.s + (int64_t)n0 * G2, rows_n * G2);
  const auto B = rsrc(a.b + (int64_t)n0 * G2, rows_n * G2);
  // x: a load covers 8 rows x 128 bytes, weights: 16 rows x 64 bytes (4 bits) or 8 x 128
  uint32_t xoff[MT][2], woff[NT][kWL];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 16 * t + 8 * h + (lane >> 3);
      xoff[t][h] = row < rows_m ? row * xrow + 16 * (lane & 7) : kOffRow;
    }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < kWL; ++e) {
      const int row = BITS == 4 ? 16 * t + (lane >> 2) : 16 * t + 8 * e + (lane >> 3);
      woff[t][e] = row < rows_n ? row * wrow + 16 * (BITS == 4 ? lane & 3 : lane & 7) : kOffRow;
    }

  const int units = a.K / kUnit;
  // units wave, wave + 8, ... of a walk of K that starts at another place in each workgroup
  const int count = (units - wave + kKsWaves - 1) / kKsWaves;
  int u = ((nt / 8 * a.mtiles + mt) * kKsWaves + wave) % units;

  u32x4 xr[2][MT][2], wr[NT][kWL];  // x: [line of the unit][row tile][half of its rows]
  auto load_w = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < kWL; ++e)
        wr[t][e] = __builtin_amdgcn_raw_buffer_load_b128(W, woff[t][e], u * (kUnit * BITS / 8), 0);
  };
  auto load_x = [&](int u, int ln, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      xr[ln][t][h] = __builtin_amdgcn_raw_buffer_load_b128(X, xoff[t][h] + 128 * ln, u * (kUnit * 2), 0);
  };

  uint32_t* const groups = reinterpret_cast<uint32_t*>(smem);
  const uint32_t gs4 = group_stride((uint32_t)a.G);
  const uint32_t* const gl = groups + c * gs4;  // the pairs of this lane's column
  GroupStage<NT> gst((uint32_t)a.G, wave, lane);
  gst.load(S, B, (uint32_t)a.G, rows_n, gst.g0);
  gst.store(groups, (uint32_t)a.G, gst.g0);
  for (uint32_t g = 256; g < (uint32_t)a.G; g += 256) {
    gst.load(S, B, (uint32_t)a.G, rows_n, g + gst.g0);
    gst.store(groups, (uint32_t)a.G, g + gst.g0);
  }

  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The wave's LDS scratch: slots of 16 rows x 128 bytes, 16-byte piece p of row r at
  // p ^ ((r >> 1) & 7); 16 rows x 64 bytes for 4-bit weights, piece p at p ^ (r >> 2) (both
  // free of bank conflicts). A slot is written again four exchanges later, behind the fences of
  // the three in between.
  uint8_t* const slots = smem + slot_off + (uint32_t)wave * (kSlots * kSlot);
  const uint32_t wr8 = lane >> 3, wp8 = lane & 7, wr4 = lane >> 2;
  const uint32_t put8 = wr8 * 128 + 16 * (wp8 ^ (wr8 >> 1));  // rows 0 .. 7; rows 8 .. 15 below
  const uint32_t put8h = (wr8 + 8) * 128 + 16 * (wp8 ^ ((wr8 + 8) >> 1));
  const uint32_t put4 = wr4 * 64 + 16 * ((lane & 3) ^ (wr4 >> 2));
  const uint32_t xj = BITS == 4 ? j : 2 * (j & 1) + (j >> 1);  // x piece of lane row j in a step
  uint32_t slot = 0;
  auto next_slot = [&]() __attribute__((always_inline)) {
    uint8_t* const p = slots + slot * kSlot;
    slot = (slot + 1) % kSlots;
    return p;
  };

  // one unit; the loads of the next one go out as the registers of this one are read
  auto unit = [&](int cur, int next, auto refill) __attribute__((always_inline)) {
    uint32_t wd[NT][4 * kWL];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint8_t* const sl = next_slot();
      if constexpr (BITS == 4) {
        *reinterpret_cast<u32x4*>(sl + put4) = wr[t][0];
        wave_lds_fence();
        const u32x4 v = *reinterpret_cast<const u32x4*>(sl + c * 64 + 16 * (j ^ (c >> 2)));
        uint32_t d0 = v[0], d1 = v[1], d2 = v[2], d3 = v[3];
        swap16(d0, d1);
        swap16(d2, d3);
        swap32(d0, d2);
        swap32(d1, d3);
        wd[t][0] = d0;
        wd[t][1] = d1;
        wd[t][2] = d2;
        wd[t][3] = d3;
      } else {
        *reinterpret_cast<u32x4*>(sl + put8) = wr[t][0];
        *reinterpret_cast<u32x4*>(sl + put8h) = wr[t][kWL - 1];
        wave_lds_fence();
#pragma unroll
        for (int e = 0; e < kWL; ++e) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(sl + c * 128 + 16 * ((4 * e + j) ^ (c >> 1)));
          uint32_t d0 = v[0], d1 = v[1], d2 = v[2], d3 = v[3];
          swap32(d0, d2);
          swap32(d1, d3);
          wd[t][4 * e] = d0;
          wd[t][4 * e + 1] = d1;
          wd[t][4 * e + 2] = d2;
          wd[t][4 * e + 3] = d3;
        }
      }
    }
    if constexpr (refill.value) load_w(next);
    // x by row tile, each multiplied right behind its reads: the fences keep the exchanges in
    // this order, and all row tiles of a line read first took 20 registers too many at 5 x 3
    // (4 bits, N = 6144, K = 4096, 157 rows: 24.1 us against 18.4)
#pragma unroll
    for (int ln = 0; ln < 2; ++ln) {
      u32x4 wv[2][NT];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int st = 2 * ln + h;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const uint32_t sb = gl[16 * t * gs4 + cur * (kUnit / GS) + st * 32 / GS];
          const float s = act_to_f32<F16>(sb & 0xffffu), b = act_to_f32<F16>(sb >> 16);
          if constexpr (BITS == 4) wv[h][t] = dequant8<BITS, F16>(wd[t][st], 0u, s, b);
          else wv[h][t] = dequant8<BITS, F16>(wd[t][2 * st], wd[t][2 * st + 1], s, b);
        }
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint8_t* const sl = next_slot();
        *reinterpret_cast<u32x4*>(sl + put8) = xr[ln][t][0];
        *reinterpret_cast<u32x4*>(sl + put8h) = xr[ln][t][1];
        wave_lds_fence();
        u32x4 xv[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          xv[h] = *reinterpret_cast<const u32x4*>(sl + c * 128 + 16 * ((4 * h + xj) ^ (c >> 1)));
        if constexpr (refill.value) load_x(next, ln, t);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[n][t] = mma<F16>(wv[h][n], xv[h], acc[n][t]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (count > 0) {
    load_w(u);
#pragma unroll
    for (int ln = 0; ln < 2; ++ln)
#pragma unroll
      for (int t = 0; t < MT; ++t) load_x(u, ln, t);
  }
  __syncthreads();
  if (count > 0) {
    for (int i = 1; i < count; ++i) {
      const int next = u + kKsWaves >= units ? u + kKsWaves - units : u + kKsWaves;
      unit(u, next, std::true_type{});
      u = next;
    }
    unit(u, 0, std::false_type{});
  }
  __syncthreads();  // the partial tiles take the place of the scales

  // add the eight partial tiles: lane (c, j) of tile (n, m) holds columns 16 n + 4 j .. + 3
  // of row 16 m + c
  f32x4* const red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((wave * MT + m) * NT + n) * 64 + lane] = acc[n][m];
  __syncthreads();
  const bool wide = (((uintptr_t)a.y | (uint64_t)a.ldy * 2) & 7) == 0;
  for (int e = threadIdx.x; e < MT * NT * 64; e += 64 * kKsWaves) {
    f32x4 v = red[e];
#pragma unroll
    for (int w = 1; w < kKsWaves; ++w) {
      const f32x4 p = red[w * (MT * NT * 64) + e];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] += p[q];
    }
    const int tile = e >> 6, m = tile / NT, n = tile % NT;
    const int row = 16 * m + (e & 15), col = 16 * n + 4 * ((e >> 4) & 3);
    if (row >= rows_m || col >= rows_n) continue;
    uint16_t* const y = reinterpret_cast<uint16_t*>(a.y) + (int64_t)(m0 + row) * a.ldy + n0 + col;
    uint16_t o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = f32_to_act<F16>(v[q]);
    if (wide && col + 4 <= rows_n) {
      *reinterpret_cast<u32x2*>(y) = u32x2{o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16};
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (col + q < rows_n) y[q] = o[q];
    }
  }
}

// The exact products of up to 32 rows (see qmatmul.hip), split over K the same way: per group
// an MFMA chain over C + q and one over ones, combined as tot += s a_q + (b - C s) a_1. Four
// units of weights (the HBM stream) and two of x are in flight per wave; a unit past the
// wave's share loads nothing and is skipped.
// Bound by the load round trips of a launch of few waves and, at 32 rows, by VALU and MFMA (the
// chain over ones runs once per row tile: a wave owns all columns of the workgroup). Measured,
// 4 bits, group 64, K = 4096, against qmatmul.hip's staged kernels: N = 6144 10.8 us against
// 14.6 at 32 rows, 7.5 against 9.7 at 8; N = 4096 8.7 against 12.2 and 6.0 against 7.3. Those
// stage x by DMA with a quarter wave on 16 rows (64 line accesses per KB) and pass a barrier
// per chunk.
template <int BITS, int GS, bool F16, int MX, int NT>
__global__ __launch_bounds__(64 * kKsWaves) void qmv_ks_kernel(QmmArgs a, uint32_t slot_off) {
  using F = Fields<BITS, F16>;
  constexpr int MT = MX > 16 ? 2 : 1;
  constexpr int H = MX > 8 ? 2 : 1;  // halves of 8 rows loaded per row tile
  constexpr int kWL = BITS / 4, kRows = 16 * NT, kXU = 2, kWU = 4;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int n0 = blockIdx.x * kRows;
  const int rows_n = min(kRows, a.N - n0), rows_m = a.M;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, j = lane >> 4;

  const uint32_t wrow = (uint32_t)a.K * BITS / 8, xrow = (uint32_t)a.ldx * 2, G2 = (uint32_t)a.G * 2;
  const auto X = rsrc(a.x, (rows_m - 1) * xrow + (uint32_t)a.K * 2);
  const auto W = rsrc(a.w + (int64_t)n0 * wrow, rows_n * wrow);
  const auto S = rsrc(a.s + (int64_t)n0 * G2, rows_n * G2);
  const auto B = rsrc(a.b + (int64_t)n0 * G2, rows_n * G2);
  uint32_t xoff[MT][H], woff[NT][kWL];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int row = 16 * t + 8 * h + (lane >> 3);
      xoff[t][h] = row < rows_m ? row * xrow + 16 * (lane & 7) : kOffRow;
    }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < kWL; ++e) {
      const int row = BITS == 4 ? 16 * t + (lane >> 2) : 16 * t + 8 * e + (lane >> 3);
      woff[t][e] = row < rows_n ? row * wrow + 16 * (BITS == 4 ? lane & 3 : lane & 7) : kOffRow;
    }

  const int units = a.K / kUnit;
  const int count = (units - wave + kKsWaves - 1) / kKsWaves;  // units wave, wave + 8, ...
  u32x4 xr[kXU][2][MT][H], wr[kWU][NT][kWL];
  auto load_w = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t none = i < count ? 0u : kOffRow, u = i < count ? wave + i * kKsWaves : 0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < kWL; ++e)
        wr[slot][t][e] = __builtin_amdgcn_raw_buffer_load_b128(W, woff[t][e] | none, u * (kUnit * BITS / 8), 0);
  };
  auto load_x = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t none = i < count ? 0u : kOffRow, u = i < count ? wave + i * kKsWaves : 0;
#pragma unroll
    for (int ln = 0; ln < 2; ++ln)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < H; ++h)
          xr[slot][ln][t][h] =
              __builtin_amdgcn_raw_buffer_load_b128(X, (xoff[t][h] | none) + 128 * ln, u * (kUnit * 2), 0);
  };

  uint32_t* const groups = reinterpret_cast<uint32_t*>(smem);
  const uint32_t gs4 = group_stride((uint32_t)a.G);
  const uint32_t* const gl = groups + c * gs4;  // the pairs of this lane's column
  GroupStage<NT> gst((uint32_t)a.G, wave, lane);
  gst.load(S, B, (uint32_t)a.G, rows_n, gst.g0);
  gst.store(groups, (uint32_t)a.G, gst.g0);
  for (uint32_t g = 256; g < (uint32_t)a.G; g += 256) {
    gst.load(S, B, (uint32_t)a.G, rows_n, g + gst.g0);
    gst.store(groups, (uint32_t)a.G, g + gst.g0);
  }
  load_w(0, 0);
  load_x(0, 0);
  load_w(1, 1);
  load_x(1, 1);
  load_w(2, 2);
  load_w(3, 3);

  uint8_t* const slots = smem + slot_off + (uint32_t)wave * (kSlots * kSlot);
  const uint32_t wr8 = lane >> 3, wp8 = lane & 7, wr4 = lane >> 2;
  const uint32_t put8 = wr8 * 128 + 16 * (wp8 ^ (wr8 >> 1));
  const uint32_t put8h = (wr8 + 8) * 128 + 16 * (wp8 ^ ((wr8 + 8) >> 1));
  const uint32_t put4 = wr4 * 64 + 16 * ((lane & 3) ^ (wr4 >> 2));
  const uint32_t xj = BITS == 4 ? j : 2 * (j & 1) + (j >> 1);
  uint32_t slot = 0;
  auto next_slot = [&]() __attribute__((always_inline)) {
    uint8_t* const p = slots + slot * kSlot;
    slot = (slot + 1) % kSlots;
    return p;
  };
  const u32x4 ones = {F::kOnes, F::kOnes, F::kOnes, F::kOnes};
  f32x4 tot[NT][MT], aq[NT][MT], a1[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) tot[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto unit = [&](int i, int ws, int xs) __attribute__((always_inline)) {
    const int cur = wave + i * kKsWaves;
    uint32_t wd[NT][4 * kWL];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint8_t* const sl = next_slot();
      if constexpr (BITS == 4) {
        *reinterpret_cast<u32x4*>(sl + put4) = wr[ws][t][0];
        wave_lds_fence();
        const u32x4 v = *reinterpret_cast<const u32x4*>(sl + c * 64 + 16 * (j ^ (c >> 2)));
        uint32_t d0 = v[0], d1 = v[1], d2 = v[2], d3 = v[3];
        swap16(d0, d1);
        swap16(d2, d3);
        swap32(d0, d2);
        swap32(d1, d3);
        wd[t][0] = d0;
        wd[t][1] = d1;
        wd[t][2] = d2;
        wd[t][3] = d3;
      } else {
        *reinterpret_cast<u32x4*>(sl + put8) = wr[ws][t][0];
        *reinterpret_cast<u32x4*>(sl + put8h) = wr[ws][t][kWL - 1];
        wave_lds_fence();
#pragma unroll
        for (int e = 0; e < kWL; ++e) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(sl + c * 128 + 16 * ((4 * e + j) ^ (c >> 1)));
          uint32_t d0 = v[0], d1 = v[1], d2 = v[2], d3 = v[3];
          swap32(d0, d2);
          swap32(d1, d3);
          wd[t][4 * e] = d0;
          wd[t][4 * e + 1] = d1;
          wd[t][4 * e + 2] = d2;
          wd[t][4 * e + 3] = d3;
        }
      }
    }
    // the unit's pairs ahead of x's fences, which they could not pass (8 bits, group 32, N = K =
    // 5120, 16 rows: 14.0 us when read at the end of a group, 13.2 here)
    uint32_t sb[NT][kUnit / GS];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int g = 0; g < kUnit / GS; ++g) sb[n][g] = gl[16 * n * gs4 + cur * (kUnit / GS) + g];
#pragma unroll
    for (int ln = 0; ln < 2; ++ln) {
      u32x4 xv[2][MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint8_t* const sl = next_slot();
        *reinterpret_cast<u32x4*>(sl + put8) = xr[xs][ln][t][0];
        // rows 8 .. 15 of an 8-row call hold what the slot held: rows that are not stored
        if constexpr (H == 2) *reinterpret_cast<u32x4*>(sl + put8h) = xr[xs][ln][t][H - 1];
        wave_lds_fence();
#pragma unroll
        for (int h = 0; h < 2; ++h)
          xv[h][t] = *reinterpret_cast<const u32x4*>(sl + c * 128 + 16 * ((4 * h + xj) ^ (c >> 1)));
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int st = 2 * ln + h;
        if (st * 32 % GS == 0) {
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            a1[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int n = 0; n < NT; ++n) aq[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
        u32x4 wv[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) wv[t] = F::weights(wd[t], st);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const uint32_t xd[4] = {xv[h][m][0], xv[h][m][1], xv[h][m][2], xv[h][m][3]};
          const u32x4 A = F::acts(xd);
          a1[m] = mma<F16>(A, ones, a1[m]);
#pragma unroll
          for (int n = 0; n < NT; ++n) aq[n][m] = mma<F16>(A, wv[n], aq[n][m]);
        }
        if ((st + 1) * 32 % GS == 0) {
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const uint32_t p = sb[n][st * 32 / GS];
            const float sc = act_to_f32<F16>(p & 0xffffu), bc = act_to_f32<F16>(p >> 16) - F::kOff * sc;
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                tot[n][m][q] = fmaf(sc, aq[n][m][q], fmaf(bc, a1[m][q], tot[n][m][q]));
          }
        }
      }
    }
  };
  __syncthreads();  // the scales
  for (int base = 0; base < count; base += kWU) {
#pragma unroll
    for (int i = 0; i < kWU; ++i) {
      if (base + i < count) unit(base + i, i, i % kXU);
      load_w(base + i + kWU, i);
      load_x(base + i + kXU, i % kXU);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // the partial tiles take the place of the scales

  // add the eight partial tiles: lane (c, j) of tile (n, m) holds rows 16 m + 4 j .. + 3 of
  // column 16 n + c
  f32x4* const red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((wave * MT + m) * NT + n) * 64 + lane] = tot[n][m];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * NT * 256; e += 64 * kKsWaves) {
    // element e: column fastest, then row of the tile, then tile
    const int tile = e >> 8, r = (e >> 4) & 15, col16 = e & 15;
    const int idx = tile * 256 + ((r >> 2) * 16 + col16) * 4 + (r & 3);
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kKsWaves; ++w) v += reinterpret_cast<const float*>(smem)[w * (MT * NT * 256) + idx];
    const int row = 16 * (tile / NT) + r, col = 16 * (tile % NT) + col16;
    if (row < rows_m && col < rows_n)
      reinterpret_cast<uint16_t*>(a.y)[(int64_t)row * a.ldy + n0 + col] = f32_to_act<F16>(v);
  }
}

template <int BITS, int GS, bool F16, int MT, int NT>
int32_t launch(hipStream_t st, const QmmArgs& a) {
  constexpr uint32_t kRed = kKsWaves * MT * NT * 1024;
  static std::atomic<uint64_t> lds_set{0};  // this instantiation's LDS above 64 KB, per device
  const int32_t rc = allow_lds_once((const void*)qgemm_ks_kernel<BITS, GS, F16, MT, NT>, kKsMaxLds, &lds_set,
                                    "quantized_matmul: LDS attribute");
  if (rc) return rc;
  const int ntiles = (a.N + 16 * NT - 1) / (16 * NT);
  const uint32_t slot_off = group_stride((uint32_t)a.G) * 16 * NT * 4, used = slot_off + kKsWaves * kSlots * kSlot;
  const uint32_t lds = used > kRed ? used : kRed;
  QmmArgs b = a;
  b.mtiles = (a.M + 16 * MT - 1) / (16 * MT);
  hipLaunchKernelGGL((qgemm_ks_kernel<BITS, GS, F16, MT, NT>), dim3((unsigned)(ntiles * b.mtiles)),
                     dim3(64 * kKsWaves), lds, st, b, slot_off);
  return check_hip(hipGetLastError(), "quantized_matmul launch");
}

template <int BITS, int GS, bool F16, int MX, int NT>
int32_t launch_v(hipStream_t st, const QmmArgs& a) {
  constexpr uint32_t kRed = kKsWaves * (MX > 16 ? 2 : 1) * NT * 1024;
  static std::atomic<uint64_t> lds_set{0};  // this instantiation's LDS above 64 KB, per device
  const int32_t rc = allow_lds_once((const void*)qmv_ks_kernel<BITS, GS, F16, MX, NT>, kKsMaxLds, &lds_set,
                                    "quantized_matmul: LDS attribute");
  if (rc) return rc;
  const uint32_t slot_off = group_stride((uint32_t)a.G) * 16 * NT * 4, used = slot_off + kKsWaves * kSlots * kSlot;
  const uint32_t lds = used > kRed ? used : kRed;
  hipLaunchKernelGGL((qmv_ks_kernel<BITS, GS, F16, MX, NT>), dim3((a.N + 16 * NT - 1) / (16 * NT)),
                     dim3(64 * kKsWaves), lds, st, a, slot_off);
  return check_hip(hipGetLastError(), "quantized_matmul launch");
}

template <int BITS, int GS, bool F16>
int32_t launch_tile_v(hipStream_t st, const QmmArgs& a, const KsPlan& p) {
  if (p.nt == 1)
    return a.M <= 8    ? launch_v<BITS, GS, F16, 8, 1>(st, a)
           : a.M <= 16 ? launch_v<BITS, GS, F16, 16, 1>(st, a)
                       : launch_v<BITS, GS, F16, 32, 1>(st, a);
  return a.M <= 8    ? launch_v<BITS, GS, F16, 8, 2>(st, a)
         : a.M <= 16 ? launch_v<BITS, GS, F16, 16, 2>(st, a)
                     : launch_v<BITS, GS, F16, 32, 2>(st, a);
}

template <int BITS, int GS, bool F16>
int32_t launch_tile(hipStream_t st, const QmmArgs& a, const KsPlan& p) {
#define EMA_KS(m, n) \
  if constexpr (ks_tile(BITS, m, n)) \
    if (p.mt == m && p.nt == n) return launch<BITS, GS, F16, m, n>(st, a);
  EMA_KS(3, 2) EMA_KS(4, 2) EMA_KS(5, 2) EMA_KS(3, 3) EMA_KS(4, 3) EMA_KS(5, 3) EMA_KS(3, 4) EMA_KS(4, 4)
#undef EMA_KS
  return set_error(EMA_ERR_UNSUPPORTED, "quantized_matmul: no kernel for tile %d x %d", p.mt, p.nt);
}

}  // namespace

int32_t launch_qmv_ks(hipStream_t st, const QmmArgs& a, const KsPlan& p, int gs, int bits, bool f16) {
#define EMA_KS(f) \
  if (bits == 4) \
    return gs == 32   ? launch_tile_v<4, 32, f>(st, a, p) \
           : gs == 64 ? launch_tile_v<4, 64, f>(st, a, p) \
                      : launch_tile_v<4, 128, f>(st, a, p); \
  return gs == 32   ? launch_tile_v<8, 32, f>(st, a, p) \
         : gs == 64 ? launch_tile_v<8, 64, f>(st, a, p) \
                    : launch_tile_v<8, 128, f>(st, a, p);
  if (f16) {
    EMA_KS(true)
  }
  EMA_KS(false)
#undef EMA_KS
}

int32_t launch_qgemm_ks(hipStream_t st, const QmmArgs& a, const KsPlan& p, int gs, int bits, bool f16) {
#define EMA_KS(f) \
  if (bits == 4) \
    return gs == 32   ? launch_tile<4, 32, f>(st, a, p) \
           : gs == 64 ? launch_tile<4, 64, f>(st, a, p) \
                      : launch_tile<4, 128, f>(st, a, p); \
  return gs == 32   ? launch_tile<8, 32, f>(st, a, p) \
         : gs == 64 ? launch_tile<8, 64, f>(st, a, p) \
                    : launch_tile<8, 128, f>(st, a, p);
  if (f16) {
    EMA_KS(true)
  }
  EMA_KS(false)
#undef EMA_KS
}

}  // namespace ema
