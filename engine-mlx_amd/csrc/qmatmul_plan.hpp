// Which kernel takes a quantised projection, and with which tiles: host rules on sizes, row
// stride and alignment only, free of HIP, so that the CPU test (tests/cpp/test_qmm_route.cpp)
// checks the definitions that the launches use.
#pragma once

#include "ema_schedule.hpp"

#include <stdint.h>

namespace ema {

struct QmmArgs {
  const uint8_t* x;  // [M, ldx] activations
  const uint8_t* w;  // [N, K * BITS / 8] packed fields
  const uint8_t* s;  // [N, G] scales
  const uint8_t* b;  // [N, G] biases
  uint8_t* y;        // [M, ldy]
  int64_t ldx, ldy;  // row strides in elements
  int M, N, K, G;    // G = K / GS
  int mtiles;        // row tiles of x (16 * MR rows each)
  int remap;         // grid size divisible by 8: give each XCD a contiguous range of tiles
};

constexpr int kMaxWaves = 8;

// Stride, in pairs, of the rows of {scale, bias} pairs in LDS: an odd number of 16-byte
// pieces, so that 16 rows are read without bank conflicts.
EMA_HD uint32_t group_stride(uint32_t G) { return ((G >> 2) | 1) << 2; }

// ------------------------------------------------------------------ dequantising GEMM
constexpr int kDqBN = 128, kDqKC = 64, kDqCompute = 8, kDqLoaders = 8;
// Time of the dequantising GEMM with 64 mt x 128 tiles, in units of 25 ns, one workgroup per
// CU at a time: measured 6 us per round and 0.63, 0.70 and 0.84 us per 64 k at mt = 2, 3, 4.
inline int64_t dq_cost(int M, int N, int K, int mt, int cus) {
  const int64_t tiles = ((int64_t)M + 64 * mt - 1) / (64 * mt) * (((int64_t)N + 127) / 128);
  return (tiles + cus - 1) / cus * (240 + (int64_t)(K / 64) * (mt == 2 ? 25 : mt == 3 ? 28 : 34));
}
// The mt of the least time: fewer rows per tile where that fills a last round better (M = 1531,
// N = 6144, K = 4096: two rounds of 192 rows 106 us, of 256 rows 127; M = 520, one round: 47, 51
// and 61 us with 128, 192 and 256 rows).
inline int dq_row_tiles(int M, int N, int K, int cus) {
  int best = 4;
  for (int mt = 3; mt >= 2; --mt)
    if (dq_cost(M, N, K, mt, cus) < dq_cost(M, N, K, best, cus)) best = mt;
  return best;
}

struct DqPlan {
  int mtiles, ntiles;
  int rm, rn;  // tile rows / columns per region (regions: mtiles / rm x ntiles / rn = 8), or 0
};

// Whether 256 rows of x lie within one buffer range: the row stride up to which a call of more
// than 32 rows takes dequantised weights. One line for every tile height and for the K-split GEMM,
// so that the arithmetic of a call does not depend on which of them its sizes choose.
inline bool dq_x_fits(int64_t ldx, int K) { return 256 * ldx * 2 + (int64_t)K * 2 < ((int64_t)1 << 31); }

// LDS of its two buffers (x and weight rows of a chunk): 96, 80 or 64 KB.
constexpr uint32_t dq_lds(int mt) { return 2 * (64 * mt + kDqBN) * 128; }

// Whether the dequantising GEMM stages all of K's scales and biases in LDS: from 32 groups a row
// on. Loaded per chunk, their 2-byte loads each fetch a cache line, so with the weights in HBM
// staging is 7 to 22 % faster at 64 groups and 0 to 4 % at 32; at 8 to 24 it is up to 3 % slower,
// for its barrier ahead of the first chunk, and 128-row tiles, two workgroups of which share a CU,
// gain nothing from the pairs' LDS. Four groups per 8-byte load, all pairs beside the buffers.
inline bool dq_stages_scales(const QmmArgs& a, int mt) {
  return a.G >= 32 && a.G % 4 == 0 && (((uintptr_t)a.s | (uintptr_t)a.b) & 7) == 0 &&
         dq_lds(mt) + (uint64_t)kDqBN * group_stride((uint32_t)a.G) * 4 <= 160 * 1024;
}

// Plan of the dequantising GEMM: K a multiple of the chunk and of the group, x within one
// buffer range per tile. Regions: 2 x 4, 4 x 2, 1 x 8 or 8 x 1 whole tile rows and columns,
// the one with the least bytes per region, when the grid divides into them.
inline bool plan_dq(int M, int N, int K, int gs, int bits, int64_t ldx, int mt, DqPlan* p) {
  const int kDqBM = 64 * mt;
  if (K % kDqKC || K % gs || !dq_x_fits(ldx, K)) return false;
  p->mtiles = (M + kDqBM - 1) / kDqBM;
  p->ntiles = (N + kDqBN - 1) / kDqBN;
  p->rm = p->rn = 0;
  const double xb = (double)kDqBM * K * 2, wb = (double)kDqBN * K * (bits / 8.0 + 4.0 / gs);
  double best = 0;
  for (int gm = 1; gm <= 8; gm *= 2) {  // regions along M
    const int gn = 8 / gm;
    if (p->mtiles % gm || p->ntiles % gn) continue;
    const int rm = p->mtiles / gm, rn = p->ntiles / gn;
    const double bytes = rm * xb + rn * wb;
    if (p->rm == 0 || bytes < best) {
      best = bytes;
      p->rm = rm;
      p->rn = rn;
    }
  }
  return true;
}

// ------------------------------------------------------------------ K-split kernels
constexpr int kKsWaves = 8;
constexpr int kKsMaxLds = 160 * 1024;
constexpr int kUnit = 128;                // k per unit
constexpr int kKsSlotBytes = 64 * 1024;   // the waves' exchange slots

// Column and row tiles of 16 of the K-split GEMM (qgemm_ks.hip); mt = 0: it does not apply.
struct KsPlan {
  int mt, nt;
};
// Tiles whose kernel fits the registers: 8-bit weights take twice the registers in flight,
// and at 5 x 3 and 4 x 4 they spill.
constexpr bool ks_tile(int bits, int mt, int nt) {
  return mt >= 3 && mt <= 5 && nt >= 2 && nt <= 4 && mt + nt <= (bits == 4 ? 8 : 7);
}

// Whole units, four groups' scales or biases per 8-byte load, the pairs of 64 rows and the
// slots within the LDS, 32-bit offsets inside a tile of 80 rows (the GEMM: dq_x_fits also).
inline bool ks_fits(const QmmArgs& a) {
  return a.K % kUnit == 0 && a.G % 4 == 0 && (((uintptr_t)a.s | (uintptr_t)a.b) & 7) == 0 &&
         (a.G + 4) * 64 * 4 + kKsSlotBytes <= kKsMaxLds &&
         80 * a.ldx * 2 + (int64_t)a.K * 2 < ((int64_t)1 << 31);
}

// The tile, or mt = 0 when qgemm_dq_kernel is the better kernel or this one does not apply.
// One workgroup per CU at a time, so a call takes rounds * time of a workgroup; measured at K
// = 2048 and 4096, in units of 25 ns: a workgroup takes 140 and, per turn of its eight waves
// over a unit each, 4 + 16 per row tile + 18 per column tile (qgemm_dq_kernel: dq_cost; K =
// 4096, N = 4096: 33 us here against 45 at 300 rows, 45 against 45 at 520, 58 against 46 at
// 700). The column tiles of an XCD all read all of x, and past its 4 MB L2 they read it from
// further off; the line at 5 MB was measured at K = 2048, N = 1024: 21.5 us here against 24 at 1200
// rows (4.7 MB), 25.1 against 24.5 at 1531 (6 MB) and 39.9 against 23.8 at 2048 (8 MB). It does not
// hold everywhere: with K >= 3072, N <= 2048 and x of 5 to 8 MB this kernel would still be the
// faster one (K = 4096, N = 1024, 700 rows 17.3 us against 42.1), with N >= 4096 it is not (600 rows
// 54 against 44).
inline KsPlan plan_ks(const QmmArgs& a, int bits, int cus) {
  KsPlan best{0, 0};
  if (!ks_fits(a) || !dq_x_fits(a.ldx, a.K) || (int64_t)a.M * a.K * 2 > (5 << 20)) return best;
  auto rounds = [&](int rows, int cols) {
    return (((int64_t)a.M + rows - 1) / rows * (((int64_t)a.N + cols - 1) / cols) + cus - 1) / cus;
  };
  int64_t cost = dq_cost(a.M, a.N, a.K, dq_row_tiles(a.M, a.N, a.K, cus), cus);
  const int64_t turns = (a.K / kUnit + kKsWaves - 1) / kKsWaves;
  for (int mt = 3; mt <= 5; ++mt)
    for (int nt = 2; nt <= 4; ++nt) {
      if (!ks_tile(bits, mt, nt)) continue;
      const int64_t c = rounds(16 * mt, 16 * nt) * (140 + turns * (4 + 16 * mt + 18 * nt));
      if (c < cost) {
        cost = c;
        best = KsPlan{mt, nt};
      }
    }
  return best;
}

// One column tile per workgroup while those fit the CUs in one round, else two while these
// do (measured at M = 32, K = 4096: N = 6144 10.8 us with two against 12.1, N = 4096 8.6 with
// one against 10.4; N = 9216, two rounds either way, 17.3 with one against 19.5). Below K =
// 2048 (fewer than two units per wave) the staged kernel of qmatmul.hip is the faster one:
// K = 1024, N = 2048 3.6 against 3.9 us at 8 rows, 5.0 against 6.1 at 32; K = 2048 4.6
// against 4.1 and 7.6 against 6.5. With 8 bits the line for up to 16 rows is K = 4096: at M = 2,
// nine layers of K = 2048 to N = 4096 and 2048 take 87 us there and 97 here; K = N = 4096 7.9
// us against 7.6 at 2 rows and 8.5 against 7.6 at 8.
inline KsPlan plan_qmv_ks(const QmmArgs& a, int bits, int cus) {
  const int min_k = (bits == 8 && a.M <= 16 ? 4 : 2) * kKsWaves * kUnit;
  if (a.K < min_k || !ks_fits(a)) return KsPlan{0, 0};
  const int t1 = (a.N + 15) / 16, t2 = (a.N + 31) / 32;
  return KsPlan{a.M > 16 ? 2 : 1, t1 <= cus || t2 > cus ? 1 : 2};
}

// ------------------------------------------------------------------ staged kernels
constexpr uint32_t kQmvMaxLds = 160 * 1024;  // all of a gfx950 CU's LDS

struct QmvPlan {
  int NT, KCH, NC, NB;
  uint32_t U;         // weight units per row (all of K)
  uint32_t Uc;        // weight units per row per chunk
  uint32_t rb_bytes;  // one row block plus padding
  uint32_t x_off;     // first x slot
  uint32_t x_slot;    // bytes per x slot
  uint32_t nW, nX;    // DMA instructions per chunk (weights, x)
  uint32_t nS;        // DMA instructions for all scales (and again for the biases)
  uint32_t s_off, b_off, z_off, bytes;
};

// Plan of the staged kernel for M <= 32 rows, or NC = 0 when it does not apply: a chunk
// is whole DMA blocks per weight row block (KCH * bits / 128 a multiple of 8) and whole
// groups, K is a multiple of it, and K / gs is a multiple of 8 (each 16-byte scale load
// ends inside its row).
inline QmvPlan plan_qmv(int N, int K, int gs, int bits, int mx, int cus) {
  QmvPlan none{};
  none.NC = 0;
  if ((K / gs) % 8 != 0) return none;
  const int G = K / gs;
  // two column tiles per workgroup only when 16-column tiles would outnumber the CUs (a
  // second round of workgroups costs more than doubling each one's columns)
  const int nt0 = mx >= 8 && (N + 15) / 16 > cus ? 2 : 1;
  for (int nt = nt0; nt >= 1; --nt) {
    const int rows = 16 * nt;
    for (int kch = 1024; kch >= 128; kch /= 2) {
      if (K % kch || kch % gs || (kch * bits / 128) % 8) continue;
      if (nt == 2 && kch < 256) continue;  // measured: more chunks cost more than a second round
      QmvPlan q{};
      q.NT = nt;
      q.KCH = kch;
      q.NC = K / kch;
      q.U = (uint32_t)K * bits / 128;
      q.Uc = (uint32_t)kch * bits / 128;
      q.rb_bytes = q.U * 128 + 128;
      q.nW = (uint32_t)rows * q.Uc / 64;
      q.nX = ((uint32_t)mx * kch / 8 + 63) / 64;
      q.x_slot = 1024 * q.nX;
      q.nS = ((uint32_t)rows * (G / 8) + 63) / 64;
      q.x_off = ((2 * nt) * q.rb_bytes + 1023) & ~1023u;
      const uint32_t fixed = q.x_off + 2 * 1024 * q.nS;
      // all of x if it fits (then everything is in flight from the start), else the
      // deepest ring that fits beside the weights
      int nb = q.NC;
      while (nb > 2 && fixed + 16 + nb * q.x_slot > kQmvMaxLds) --nb;
      q.NB = nb;
      q.s_off = q.x_off + nb * q.x_slot;
      q.b_off = q.s_off + 1024 * q.nS;
      q.z_off = q.b_off + 1024 * q.nS;  // 16 zero bytes read by rows of x past M
      q.bytes = q.z_off + 16;
      const uint32_t red = (uint32_t)kMaxWaves * (mx > 16 ? 2 : 1) * 1024;
      if (q.bytes < red) q.bytes = red;
      // the largest chunk that fits: fewer chunks, fewer barriers (measured faster at
      // 32 rows than deeper rings of smaller chunks)
      if (q.bytes <= kQmvMaxLds) return q;
    }
  }
  return none;
}

// Plan of qmvx_kernel: all weights and scales of 16 NT rows in LDS (x not staged).
inline QmvPlan plan_qmvx(int N, int K, int gs, int bits, int cus) {
  QmvPlan none{};
  none.NC = 0;
  if ((K / gs) % 8 != 0 || (K * bits / 128) % 8 != 0) return none;
  const int G = K / gs;
  const int nt0 = (N + 15) / 16 > cus ? 2 : 1;
  for (int nt = nt0; nt >= 1; --nt) {
    const int rows = 16 * nt;
    QmvPlan q{};
    q.NT = nt;
    q.KCH = K;
    q.NC = 1;
    q.NB = 1;
    q.U = (uint32_t)K * bits / 128;
    q.Uc = q.U;
    q.rb_bytes = q.U * 128 + 128;
    q.nW = (uint32_t)rows * q.U / 64;
    q.nX = 0;
    q.x_slot = 0;
    q.nS = ((uint32_t)rows * (G / 8) + 63) / 64;
    q.x_off = ((2 * nt) * q.rb_bytes + 1023) & ~1023u;
    q.s_off = q.x_off;
    q.b_off = q.s_off + 1024 * q.nS;
    q.z_off = q.b_off + 1024 * q.nS;
    q.bytes = q.z_off + 16;
    const uint32_t red = (uint32_t)kMaxWaves * 2 * 1024;
    if (q.bytes < red) q.bytes = red;
    if (q.bytes <= kQmvMaxLds) return q;
  }
  return none;
}

inline int qmv_rows(int M) { return M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : M <= 16 ? 16 : 32; }

// ------------------------------------------------------------------ the route
// Whether the one-row kernel takes this call: K / gs a power of two up to 64, or a
// multiple of 64, and x (2 K bytes) within 64 KB of LDS.
inline bool gemv1_fits(int G, int K) { return (G % 64 == 0 || (G <= 64 && (G & (G - 1)) == 0)) && K <= 32768; }

// Up to 32 rows, K of 2048 to 3072 and more columns than one round of workgroups holds: whether
// the kernels that keep a column tile's weights in LDS (`staged`: one to three chunks at such K)
// are faster than the K-split kernel, each of whose waves has two or three units per workgroup to
// set against its fixed 3.5 us. r1, r2: rounds of workgroups with one and two column tiles each
// (K-split: one; the staged kernels: one up to 4 rows, two above, so that they gain most where
// the two-tile rounds are full). Where they don't apply, 8 bits leave the streaming kernel.
// Measured with the weights in HBM, us, K-split / the other, group 64, K = 2048, 4 bits: N = 151936
// 81.4 / 55.2 at 2 rows, N = 32768 38.3 / 32.0 at 24, N = 9216 15.3 / 16.3 at 24; 8 bits, N =
// 32768, 32 rows 56.8 / 39.1. K = 2560, 32 rows: 8 bits, N = 32768 62.0 / 49.3; 4 bits, N = 9216
// 17.6 / 22.7. From K = 4096 on the K-split kernel is faster at every N.
inline bool staged_fills_rounds(int M, int N, int K, int gs, int bits, int cus, bool staged) {
  const int t1 = (N + 15) / 16, t2 = (N + 31) / 32;
  if (t2 <= cus) return false;
  const int r1 = (t1 + cus - 1) / cus, r2 = (t2 + cus - 1) / cus;
  const bool even = r1 >= 2 * r2 || r1 > 12;
  if (!staged) return bits == 8 && M > 16 && (K == 2560 || (K <= 2304 && M <= 24 && r1 > 3));
  if (M <= 2) return K <= 2048 || (K == 2560 && r1 > 8) || (K == 3072 && (gs > 32 || r1 > 6));
  if (M <= 4) return K <= 2048 || (K == 3072 && gs == 128);
  if (M <= 8) return K <= 2048 && r1 > (gs == 32 ? 3 : 2);
  if (M <= 16) return K <= 2048 && gs > 32 && (even || r1 > 6);
  if (bits == 4) return K <= 2048 ? r1 > (gs == 32 && M <= 24 ? 2 : 3) : K <= 3072 && gs == 32 && even;
  return K <= 2048 || (K <= 2560 && r1 > (K == 2560 && M <= 24 ? 2 : 3)) || (K <= 3072 && even);
}

enum class QmmKernel { gemv1, qmv_ks, qgemm_ks, qmv, qmvx, qgemm_dq, qmm };
struct QmmRoute {
  QmmKernel kernel;
  int mt, nt;   // row and column tiles: of 16, of 64 x 128 (qgemm_dq); mt of qmv and qmvx: rows of x
  QmvPlan qmv;  // qmv, qmvx
  DqPlan dq;    // qgemm_dq
};
inline QmmRoute qmm_route(const QmmArgs& a, int gs, int bits, int cus) {
  QmmRoute r{QmmKernel::qmm, a.M <= 16 ? 1 : 2, 1, QmvPlan{}, DqPlan{}};
  if (a.M == 1 && gemv1_fits(a.G, a.K)) {
    r.kernel = QmmKernel::gemv1;
    return r;
  }
  if (a.M <= 32) {
    const int mx = qmv_rows(a.M);
    QmvPlan p = plan_qmv(a.N, a.K, gs, bits, mx, cus);
    QmmKernel kernel = QmmKernel::qmv;
    if (mx >= 16) {
      // x through an LDS ring shared by the column tiles (qmv_kernel) when it reaches the
      // wanted tile count, else x through registers (qmvx_kernel), whose LDS holds only
      // the weights (8 bits, N = 6144, K = 4096, 32 rows, scales that are not 8-byte aligned:
      // 21.9 us with two tiles against 23.7 with one)
      const int want = (a.N + 15) / 16 > cus ? 2 : 1;
      const QmvPlan px = p.NC > 0 && p.NT == want ? QmvPlan{} : plan_qmvx(a.N, a.K, gs, bits, cus);
      if (px.NC > 0 && (p.NC == 0 || px.NT == want)) {
        p = px;
        kernel = QmmKernel::qmvx;
      }
    }
    const KsPlan kp = plan_qmv_ks(a, bits, cus);
    if (kp.mt > 0 && !staged_fills_rounds(a.M, a.N, a.K, gs, bits, cus, p.NC > 0)) {
      r.kernel = QmmKernel::qmv_ks;
      r.mt = kp.mt;
      r.nt = kp.nt;
    } else if (p.NC > 0) {
      r.kernel = kernel;
      r.mt = mx;
      r.nt = p.NT;
      r.qmv = p;
    }
    return r;
  }
  const KsPlan kp = plan_ks(a, bits, cus);
  if (kp.mt > 0) {
    r.kernel = QmmKernel::qgemm_ks;
    r.mt = kp.mt;
    r.nt = kp.nt;
    return r;
  }
  const int mt = dq_row_tiles(a.M, a.N, a.K, cus);
  if (plan_dq(a.M, a.N, a.K, gs, bits, a.ldx, mt, &r.dq)) {
    r.kernel = QmmKernel::qgemm_dq;
    r.mt = mt;
  }
  return r;
}

}  // namespace ema
