// w8a16_gemm.hip — the W8A16 linear over many activation rows (prefill, verify
// and decode batches past 16 rows) for gfx950: an MFMA GEMM that dequantizes the
// int8 weights between LDS and the matrix cores.
//
//   y[m, n] = scale[n] * sum_k x[m, k] * w[n, k] (+ bias[n])           per channel
//   y[m, n] = sum_g scale[n, g] * sum_{k in g} x[m, k] * w[n, k] (+ bias)  per group
//
// Bound by operations (2 M N K against N K + 2 M (N + K) bytes) from about 200 rows up, by
// bytes below. Counters (bf16): 4096 x 19456 x 2560, 256 x 256 tiles, 370 us: MFMA busy 52% of
// the SIMD cycles, vector issue 37%; 56 x 19456 x 2560, 64 x 96 tiles, 22 us: MFMA 10%, vector
// 12%, 52% of the wave cycles waiting at under one wave per SIMD; 56 x 151936 x 1024, 64 x 128
// tiles, 50 us: 15%, 21%, 42%. Layout of one step (64 columns of K):
//  * x rows (128 B) and weight rows (64 B) go from HBM / L2 straight into LDS
//    (global_load_lds, 16 B per lane, no registers); the 16-byte units of a row are
//    permuted by the global address of each lane, so that the 16 lanes of an operand read
//    hit 16 different 16-byte slots of the 256-byte bank row (x_swizzle, w_swizzle);
//  * the weights stay int8 in LDS (half the LDS traffic of a 16-bit tile) and each
//    wave dequantizes the operands it reads (sd::dequant8): 96 VALU instructions beside
//    64 MFMAs per wave and step at 128 x 64 outputs per wave;
//  * the weights are the MFMA A operand. Tile row 4 g + i of tile t is weight row
//    4 NT g + 4 t + i of the wave, so a lane's sums are 4 NT consecutive outputs of one
//    row and leave in 16-byte stores.
// The loop runs half a step ahead: the second half's x operands load under the first
// half's MFMAs; then one barrier (the next step has landed in every wave's view, this
// step's LDS is read), the load of step + S into the freed stage, and the next step's
// first operands under the second half's MFMAs.
//
// Sums: one fp32 accumulator per output over the K slice, in ascending k and with the
// operand order of w8a16_kernel (lane group g holds k = 16 g .. 16 g + 15 of a step, two
// MFMAs), so a shape gives the same bits on either kernel with the same K slices (which
// start on whole stages). With several slices each writes its fp32 partials and
// w8a16_gemm_reduce adds them in slice order, then scales and rounds (partial sums stay
// 32-bit).
#include "w8a16.h"

namespace {

using sd::f32x4;
using sd::u32x4;

struct GemmParams {
  sd::W8GemmArgs a;
  float* part;      // splits > 1: [splits][M][pitch] partial sums
  int64_t pitch;
  int32_t nks;      // 64-column steps of the whole K
  int32_t tiles_m, tiles_n, splits;
  int32_t vec_out;  // y rows allow 16-byte stores
};

__device__ __forceinline__ void load_lds16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

// Wait for all but the newest N vector-memory loads of this wave and for its LDS
// reads, then for the workgroup.
template <int N> __device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Position of a 16-byte unit within its LDS row: XOR with these. An operand read takes one
// unit of 16 x rows, or of the weight rows 4 NT j + i (i, j < 4): with two 128-byte x rows
// (four 64-byte weight rows) to a 256-byte bank row when KB is 1, whole bank rows (two
// 128-byte ones) when it is 2, the 16 lanes then cover 16 different 16-byte slots.
// (SQ_LDS_BANK_CONFLICT counts none with KB = 2, but 4 cycles per read with KB = 1.)
template <int KB> __device__ __forceinline__ int x_swizzle(int r) { return KB == 1 ? (r >> 1) & 7 : r & 15; }
template <int KB, int NT> __device__ __forceinline__ int w_swizzle(int r) {
  const int j = (r / (4 * NT)) & 3;
  return KB == 1 ? j : (((r >> 1) & 1) | (j << 1));
}

// WM x WN waves, each MT x NT tiles of 16 x 16 outputs; S stages of KB 64-column steps.
template <typename T, int WM, int WN, int MT, int NT, int S, int KB, int WPE, bool PG, bool FLOOR>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(WPE)))
void w8a16_gemm_kernel(GemmParams p) {
  constexpr int NW = WM * WN, BM = WM * MT * 16, BN = WN * NT * 16;
  constexpr int XR = 128 * KB, WR = 64 * KB;       // bytes of an x row, of a weight row
  constexpr int XB = BM * XR, SB = XB + BN * WR;   // bytes of a stage: x rows, weight rows
  // 1 KB loads per wave and stage: where the x rows don't divide by the waves, the last
  // waves load the last KB again (the same bytes to the same place, each wave waits for its own)
  constexpr int KX = XB / 1024, CX = (KX + NW - 1) / NW, CW = BN * WR / 1024 / NW;
  constexpr int LPW = CX + CW;
  static_assert(KX * 1024 == XB && CW * NW * 1024 == SB - XB, "whole 1 KB loads");
  static_assert(KB == 1 || (KB == 2 && !PG), "stages of one or two steps");
  extern __shared__ __attribute__((aligned(1024))) char sm[];
  const sd::W8GemmArgs& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;

  // Workgroup -> (slice, tile): every eighth workgroup shares an XCD (one L2), so each
  // XCD takes a contiguous run of tiles, 8 M tiles deep before the next N tile.
  const int items = p.tiles_m * p.tiles_n * p.splits;
  int id = blockIdx.x;
  {
    const int per = items / 8, rem = items % 8, xcd = id % 8;
    id = xcd * per + min(xcd, rem) + id / 8;
  }
  const int tiles = p.tiles_m * p.tiles_n;
  const int slice = id / tiles;
  id -= slice * tiles;
  constexpr int kGroupM = 8;
  const int gi = id / (kGroupM * p.tiles_n), gr = id - gi * kGroupM * p.tiles_n;
  const int gm = min(kGroupM, p.tiles_m - gi * kGroupM);
  const int m0 = (gi * kGroupM + gr % gm) * BM, n0 = gr / gm * BN;
  const int stages = p.nks / KB;
  const int ks = KB * static_cast<int>(static_cast<int64_t>(slice) * stages / p.splits);
  const int ke = KB * static_cast<int>(static_cast<int64_t>(slice + 1) * stages / p.splits);

  // ---- loads: this lane's 16-byte unit of each 1 KB (of whole x or weight rows); rows
  //      past M / N read the last row (their outputs are not written), steps past the
  //      slice read its last ones (into a stage nobody reads)
  const char* xbase = reinterpret_cast<const char*>(a.x + static_cast<int64_t>(m0) * a.xs);
  const char* wbase = reinterpret_cast<const char*>(a.w + static_cast<int64_t>(n0) * a.ws);
  uint32_t xoff[CX], woff[CW];
#pragma unroll
  for (int i = 0; i < CX; ++i) {
    const int at = min(wave * CX + i, KX - 1) * 64 + lane, r = at / (XR / 16);
    const int unit = (at % (XR / 16)) ^ x_swizzle<KB>(r);
    xoff[i] = static_cast<uint32_t>(min(r, a.M - 1 - m0)) * static_cast<uint32_t>(a.xs * 2) + unit * 16;
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int at = (wave * CW + i) * 64 + lane, r = at / (WR / 16);
    const int unit = (at % (WR / 16)) ^ w_swizzle<KB, NT>(r);
    woff[i] = static_cast<uint32_t>(min(r, a.N - 1 - n0)) * static_cast<uint32_t>(a.ws) + unit * 16;
  }
  auto issue = [&](int step, int st) {
    const int s = min(step, ke - KB);
    const char* xb = xbase + static_cast<int64_t>(s) * 128;
    const char* wb = wbase + static_cast<int64_t>(s) * 64;
    char* stage = sm + st * SB;
#pragma unroll
    for (int i = 0; i < CX; ++i) load_lds16(xb + xoff[i], stage + min(wave * CX + i, KX - 1) * 1024);
#pragma unroll
    for (int i = 0; i < CW; ++i) load_lds16(wb + woff[i], stage + XB + (wave * CW + i) * 1024);
  };

  if constexpr (FLOOR) {  // the loads and barriers alone
#pragma unroll
    for (int s = 0; s < S; ++s) issue(ks + s * KB, s);
    wait_barrier<(S - 1) * LPW>();
    int st = 0;
    for (int step = ks; step < ke; step += KB) {
      wait_barrier<(S - 2) * LPW>();
      issue(step + S * KB, st);
      st = st + 1 == S ? 0 : st + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  const int nb = n0 + wn * NT * 16 + lg * 4 * NT;  // first of this lane's 4 NT outputs per row

  // ---- per-channel scales of this lane's outputs, ahead of the loop (one after another:
  //      load_scale branches on their type; the bias follows the loop); per group: the
  //      slice's table in LDS after the stages, [group][BN] in fp32
  float sc[PG ? 1 : NT][4];
  float* tab = reinterpret_cast<float*>(sm + S * SB);
  const int spg = PG ? a.group / 64 : 1;           // steps per group
  const int ng = PG ? a.K / a.group : 1, g0 = ks / spg;
  if constexpr (PG) {
    const int groups = (ke - 1) / spg - g0 + 1;
    for (int i = tid; i < BN * groups; i += NW * 64) {
      const int n = i / groups, g = i - n * groups;
      tab[g * BN + n] = sd::load_scale(a.scale, a.scale_dtype,
                                       static_cast<int64_t>(min(n0 + n, a.N - 1)) * ng + g0 + g);
    }
  } else if (p.splits == 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[t][i] = sd::load_scale(a.scale, a.scale_dtype, min(nb + 4 * t + i, a.N - 1));
  }

  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- LDS operand addresses. x: row lr of tile m; half h (32 columns) of a stage takes the
  //      16-byte unit 8 (h / 2) + 2 lg + h % 2. Weights: row 4 NT (lr / 4) + 4 t + lr % 4 of
  //      the wave, unit 4 (h / 2) + lg (16 int8: two halves).
  const int xrow = wm * MT * 16 + lr, wrow = wn * NT * 16 + (lr >> 2) * 4 * NT + (lr & 3);
  const int xa = xrow * XR + ((lg * 2) ^ x_swizzle<KB>(xrow)) * 16;
  const int wa = XB + wrow * WR + (lg ^ w_swizzle<KB, NT>(wrow)) * 16;
  u32x4 xf[2][MT], wr[NT];
  auto read_x = [&](int st, int h) {
    const char* b = sm + st * SB + (xa ^ ((h & 1) * 16 + (h >> 1) * 128));
#pragma unroll
    for (int m = 0; m < MT; ++m) xf[h & 1][m] = sd::load16(b + m * 16 * XR);
  };
  auto read_w = [&](int st, int step) {
    const char* b = sm + st * SB + (wa ^ (step * 64));
#pragma unroll
    for (int t = 0; t < NT; ++t) wr[t] = sd::load16(b + t * 4 * WR);
  };

  int st = 0;
  if constexpr (PG) {
    // one partial sum per step, scaled into the accumulators; the loads run S - 1 steps ahead
#pragma unroll
    for (int s = 0; s < S - 1; ++s) issue(ks + s, s);
    for (int step = ks; step < ke; ++step) {
      wait_barrier<(S - 2) * LPW>();
      issue(step + S - 1, st == 0 ? S - 1 : st - 1);
      read_w(st, 0);
      read_x(st, 0);
      read_x(st, 1);
      const float* tg = tab + (step / spg - g0) * BN + (nb - n0);
      f32x4 gs[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) gs[t] = *reinterpret_cast<const f32x4*>(tg + 4 * t);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const u32x4 w0 = sd::dequant8<T>(wr[t].x, wr[t].y), w1 = sd::dequant8<T>(wr[t].z, wr[t].w);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4 z = {0.f, 0.f, 0.f, 0.f};
          z = sd::Elem<T>::mfma(w0, xf[0][m], z);
          z = sd::Elem<T>::mfma(w1, xf[1][m], z);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][m][i] += z[i] * gs[t][i];
        }
      }
      st = st + 1 == S ? 0 : st + 1;
    }
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) issue(ks + s * KB, s);
    wait_barrier<(S - 1) * LPW>();
    read_w(0, 0);
    read_x(0, 0);
    for (int step = ks; step < ke; step += KB) {
#pragma unroll
      for (int h = 0; h < 2 * KB; ++h) {
        u32x4 wd[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          wd[t] = h & 1 ? sd::dequant8<T>(wr[t].z, wr[t].w) : sd::dequant8<T>(wr[t].x, wr[t].y);
        if (h < 2 * KB - 1) {
          read_x(st, h + 1);
          if (h & 1) read_w(st, (h + 1) / 2);
        } else {
          wait_barrier<(S - 2) * LPW>();
          issue(step + S * KB, st);
          st = st + 1 == S ? 0 : st + 1;
          read_w(st, 0);
          read_x(st, 0);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[t][m] = sd::Elem<T>::mfma(wd[t], xf[h & 1][m], acc[t][m]);
      }
    }
  }
  // no load of this workgroup may reach LDS after it has ended
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- outputs: lane holds y[m0 + 16 (wm MT + m) + lr][nb + 4 t + i]
  if (p.splits > 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int r = m0 + (wm * MT + m) * 16 + lr;
      if (r >= a.M) continue;
      float* dst = p.part + (static_cast<int64_t>(slice) * a.M + r) * p.pitch + nb;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (nb + 4 * t < a.N) *reinterpret_cast<f32x4*>(dst + 4 * t) = acc[t][m];
    }
    return;
  }
  float bi[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) bi[t][i] = a.bias ? sd::from_bits<T>(a.bias[min(nb + 4 * t + i, a.N - 1)]) : 0.f;
  const bool whole = p.vec_out && nb + 4 * NT <= a.N;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int r = m0 + (wm * MT + m) * 16 + lr;
    if (r >= a.M) continue;
    uint16_t* dst = a.y + static_cast<int64_t>(r) * a.ys + nb;
    float v[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[t][i] = acc[t][m][i] * (PG ? 1.f : sc[PG ? 0 : t][i]) + bi[t][i];
    if (whole) {
      uint32_t o[2 * NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        o[2 * t] = sd::pack2<T>(v[t][0], v[t][1]);
        o[2 * t + 1] = sd::pack2<T>(v[t][2], v[t][3]);
      }
      if constexpr (NT == 1) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(o[0], o[1]);
      } else {
#pragma unroll
        for (int t = 0; t < NT; t += 2)
          sd::store16(dst + 4 * t, u32x4{o[2 * t], o[2 * t + 1], o[2 * t + 2], o[2 * t + 3]});
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nb + 4 * t + i < a.N) dst[4 * t + i] = sd::to_bits<T>(v[t][i]);
    }
  }
}

// Partial sums of the K slices, added in slice order, scaled, rounded: one thread per
// four outputs of a row, every slice's load in flight at once.
template <typename T, int SPLITS>
__global__ __launch_bounds__(256) void w8a16_gemm_reduce(GemmParams p) {
  const sd::W8GemmArgs& a = p.a;
  const int nq = (a.N + 3) / 4;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(a.M) * nq) return;
  const int m = static_cast<int>(i / nq), n = static_cast<int>(i - static_cast<int64_t>(m) * nq) * 4;
  const float* src = p.part + static_cast<int64_t>(m) * p.pitch + n;
  const int64_t slice = static_cast<int64_t>(a.M) * p.pitch;
  f32x4 v[SPLITS];
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) v[s] = *reinterpret_cast<const f32x4*>(src + s * slice);
  float sc[4], bi[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = min(n + e, a.N - 1);
    sc[e] = a.group ? 1.f : sd::load_scale(a.scale, a.scale_dtype, c);
    bi[e] = a.bias ? sd::from_bits<T>(a.bias[c]) : 0.f;
  }
  f32x4 acc = v[0];
#pragma unroll
  for (int s = 1; s < SPLITS; ++s) acc += v[s];
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = acc[e] * sc[e] + bi[e];
  uint16_t* dst = a.y + static_cast<int64_t>(m) * a.ys + n;
  if (p.vec_out && n + 4 <= a.N) {
    *reinterpret_cast<uint2*>(dst) = make_uint2(sd::pack2<T>(o[0], o[1]), sd::pack2<T>(o[2], o[3]));
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < a.N) dst[e] = sd::to_bits<T>(o[e]);
  }
}

// ------------------------------------------------------------------- launches
enum Tile { kT32x64, kT64x64, kT64x80, kT64x96, kT64x128, kT64x256, kT128x128, kT128x256, kT256x256 };

struct Shape {
  int bm, bn, kb;
};
constexpr Shape kShapes[] = {{32, 64, 2},   {64, 64, 2},   {64, 80, 2},   {64, 96, 2},  {64, 128, 1},
                             {64, 256, 1},  {128, 128, 1}, {128, 256, 1}, {256, 256, 1}};

int64_t tiles_of(Tile t, int64_t M, int64_t N) {
  return ((M + kShapes[t].bm - 1) / kShapes[t].bm) * ((N + kShapes[t].bn - 1) / kShapes[t].bn);
}

int64_t pitch_of(int64_t N) { return (N + 3) / 4 * 4; }

// LDS of the per-group scale table of a K slice.
size_t table_bytes(Tile t, int64_t K, int32_t group, int splits) {
  if (!group) return 0;
  const int64_t nks = K / 64, spg = group / 64, per = (nks + splits - 1) / splits;
  return static_cast<size_t>(kShapes[t].bn) * static_cast<size_t>((per + spg - 2) / spg + 1) * sizeof(float);
}

// The per-group tile: its stages, their bytes with the table.
constexpr Tile kGroupTile = kT64x128;
constexpr int kGroupStages = 3;
size_t group_lds(int64_t K, int32_t group, int splits) {
  return static_cast<size_t>(kGroupStages) * (kShapes[kGroupTile].bm * 128 + kShapes[kGroupTile].bn * 64) +
         table_bytes(kGroupTile, K, group, splits);
}

// What a tile costs, in microseconds per 64-column step, measured at 256 CUs (M 17 - 6896;
// N x K 1024 x 2048 to 19456 x 2560 and 151936 x 1024): `alone` with at most one workgroup
// per CU, `full` per workgroup of a CU that always has more. The large tiles win where they
// fill the chip (4096 x 19456 x 2560: 64 x 128 520, 128 x 128 409, 128 x 256 388, 256 x 256
// 361 us), the small ones at few rows: 19456 x 2560 at M = 24 64 x 128 20.5, 32 x 64 15.0 us;
// at M = 56 23.0 and 18.6; at M = 100 64 x 128 28.1, 64 x 256 25.5). The 80- and 96-row tiles
// are for widths whose 64-row tiles just miss a whole number of workgroups per CU: 19456 x 2560
// is 304 tiles of 64 rows, 203 of 96 (weights from HBM: M = 56 21.7 -> 18.6 us, M = 100 64 x 256
// 29.9, 64 x 80 25.0); five stages instead of three measured 2 - 5% slower there. Per group the step sums
// and scales come on top (a 128 x 128 tile took 0.82 us, more than two of 64 x 128).
struct Cost {
  Tile tile;
  double alone, full;
};
constexpr Cost kCosts[] = {{kT32x64, 0.188, 0.126},  {kT64x64, 0.256, 0.197},  {kT64x80, 0.307, 0.23},
                           {kT64x96, 0.303, 0.30},  {kT64x128, 0.44, 0.36},   {kT64x256, 0.50, 0.68},
                           {kT128x128, 0.63, 0.535}, {kT128x256, 1.0, 1.01},   {kT256x256, 1.43, 1.78}};
constexpr Cost kCostsGroup[] = {{kGroupTile, 0.50, 0.38}};

// 3, 6 and 12 beside the powers of two: 40 tiles of 2560 rows are 240 workgroups in 6 slices
// (2560 x 9728, M = 56: 4 slices 18.3 us, 6 slices 15.8; M = 2048 142 -> 114 us with 3).
constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};

// The tile and the K slices of least estimated time: rounds of workgroups per CU (between
// the mean and the largest share: workgroups of a CU run together), about three steps to
// fill and drain a tile, and for several slices the second launch and the partial sums
// through memory (4.3 TB/s). Checked against the measured best of all tiles and slices at
// the sizes above: 3% more time in the mean.
sd::W8GemmPlan plan_for(int64_t M, int64_t N, int64_t K, int32_t group, bool sliced = true) {
  const int64_t nks = K / 64;
  const double cus = sd::device_cus();
  sd::W8GemmPlan best{kT64x128, 1, 1};
  double best_us = 1e30;
  const Cost* costs = group ? kCostsGroup : kCosts;
  const int ncosts = group ? 1 : 9;
  for (int c = 0; c < ncosts; ++c)
    for (int splits : kSplits) {
      const int64_t kb = kShapes[costs[c].tile].kb;
      if (splits > 1 && (!sliced || nks < 4 * splits)) break;
      if (nks % kb) break;  // whole stages
      double full = costs[c].full;
      // (a scale table that leaves room for one workgroup per CU)
      if (group && group_lds(K, group, splits) > 80 * 1024) full = costs[c].alone;
      const double n = static_cast<double>(tiles_of(costs[c].tile, M, N)) * splits / cus;
      const double whole = static_cast<double>(static_cast<int64_t>(n)) + (n > static_cast<int64_t>(n) ? 1 : 0);
      const double shared = n > 1 ? 0.5 * (n + whole) * full : n * full;
      const double step = shared > costs[c].alone ? shared : costs[c].alone;
      double us = (static_cast<double>((nks / kb + splits - 1) / splits * kb) + 3) * step;
      if (splits > 1) us += 3.5 + 8.0 * splits * static_cast<double>(M) * static_cast<double>(N) / 4.3e6;
      if (us < best_us) {
        best_us = us;
        best = sd::W8GemmPlan{costs[c].tile, splits, static_cast<int>(kb)};
      }
    }
  return best;
}

template <typename T, int WM, int WN, int MT, int NT, int S, int KB, int WPE, bool PG, bool FLOOR>
int launch(GemmParams p, Tile t, hipStream_t st) {
  constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
  p.tiles_m = (p.a.M + BM - 1) / BM;
  p.tiles_n = (p.a.N + BN - 1) / BN;
  const size_t lds = static_cast<size_t>(S) * (BM * 128 + BN * 64) * KB +
                     table_bytes(t, p.a.K, FLOOR ? 0 : p.a.group, p.splits);
  hipLaunchKernelGGL((w8a16_gemm_kernel<T, WM, WN, MT, NT, S, KB, WPE, PG, FLOOR>),
                     dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits)),
                     dim3(WM * WN * 64), lds, st, p);
  return SD_OK;
}

// Waves per tile: the waves of the small tiles wait about half of their cycles, so these take
// 16 weight rows per wave and several workgroups per CU, and read 128-byte pieces of a row.
// (The fp16 128 x 256 instance spills two registers under its four waves per SIMD.) Two stages where the tiles are many:
// more workgroups per CU measured better than more stages (128 x 128 at 4096 x 19456 x 2560
// 398 against 424 us), three or four where loads wait for HBM (64 x 128 at M = 56 of
// 19456 x 2560 23 us with two, 20 with four, 24 with eight and one workgroup per CU).
template <typename T, bool PG, bool FLOOR>
int launch_tile(Tile t, const GemmParams& p, hipStream_t st) {
  if constexpr (PG) {
    return launch<T, 1, 4, 4, 2, kGroupStages, 1, 2, true, FLOOR>(p, t, st);
  } else {
    switch (t) {
      case kT32x64: return launch<T, 1, 4, 2, 1, 3, 2, 4, false, FLOOR>(p, t, st);
      case kT64x80: return launch<T, 1, 5, 4, 1, 3, 2, 4, false, FLOOR>(p, t, st);
      case kT64x96: return launch<T, 1, 6, 4, 1, 3, 2, 4, false, FLOOR>(p, t, st);
      case kT64x64: return launch<T, 1, 4, 4, 1, 3, 2, 4, false, FLOOR>(p, t, st);
      case kT64x128: return launch<T, 1, 4, 4, 2, 4, 1, 2, false, FLOOR>(p, t, st);
      case kT64x256: return launch<T, 1, 8, 4, 2, 3, 1, 4, false, FLOOR>(p, t, st);
      case kT128x128: return launch<T, 2, 2, 4, 4, 2, 1, 3, false, FLOOR>(p, t, st);
      case kT128x256: return launch<T, 2, 4, 4, 4, 2, 1, 4, false, FLOOR>(p, t, st);
      default: return launch<T, 2, 4, 8, 4, 2, 1, 2, false, FLOOR>(p, t, st);
    }
  }
}

template <typename T>
void launch_reduce(const GemmParams& p, hipStream_t st) {
  const int64_t n = static_cast<int64_t>(p.a.M) * ((p.a.N + 3) / 4);
  const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
  switch (p.splits) {
    case 2: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 2>), grid, block, 0, st, p); break;
    case 3: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 3>), grid, block, 0, st, p); break;
    case 4: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 4>), grid, block, 0, st, p); break;
    case 6: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 6>), grid, block, 0, st, p); break;
    case 8: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 8>), grid, block, 0, st, p); break;
    case 12: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 12>), grid, block, 0, st, p); break;
    default: hipLaunchKernelGGL((w8a16_gemm_reduce<T, 16>), grid, block, 0, st, p); break;
  }
}

template <typename T>
int run(Tile t, const GemmParams& p, hipStream_t st, bool floor) {
  if (floor) return launch_tile<T, false, true>(t, p, st);
  const int rc = p.a.group ? launch_tile<T, true, false>(t, p, st) : launch_tile<T, false, false>(t, p, st);
  if (rc != SD_OK || p.splits == 1) return rc;
  launch_reduce<T>(p, st);
  return SD_OK;
}

GemmParams params(const sd::W8GemmArgs& a, int splits, void* workspace) {
  GemmParams p{};
  p.a = a;
  p.part = static_cast<float*>(workspace);
  p.pitch = pitch_of(a.N);
  p.nks = a.K / 64;
  p.splits = splits;
  p.vec_out = sd::aligned16(a.y) && a.ys % 8 == 0;
  return p;
}

}  // namespace

namespace sd {

// From 17 rows up, except where the 16-row kernels are faster. Both were timed from graphs
// at 6481 shapes (M 17 - 1024, N 64 - 262144, K 64 - 9728, per channel and in groups of 128),
// weights rotating through HBM; "there" is the 16-row kernel:
//  * layers of at most 8 Mi weights while M <= 128 and M N K <= 5.4e8 (one launch, K split
//    inside a workgroup): 1024 x 2048 at M = 56 6.1 us there against 9.2 here, at M = 128
//    10.0 against 10.5; 6144 x 1024 at M = 56 9.2 against 11.0, at M = 128 13.6 against 12.0;
//  * few 16 x 16 output tiles, whatever M: the tiles here are too few for the device, and a
//    second launch for K slices costs more than it saves. Up to three tiles per CU at K <= 1024
//    (256 x 1024 at M = 512 5.1 us there, 6.6 here; 1024 x 1024 at M = 192 6.2 and 7.1, at
//    M = 256, four per CU, 6.9 and 7.0), one per CU up to K = 3072 (256 x 2048 at M = 256 5.7
//    and 7.2; past 512 rows a 16-row grid of that few columns is too narrow: 64 x 2048 at
//    M = 768 18.4 and 6.9). Per group six and four below K = 512, one up to K = 2048
//    (1024 x 1024 at M = 256 8.4 and 10.0; 6144 x 1024 at M = 64 10.1 and 13.2). From K = 256:
//    a few steps do not split there (256 x 128 at M = 256 6.1 and 4.0);
//  * many rows of few columns (vocabulary heads), read there as whole rows against the staged
//    activations, here in tiles of few steps: up to 32 rows from 64 Ki weight rows at
//    K <= 1024 (151936 x 1024 at M = 17 37.5 and 39.5, 65536 x 1024 17.7 and 20.7, but
//    40000 x 1024 16.4 and 14.9), up to 64 from 96 Ki rows while M K <= 36 Ki and within
//    100 Mi weights (100000 x 256 at M = 48 14.9 and 20.1, x 768 28.7 and 32.6; 262144 x 512
//    at M = 48, past that, 41.8 and 40.2). Per group up to 32 rows at K <= 512 from 32 Mi weights
//    (65536 x 512 at M = 24 12.1 and 14.4).
// What is left: 129 - 224 rows of K <= 256 at 12288 columns and more are 5 - 13% slower here,
// where 64-row blocks fit the row count better than these tiles.
bool stays_on_16_rows(int64_t M, int64_t N, int64_t K, int32_t group) {
  constexpr int64_t kKi = 1024, kMi = 1024 * 1024;
  if (M <= 16) return true;
  if (M <= 128 && N * K <= 8 * kMi && static_cast<double>(M) * N * K <= 5.4e8) return true;
  const int64_t cus = device_cus(), tiles = (M + 15) / 16 * ((N + 15) / 16);
  if (K >= 256 && K <= 1024) {
    if (tiles <= (group == 0 ? 3 : K < 512 ? 4 : 6) * cus) return true;
  } else if (K > 1024 && K <= (group ? 2048 : 3072)) {
    if (M <= 512 && tiles <= cus) return true;
  }
  if (group) return M <= 32 && K <= 512 && N * K >= 32 * kMi;
  return (M <= 32 && K <= 1024 && N >= 64 * kKi) ||
         (M <= 64 && M * K <= 36 * kKi && N >= 96 * kKi && N * K <= 100 * kMi);
}

W8GemmPlan w8a16_gemm_plan(int64_t M, int64_t N, int64_t K, int32_t group) {
  constexpr W8GemmPlan kNone{0, 0, 1};
  if (stays_on_16_rows(M, N, K, group)) return kNone;
  const W8GemmPlan pl = plan_for(M, N, K, group);
  // a launch takes fewer than 2^32 work-items; a workgroup has up to 512
  return tiles_of(static_cast<Tile>(pl.tile), M, N) * pl.slices < (int64_t{1} << 23) ? pl : kNone;
}

// Up to two 16 x 16 output tiles per CU (three per group, where this kernel's step is dearer)
// the 16-row kernels are faster than one slice here: 2560 x 9728 at M = 48 27.6 us there, 33.5
// here, at M = 64, 2.5 per CU, 39.8 and 33.8; 4096 x 2560 at M = 32 10.8 and 11.4, 6144 x 2560
// at M = 17, three per CU, 13.6 and 11.7; in groups of 128 2560 x 4096 at M = 64 31.0 and 41.2,
// 4096 x 2560 at M = 64, four per CU, 31.6 and 27.1.
W8GemmPlan w8a16_gemm_plan_unsliced(int64_t M, int64_t N, int64_t K, int32_t group) {
  const int64_t tiles = (M + 15) / 16 * ((N + 15) / 16);
  if (stays_on_16_rows(M, N, K, group) || tiles <= (group ? 3 : 2) * device_cus()) return W8GemmPlan{0, 0, 1};
  return plan_for(M, N, K, group, false);
}

int64_t w8a16_gemm_plan_code(const W8GemmPlan& pl) {
  if (pl.slices == 0) return 0;
  return pl.slices | static_cast<int64_t>(kShapes[pl.tile].bn) << 8 |
         static_cast<int64_t>(kShapes[pl.tile].bm) << 20;
}

size_t w8a16_gemm_workspace(const W8GemmPlan& pl, int64_t M, int64_t N) {
  if (pl.slices <= 1) return 0;
  return static_cast<size_t>(pl.slices) * static_cast<size_t>(M) * static_cast<size_t>(pitch_of(N)) * sizeof(float);
}

bool w8a16_gemm_fits(const W8GemmArgs& a, const W8GemmPlan& pl) {
  // a tile's x rows within 32-bit byte offsets; its LDS
  if (a.xs >= (int64_t{1} << 23)) return false;
  return !a.group || group_lds(a.K, a.group, pl.slices) <= static_cast<size_t>(device_lds_per_block());
}

int w8a16_gemm(const W8GemmArgs& a, const W8GemmPlan& pl, void* workspace, hipStream_t st, bool floor) {
  const Tile t = static_cast<Tile>(pl.tile);
  const GemmParams p = params(a, pl.slices, workspace);
  const int rc = a.dtype == SD_BF16 ? run<__bf16>(t, p, st, floor) : run<_Float16>(t, p, st, floor);
  return rc != SD_OK ? rc : check_launch(floor ? "w8a16 floor" : "w8a16");
}

}  // namespace sd
