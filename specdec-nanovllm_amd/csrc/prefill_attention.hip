// prefill_attention.hip — variable-length causal attention for gfx950: the
// prefill branch of the engine's attention layer, `flash_attn_varlen_func(q,
// k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, softmax_scale,
// causal=True, block_table)` (nanovllm/layers/attention.py:64-70), with K/V
// either contiguous (total_k, Hkv, D) rows or the paged cache (prefix cache).
//
// Math (sequence b with nq query rows and nk keys, GQA G = Hq / Hkv):
//   o[t, h] = softmax_j( q[t, h] . K[j, h / G] * scale ) . V[.., h / G],
//   j in [0, nk - nq + t]  (bottom-right aligned causal rule)
//
// Work: one workgroup per (128-row tile, kv head, sequence); the 128 rows are
// 128 / G consecutive tokens x the G query heads sharing the kv head, heaviest
// (last) tiles dispatched first. Each of the 8 wave64s owns 16 rows and its own
// online softmax. Per step of 64 keys the K and V rows go straight from HBM / L2
// into LDS (global_load_lds, two stages: the next step's rows land while this step
// computes, one barrier per step) and every wave computes
//   S^T = K . Q^T      16 x MFMA 16x16x32 (K is the A operand, read from LDS)
//   online softmax     exp2 domain, one row per lane (l % 16)
//   O^T += V^T . P^T   16 x MFMA (P rounded once; 32 with the lo part of P for
//                      tiles with rows that see few keys), V^T gathered with
//                      ds_read_b64_tr_b16
// Rows are written normalised at the end (no split over keys: a prefill has
// rows enough to fill the machine).
//
// Bound: the issue of the softmax's vector instructions beside the MFMAs, and power
// (a clock of 2.4 GHz falls as the kernel gets denser). 4 x 2048 tokens, 32 heads over 8:
// 193 us; ragged prompts over cached pages: 117. Four waves per SIMD hide each other's LDS
// and barrier waits: 8 waves of 16 rows against 4 of 32 (half the LDS reads, two waves per
// SIMD) measured 184 against 181 us there, 114 against 119, before the row sums went back
// to fp32 weights. The version that staged rows through registers, rescaled at every rise in
// any of 32 rows and ran each tile on any XCD took 354 and 266 us, with the same bits.
// What the loop leaves out:
//  * the lane exchange and the rescaling of 32 accumulators happen only where a vote says
//    that a maximum of the wave's 16 rows rises. (Raising it only by more than 1, 2 or 8 in
//    log2 units measured 3, 5 and 7% faster, but the rows' largest weight is then no longer
//    exactly 1: 1 - 4% more error against 64 bits.)
// What it does not leave out (193 and 117 us instead of 184 and 113): the weights enter the
// row sums in fp32, before they are rounded for P.V (sums of the rounded ones, a row of ones
// times P^T on the matrix cores, lose in fp16 every weight below 2^-25 of the row's largest),
// and a score is scaled and rounded once, ahead of the maximum (a multiply-add in the
// exponent gives other bits).
// All tiles of a (sequence, kv head) run on one XCD where the pairs divide by 8, so its
// K / V rows are read from that XCD's L2 (4 MB; 2048 keys are 1 MB).

#include <type_traits>

#include "sd_common.h"

namespace {

using sd::f32x4;
using sd::u32x4;

constexpr int kD = 128;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kRT = 1;                    // 16-row MFMA tiles per wave
constexpr int kRows = kWaves * 16 * kRT;  // query rows per workgroup
constexpr int kKeys = 64;               // keys per step
constexpr int kRowBytes = kD * 2;            // one key's K (or V) row
constexpr int kTile = kKeys * kRowBytes;     // one stage: the K tile, then the V tile

struct PrefillParams {
  const uint16_t* q;
  int64_t q_stok, q_shead;
  const uint16_t* k;  // contiguous (total_k, Hkv, D) rows, or the paged cache
  const uint16_t* v;
  int64_t s_tok;   // contiguous: token stride; paged: position stride within a block
  int64_t s_head;  // head stride
  int64_t s_blk;   // paged: block stride
  int32_t block_size, bs_shift, num_blocks;
  const int32_t* bt;  // (B, bt_stride) block table, NULL: contiguous K/V
  int64_t bt_stride;
  int32_t max_ctx;    // paged: table width x block size
  const int32_t* cu_q;  // (B + 1,)
  const int32_t* cu_k;  // (B + 1,)
  int32_t num_seqs, G, Hkv;
  int64_t total_q;
  float scale_log2;   // scale log2(e)
  uint16_t* out;
  int64_t o_stok, o_shead;
  int32_t by_xcd;  // (head, sequence) pairs are dealt to the XCDs
};

// K / V row addressing: contiguous rows; pages that hold whole 64-key steps (one block
// lookup per page, scalar); anything else (one lookup and a whole address per row).
enum Rows { kContiguous, kPagedSteps, kAnyRows };
constexpr int64_t kMaxStep = int64_t{1} << 24;  // row strides below keep a step within 32-bit offsets

// 16 bytes per lane from base + off to LDS byte 16 * lane of the wave-uniform address l.
// Written as assembly for the scalar-base form (no address arithmetic per step) and because
// the compiler makes a transpose read of LDS wait for every such load in flight; the loop
// waits itself, before its barrier. No register is written, and the address registers are
// read when the instruction issues.
__device__ __forceinline__ void load_lds16(const char* base, uint32_t off, const void* l) {
  const uint32_t dst = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)l));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(__builtin_amdgcn_readfirstlane(dst)), "v"(off), "s"(base)
               : "memory", "m0");
}
// The same with a whole address per lane.
__device__ __forceinline__ void load_lds16(const char* g, const void* l) {
  const uint32_t dst = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)l));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               ::"s"(__builtin_amdgcn_readfirstlane(dst)), "v"(g)
               : "memory", "m0");
}

// Tiles whose first token sees fewer than kSplitKeys keys ("split"): P enters P.V
// as hi + lo 16-bit parts (~16 mantissa bits, twice the P.V MFMAs). With n keys,
// rounding each P once costs about 2^-9 |v| / sqrt(n_eff) of absolute error, which
// nears the 2e-3 output tolerance when only a handful of keys are visible. Other
// tiles round P once to T, as flash attention does. Only the first
// ceil(kSplitKeys / tokens per tile) tiles of a sequence can be split.
constexpr int kSplitKeys = 128;

// Maximum over the four lanes that share l % 16 (v_permlane32_swap / 16_swap of v with
// itself leave a lane its own and its partner's value).
__device__ __forceinline__ float max_over_groups(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(a[0])),
            __builtin_bit_cast(float, static_cast<uint32_t>(a[1])));
  const uint32_t w = __builtin_bit_cast(uint32_t, v);
  const auto c = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(c[0])),
               __builtin_bit_cast(float, static_cast<uint32_t>(c[1])));
}

template <typename T, Rows ROWS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
void prefill_kernel(PrefillParams p) {
  __shared__ __attribute__((aligned(1024))) char sm[2][2 * kTile];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup -> (tile, kv head, sequence). Consecutive workgroups go to the 8 XCDs in
  // turn; with a multiple of 8 (head, sequence) pairs each XCD takes every eighth pair,
  // kPairs of them at a time: the heaviest tile of each, then the next (a heavy tile
  // started late would run alone at the end), the rows of all of them in that XCD's L2.
  int tile = static_cast<int>(gridDim.x) - 1 - static_cast<int>(blockIdx.x);
  int h = blockIdx.y, b = blockIdx.z;
  if (p.by_xcd) {
    constexpr uint32_t kPairs = 8;
    const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const uint32_t idx = lin >> 3, per = gridDim.y * gridDim.z / 8;
    const uint32_t chunk = idx / (gridDim.x * kPairs), in = idx - chunk * gridDim.x * kPairs;
    const uint32_t width = min(kPairs, per - chunk * kPairs);
    const uint32_t pair = (chunk * kPairs + in % width) * 8 + (lin & 7);
    tile = static_cast<int>(gridDim.x - 1 - in / width);
    h = static_cast<int>(pair % gridDim.y);
    b = static_cast<int>(pair / gridDim.y);
  }
  const int64_t q0 = p.cu_q[b];
  const int nq = max(p.cu_q[b + 1] - p.cu_q[b], 0);
  const int64_t k0 = p.cu_k[b];
  int nk = max(p.cu_k[b + 1] - p.cu_k[b], 0);
  nk = min(nk, p.max_ctx);
  const int tpw = kRows / p.G;  // tokens per workgroup
  const int t0 = tile * tpw;
  if (t0 >= nq) return;
  const int split_tiles = (kSplitKeys + tpw - 1) / tpw;
  const bool split = tile < split_tiles && nk - nq + t0 + 1 < kSplitKeys;
  const int tl = min(t0 + tpw, nq) - 1;  // last token of the tile

  // ---- this lane's rows (one per row tile): Q operand, causal limit
  int lim[kRT], qi[kRT], gq[kRT];
  bool valid[kRT];
  u32x4 qop[kRT][4];
  int wlast = -1, wfull = 0x7fffffff;
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    const int row = wave * 16 * kRT + rt * 16 + lr;
    qi[rt] = t0 + row / p.G;
    gq[rt] = row % p.G;
    valid[rt] = row < tpw * p.G && qi[rt] < nq && q0 + qi[rt] < p.total_q;
    lim[rt] = valid[rt] ? nk - nq + qi[rt] : -1;  // last visible key (-1: none)
    const uint16_t* qp =
        p.q + (valid[rt] ? (q0 + qi[rt]) * p.q_stok +
                               static_cast<int64_t>(h * p.G + gq[rt]) * p.q_shead
                         : 0) +
        lg * 8;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      qop[rt][s] = valid[rt] ? sd::load16(qp + s * 32) : u32x4{0u, 0u, 0u, 0u};
    wlast = max(wlast, lim[rt]);
    if (valid[rt]) wfull = min(wfull, lim[rt]);
  }
  // wave-uniform key range of this wave's rows: [0, wlast], and the keys every
  // valid row of the wave sees (no mask needed up to wfull)
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    wlast = max(wlast, __shfl_xor(wlast, off));
    wfull = min(wfull, __shfl_xor(wfull, off));
  }
  wlast = __builtin_amdgcn_readfirstlane(wlast);
  wfull = __builtin_amdgcn_readfirstlane(wfull);
  // workgroup key range: every key any of its rows sees
  const int glast = nk - nq + tl;
  const int nsteps = glast < 0 ? 0 : (glast + kKeys) / kKeys;

  float m_run[kRT], l_run[kRT];  // the row's maximum (log2 units); this lane's share of its sum
  f32x4 acc[kRT][8];
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    m_run[rt] = -INFINITY;
    l_run[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[rt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // ---- K / V loads: wave w brings rows 16 w .. 16 w + 15 of a step, four 256-byte rows
  //      per instruction (16 lanes each). The 16-byte unit u of row r lies at position
  //      u ^ (r & 15) of its K row and u ^ 2 (r & 7) of its V row, so that the K operand
  //      reads (16 rows, one unit) and the V transpose reads (16 rows, 32 bytes) each
  //      cover all banks. Rows past the last key read it again (masked).
  const char* kh = reinterpret_cast<const char*>(p.k + static_cast<int64_t>(h) * p.s_head);
  const char* vh = reinterpret_cast<const char*>(p.v + static_cast<int64_t>(h) * p.s_head);
  if (ROWS == kContiguous || !p.bt) {
    kh += k0 * p.s_tok * 2;
    vh += k0 * p.s_tok * 2;
  }
  const int32_t* btrow = p.bt ? p.bt + static_cast<int64_t>(b) * p.bt_stride : nullptr;
  // byte offsets of this lane's units from the step's first row (rows of a step lie within
  // 32 bits of it, but for kAnyRows)
  const uint32_t row_bytes = static_cast<uint32_t>(p.s_tok) * 2;
  constexpr int kLd = kKeys / kWaves / 4;  // loads of four rows, K and V each
  uint32_t koff[kLd], voff[kLd];
#pragma unroll
  for (int i = 0; i < kLd; ++i) {
    const int r = (wave * kLd + i) * 4 + lg;
    koff[i] = static_cast<uint32_t>(r) * row_bytes + (lr ^ (r & 15)) * 16;
    voff[i] = static_cast<uint32_t>(r) * row_bytes + (lr ^ ((r & 7) * 2)) * 16;
  }
  int page = -1;
  int64_t page_off = 0;  // bytes
  auto issue = [&](int step, int st) {
    char* dst = sm[st] + wave * kLd * 1024;
    if constexpr (ROWS == kAnyRows) {
#pragma unroll
      for (int i = 0; i < kLd; ++i) {
        const int r = (wave * kLd + i) * 4 + lg, tok = min(step * kKeys + r, nk - 1);
        int64_t off = static_cast<int64_t>(tok) * p.s_tok * 2;
        if (btrow) {
          const int pg = p.bs_shift >= 0 ? tok >> p.bs_shift : tok / p.block_size;
          const int blk = min(max(btrow[pg], 0), p.num_blocks - 1);
          off = (static_cast<int64_t>(blk) * p.s_blk + static_cast<int64_t>(tok - pg * p.block_size) * p.s_tok) * 2;
        }
        load_lds16(kh + off + (lr ^ (r & 15)) * 16, dst + i * 1024);
        load_lds16(vh + off + (lr ^ ((r & 7) * 2)) * 16, dst + kTile + i * 1024);
      }
    } else {
      int64_t first = static_cast<int64_t>(step) * kKeys * p.s_tok * 2;  // the step's first row
      if constexpr (ROWS == kPagedSteps) {
        const int pg = step * kKeys / p.block_size;
        if (pg != page) {  // uniform
          page = pg;
          const int blk = min(max(sd::load_scalar_i32(btrow + pg), 0), p.num_blocks - 1);
          page_off = (static_cast<int64_t>(blk) * p.s_blk - static_cast<int64_t>(pg) * p.block_size * p.s_tok) * 2;
        }
        first += page_off;
      }
      const int spare = step * kKeys + kKeys - nk;  // rows of the step past the last key
#pragma unroll
      for (int i = 0; i < kLd; ++i) {
        uint32_t ko = koff[i], vo = voff[i];
        if (spare > 0) {  // (last step)
          const uint32_t back =
              static_cast<uint32_t>(max((wave * kLd + i) * 4 + lg - (kKeys - 1 - spare), 0)) * row_bytes;
          ko -= back;
          vo -= back;
        }
        load_lds16(kh + first, ko, dst + i * 1024);
        load_lds16(vh + first, vo, dst + kTile + i * 1024);
      }
    }
  };
  // LDS offsets of this lane's operands. K: row lr (of 16), unit 4 s + lg. V: row
  // 4 lg + lr / 4, the 8-byte chunk lr % 4 of the 32 bytes of dims 16 dt.
  const int ka_lane = lr * kRowBytes + ((lg ^ (lr & 3)) * 16);
  const int va_lane = kTile + (lg * 4 + (lr >> 2)) * kRowBytes +
                      ((((lg & 1) * 4 + (lr >> 2)) * 32) | ((lr & 3) * 8));

  // one step's math on stage `base`; SPLIT adds the lo part of P
  auto compute = [&](const char* base, int tb, auto split_tag) {
#pragma clang fp contract(off)
    constexpr bool SPLIT = decltype(split_tag)::value;
    // ---- S^T in log2 units: lane holds S[row lr][key tb + 16 j + 4 lg + i] per row tile
    f32x4 sc[kRT][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 ka[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
        ka[s] = sd::load16(base + (ka_lane | ((s ^ (lr >> 2)) * 64)) + j * 16 * kRowBytes);
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) c = sd::Elem<T>::mfma(ka[s], qop[rt][s], c);
        sc[rt][j] = c * p.scale_log2;
      }
    }
    if (tb + kKeys - 1 > wfull) {  // some row of the wave does not see all 64 keys
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            sc[rt][j][i] = tb + j * 16 + lg * 4 + i <= lim[rt] ? sc[rt][j][i] : -INFINITY;
    }
    // ---- the rows' maxima; 16 rows are rescaled when one of theirs rises
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
      float m = fmaxf(sc[rt][0][0], sc[rt][0][1]);
#pragma unroll
      for (int e = 2; e < 16; e += 2) m = fmaxf(fmaxf(m, sc[rt][e / 4][e % 4]), sc[rt][e / 4][e % 4 + 1]);
      if (__any(m > m_run[rt])) {
        const float mnew = fmaxf(m_run[rt], max_over_groups(m));
        // (m_run = -inf: nothing accumulated yet; both -inf: the row sees no key so far)
        const float alpha = mnew == -INFINITY ? 1.f : sd::fast_exp2(m_run[rt] - mnew);
        l_run[rt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) acc[rt][dt] *= alpha;
        m_run[rt] = mnew;
      }
    }
    // ---- P = 2^(s - maximum) per 32-key half, summed in fp32 before the rounding
    u32x4 phi[kRT][2], plo[SPLIT ? kRT : 1][2];
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
      const float mb = m_run[rt] == -INFINITY ? 0.f : m_run[rt];
      float ps = 0.f;
#pragma unroll
      for (int kh2 = 0; kh2 < 2; ++kh2) {
        float pv[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          pv[q] = sd::fast_exp2(sc[rt][2 * kh2 + q / 4][q % 4] - mb);
#pragma unroll
        for (int q = 0; q < 8; ++q) ps += pv[q];
        if constexpr (SPLIT) {
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) sd::split_pack<T>(pv[2 * q], pv[2 * q + 1], hi[q], lo[q]);
          phi[rt][kh2] = u32x4{hi[0], hi[1], hi[2], hi[3]};
          plo[rt][kh2] = u32x4{lo[0], lo[1], lo[2], lo[3]};
        } else {
          phi[rt][kh2] = u32x4{sd::pack2<T>(pv[0], pv[1]), sd::pack2<T>(pv[2], pv[3]),
                               sd::pack2<T>(pv[4], pv[5]), sd::pack2<T>(pv[6], pv[7])};
        }
      }
      l_run[rt] += ps;
    }
    // ---- O^T += V^T . P^T; in 32-key half kh2, k-slot 8 lg + j <-> key
    //      32 kh2 + 4 lg + j (j < 4) and 32 kh2 + 16 + 4 lg + j - 4 (j >= 4)
#pragma unroll
    for (int kh2 = 0; kh2 < 2; ++kh2)
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        const char* c = base + (va_lane ^ (dt * 32)) + kh2 * 32 * kRowBytes;
        const uint2 v0 = sd::lds_read_tr16(c);
        const uint2 v1 = sd::lds_read_tr16(c + 16 * kRowBytes);
        const u32x4 vop = {v0.x, v0.y, v1.x, v1.y};
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt) {
          acc[rt][dt] = sd::Elem<T>::mfma(vop, phi[rt][kh2], acc[rt][dt]);
          if constexpr (SPLIT) acc[rt][dt] = sd::Elem<T>::mfma(vop, plo[rt][kh2], acc[rt][dt]);
        }
      }
  };
  auto loop = [&](auto split_tag) {
    for (int step = 0; step < nsteps; ++step) {
      // this step's rows have landed, and every wave is done with the other stage
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (step + 1 < nsteps) issue(step + 1, (step + 1) & 1);
      if (step * kKeys <= wlast) compute(sm[step & 1], step * kKeys, split_tag);
    }
  };
  if (nsteps > 0) issue(0, 0);
  if (split) loop(std::true_type{});
  else loop(std::false_type{});

  // ---- normalised rows: lane holds O[row lr][dims 16 dt + 4 lg .. +4]
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    const float l = sd::sum_over_groups(l_run[rt]);
    if (!valid[rt]) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* op = p.out + (q0 + qi[rt]) * p.o_stok +
                   static_cast<int64_t>(h * p.G + gq[rt]) * p.o_shead;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      uint2 w;
      w.x = sd::pack2<T>(acc[rt][dt].x * inv, acc[rt][dt].y * inv);
      w.y = sd::pack2<T>(acc[rt][dt].z * inv, acc[rt][dt].w * inv);
      *reinterpret_cast<uint2*>(op + dt * 16 + lg * 4) = w;
    }
  }
}

template <typename T>
void launch(const PrefillParams& p, dim3 grid, hipStream_t st) {
  if (!p.bt && p.s_tok < kMaxStep)
    hipLaunchKernelGGL((prefill_kernel<T, kContiguous>), grid, dim3(kThreads), 0, st, p);
  else if (p.block_size % kKeys == 0 && p.s_tok < kMaxStep)
    hipLaunchKernelGGL((prefill_kernel<T, kPagedSteps>), grid, dim3(kThreads), 0, st, p);
  else
    hipLaunchKernelGGL((prefill_kernel<T, kAnyRows>), grid, dim3(kThreads), 0, st, p);
}

}  // namespace

extern "C" int sd_prefill_attention(
    const void* q, int64_t q_stride_tok, int64_t q_stride_head, const void* k, const void* v,
    int64_t kv_stride_tok, int64_t kv_stride_head, int64_t kv_stride_block, int64_t num_blocks,
    int32_t block_size, const int32_t* block_table, int64_t bt_stride, int32_t max_blocks_per_seq,
    const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int32_t max_seqlen_q,
    int64_t total_q, int32_t num_seqs, int32_t num_q_heads, int32_t num_kv_heads,
    int32_t head_dim, float scale, int32_t dtype, void* out, int64_t out_stride_tok,
    int64_t out_stride_head, void* stream) {
  sd::clear_error();
  if (num_seqs < 0 || max_seqlen_q < 0 || total_q < 0 || num_q_heads <= 0 || num_kv_heads <= 0 ||
      num_q_heads % num_kv_heads != 0) {
    sd::set_error("prefill_attention: invalid sizes (seqs=%d max_q=%d hq=%d hkv=%d)", num_seqs,
                  max_seqlen_q, num_q_heads, num_kv_heads);
    return SD_ERR_VALUE;
  }
  const int G = num_q_heads / num_kv_heads;
  if (head_dim != kD || G > kRows || kRows % G != 0 || (dtype != SD_BF16 && dtype != SD_F16)) {
    sd::set_error("prefill_attention: head_dim 128, q heads per kv head dividing 128, bf16/fp16 "
                  "only (head_dim=%d G=%d dtype=%d)", head_dim, G, dtype);
    return SD_ERR_UNSUPPORTED;
  }
  if (num_seqs == 0 || total_q == 0 || max_seqlen_q == 0) return SD_OK;
  if (num_seqs > 65535 || num_kv_heads > 65535) {
    sd::set_error("prefill_attention: at most 65535 sequences and kv heads per call");
    return SD_ERR_UNSUPPORTED;
  }
  if (!q || !k || !v || !cu_seqlens_q || !cu_seqlens_k || !out) {
    sd::set_error("prefill_attention: null pointer argument");
    return SD_ERR_VALUE;
  }
  if (block_table && (block_size <= 0 || num_blocks <= 0 || max_blocks_per_seq <= 0)) {
    sd::set_error("prefill_attention: paged K/V needs block_size, num_blocks, table width");
    return SD_ERR_VALUE;
  }
  const int64_t max_ctx = static_cast<int64_t>(max_blocks_per_seq) * block_size;
  if ((block_table && max_ctx > (1ll << 30)) || max_seqlen_q > (1 << 30)) {
    sd::set_error("prefill_attention: context bound %lld or query length %d too large",
                  (long long)max_ctx, max_seqlen_q);
    return SD_ERR_UNSUPPORTED;
  }
  if (!sd::strides_ok({q_stride_tok, q_stride_head, kv_stride_tok, kv_stride_head,
                       kv_stride_block, bt_stride, out_stride_tok, out_stride_head})) {
    sd::set_error("prefill_attention: strides must lie in [-2^40, 2^40] elements");
    return SD_ERR_VALUE;
  }
  if (!sd::aligned16(q) || !sd::aligned16(k) || !sd::aligned16(v) || q_stride_tok % 8 ||
      q_stride_head % 8 || kv_stride_tok % 8 || kv_stride_head % 8 || kv_stride_block % 8 ||
      (reinterpret_cast<uintptr_t>(out) & 7u) || out_stride_tok % 4 || out_stride_head % 4 ||
      kv_stride_tok < 0 || kv_stride_head < 0 || kv_stride_block < 0) {
    sd::set_error("prefill_attention: rows must be 16-byte aligned (output 8-byte)");
    return SD_ERR_UNSUPPORTED;
  }
  PrefillParams p;
  p.q = static_cast<const uint16_t*>(q);
  p.q_stok = q_stride_tok;
  p.q_shead = q_stride_head;
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.s_tok = kv_stride_tok;
  p.s_head = kv_stride_head;
  p.s_blk = kv_stride_block;
  p.block_size = block_size;
  p.bs_shift = block_size > 0 && (block_size & (block_size - 1)) == 0 ? __builtin_ctz(block_size) : -1;
  p.num_blocks = static_cast<int32_t>(num_blocks > 0x7fffffff ? 0x7fffffff : num_blocks);
  p.bt = block_table;
  p.bt_stride = bt_stride;
  p.max_ctx = block_table ? static_cast<int32_t>(max_ctx) : 0x7fffffff;
  p.cu_q = cu_seqlens_q;
  p.cu_k = cu_seqlens_k;
  p.num_seqs = num_seqs;
  p.G = G;
  p.Hkv = num_kv_heads;
  p.total_q = total_q;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.out = static_cast<uint16_t*>(out);
  p.o_stok = out_stride_tok;
  p.o_shead = out_stride_head;
  const int tpw = kRows / G;
  const int64_t longest = max_seqlen_q < total_q ? max_seqlen_q : total_q;
  const dim3 grid(static_cast<unsigned>((longest + tpw - 1) / tpw),
                  static_cast<unsigned>(num_kv_heads), static_cast<unsigned>(num_seqs));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t pairs = static_cast<int64_t>(num_kv_heads) * num_seqs;
  p.by_xcd = pairs % 8 == 0 && pairs * grid.x < (int64_t{1} << 31);
  if (dtype == SD_BF16) launch<__bf16>(p, grid, st);
  else launch<_Float16>(p, grid, st);
  return sd::check_launch("prefill_attention");
}
