// w8a16.h — what the W8A16 kernels share: dequantization in MFMA operand order
// and the interface of the many-row kernel (w8a16_gemm.hip).
#pragma once

#include "sd_common.h"

namespace sd {

__device__ __forceinline__ float load_scale(const void* s, int dtype, int64_t i) {
  if (dtype == SD_F32) return static_cast<const float*>(s)[i];
  const uint16_t b = static_cast<const uint16_t*>(s)[i];
  return dtype == SD_BF16 ? from_bits<__bf16>(b) : from_bits<_Float16>(b);
}

// 8 int8 (two dwords) -> 8 x 16-bit floats in MFMA operand order.
// fp16: (b ^ 0x80) in the low byte under exponent byte 0x64 is the fp16 value
// 1024 + b + 128, exact; subtracting 1152 (packed fp16) gives b.
// bf16: v_cvt_f32_i32 of one sign-extended byte (an SDWA operand, so the byte
// select is free) is b as fp32, whose upper half is the exact bf16 (|b| <= 128
// needs 8 significant bits): 1.5 VALU instructions per element, against 2.75
// through v_cvt_f32_ubyte of (b ^ 0x80) and a subtraction.
template <typename T> __device__ __forceinline__ u32x4 dequant8(uint32_t w0, uint32_t w1);

template <> __device__ __forceinline__ u32x4 dequant8<_Float16>(uint32_t w0, uint32_t w1) {
  const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
  const f16x2 off = {static_cast<_Float16>(1152.f), static_cast<_Float16>(1152.f)};
  auto pair = [&](uint32_t u, uint32_t sel) {
    return __builtin_bit_cast(uint32_t,
                              __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, sel)) - off);
  };
  return u32x4{pair(u0, 0x04010400u), pair(u0, 0x04030402u), pair(u1, 0x04010400u),
               pair(u1, 0x04030402u)};
}

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo),
                               0x07060302u);
}

template <> __device__ __forceinline__ u32x4 dequant8<__bf16>(uint32_t w0, uint32_t w1) {
  auto byte = [](uint32_t w, int i) { return static_cast<float>(static_cast<int8_t>(w >> (8 * i))); };
  return u32x4{bf16_pair(byte(w0, 0), byte(w0, 1)), bf16_pair(byte(w0, 2), byte(w0, 3)),
               bf16_pair(byte(w1, 0), byte(w1, 1)), bf16_pair(byte(w1, 2), byte(w1, 3))};
}

// ------------------------------------------------------------ many-row kernel
struct W8GemmArgs {
  const uint16_t* x;
  int64_t xs;
  const int8_t* w;
  int64_t ws;
  const void* scale;
  int32_t scale_dtype;
  int32_t group;  // 0: per channel
  const uint16_t* bias;
  uint16_t* y;
  int64_t ys;
  int32_t M, N, K;
  int32_t dtype;
};

// How the many-row kernel runs a shape: a tile (w8a16_gemm.hip), and K slices (1, 2, 3, 4, 6,
// 8, 12 or 16; 0: the shape stays on the 16-row kernels). Slice s of n covers the stages
// [s S / n, (s + 1) S / n) of S = K / 64 / kb stages of kb 64-column steps (1 or 2).
struct W8GemmPlan {
  int tile, slices, kb;
};
// A function of the sizes and the device's compute units, so that the forms that stay on the
// 16-row kernels (SiLU, RMSNorm) can add the same slices in the same order. About 0.7 us of
// host time: a call makes it once.
W8GemmPlan w8a16_gemm_plan(int64_t M, int64_t N, int64_t K, int32_t group);
// The same without memory for the partial sums: the 16-row kernels (no slices; they add the
// shape's slices inside a workgroup, with the same bits) or one slice.
W8GemmPlan w8a16_gemm_plan_unsliced(int64_t M, int64_t N, int64_t K, int32_t group);
// The plan as sd_w8a16_plan returns it.
int64_t w8a16_gemm_plan_code(const W8GemmPlan& pl);
// Bytes of fp32 partial sums (0 with one slice).
size_t w8a16_gemm_workspace(const W8GemmPlan& pl, int64_t M, int64_t N);
// Whether the kernel can run this call (its sizes, LDS scale table and 32-bit row offsets).
bool w8a16_gemm_fits(const W8GemmArgs& a, const W8GemmPlan& pl);
// The launch (or, with `floor`, its loads alone).
int w8a16_gemm(const W8GemmArgs& a, const W8GemmPlan& pl, void* workspace, hipStream_t st, bool floor);

}  // namespace sd
