// Shared by the quantized GEMM sources: weight formats, operand conversion, buffer loads.
#pragma once

#include "common.hpp"

namespace cir {

__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }

// 8 Q4_0 nibbles of one dword -> 8 fp16 values (q - 8) * 2^-12, all exact.  A nibble q
// masked in place reads as the fp16 subnormal q * 2^-24 (16q * 2^-24 for the high nibble
// of a byte); one packed FMA scales it by 2^12 (2^8) and subtracts 8 * 2^-12.  That is two
// VALU ops per pair, as many as an or-in of the exponent 1024 would need with one
// v_and_or_b32, which the compiler does not form from two literal masks.  The kernels'
// fp16 denormal mode (float_denorm_mode_16_64 = 3, the default) keeps the subnormals.
__device__ __forceinline__ f16x8 dq_q4(uint32_t w) {
  const f16x2 s12 = {(f16)4096.0f, (f16)4096.0f};
  const f16x2 s8 = {(f16)256.0f, (f16)256.0f};
  const f16x2 c8 = {(f16)-0.001953125f, (f16)-0.001953125f};  // -8 * 2^-12
  const uint32_t t = w >> 8;
  const f16x2 p0 = as_h2(w & 0x000F000Fu) * s12 + c8;
  const f16x2 p1 = as_h2(w & 0x00F000F0u) * s8 + c8;
  const f16x2 p2 = as_h2(t & 0x000F000Fu) * s12 + c8;
  const f16x2 p3 = as_h2(t & 0x00F000F0u) * s8 + c8;
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// 8 Q8_0 int8 values (two dwords) -> 8 exact fp16 integers q.  After the sign flip each
// byte is q + 128; one v_perm_b32 places bytes 0 and 2 (or 1 and 3) under 0x64 bytes,
// giving fp16 1024 + q + 128.  Byte selectors 4..7 pick bytes 0..3 of the first
// operand, 0..3 those of the second.
__device__ __forceinline__ f16x8 dq_q8(uint32_t w0, uint32_t w1) {
  const f16x2 c1152 = {(f16)-1152.0f, (f16)-1152.0f};
  constexpr uint32_t k64 = 0x64646464u, even = 0x00060004u, odd = 0x00070005u;
  w0 ^= 0x80808080u;
  w1 ^= 0x80808080u;
  const f16x2 p0 = as_h2(__builtin_amdgcn_perm(w0, k64, even)) + c1152;
  const f16x2 p1 = as_h2(__builtin_amdgcn_perm(w0, k64, odd)) + c1152;
  const f16x2 p2 = as_h2(__builtin_amdgcn_perm(w1, k64, even)) + c1152;
  const f16x2 p3 = as_h2(__builtin_amdgcn_perm(w1, k64, odd)) + c1152;
  return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// Row formats (per-row scale and zero point) reuse the tile layout of the block
// format with the same code width: 4-bit codes sit like Q4_0 nibbles, 8-bit codes
// like Q8_0 bytes.  Their tiled copy holds no per-block scales; after the codes come
// fp32 scale[rows] and fp32 offset[rows] (rows padded to a multiple of 16).
__host__ __device__ constexpr bool is_row_fmt(int fmt) { return fmt == CIR_I4_ROW || fmt == CIR_I8_ROW; }
__host__ __device__ constexpr int layout_fmt(int fmt) {
  return (fmt == CIR_Q4_0 || fmt == CIR_I4_ROW) ? CIR_Q4_0 : CIR_Q8_0;
}
__host__ __device__ inline size_t quant_bytes_per_lane(int fmt) { return layout_fmt(fmt) == CIR_Q4_0 ? 16 : 32; }

// Accumulators of a 4-bit layout hold 2^-12 times the dot products (dq_q4's scale); each
// kernel multiplies them by kAccScale once, when its k range is done.  Scaling by a power
// of two commutes with every fp32 rounding before it (no value comes near the fp32
// subnormal range), so the results are the ones integer weights would give.
template <int FMT> inline constexpr float kAccScale = layout_fmt(FMT) == CIR_Q4_0 ? 4096.f : 1.f;
__host__ __device__ inline size_t block_bytes(int fmt) { return fmt == CIR_Q4_0 ? 18 : 34; }
__host__ __device__ inline bool valid_fmt(int fmt) {
  return fmt == CIR_Q4_0 || fmt == CIR_Q8_0 || fmt == CIR_I4_ROW || fmt == CIR_I8_ROW;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // plain vector: no struct memcpy, stays in VGPRs

__device__ __forceinline__ uint4 buf16(rsrc_t r, uint32_t voff, uint32_t soff) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return uint4{v.x, v.y, v.z, v.w};
}
__device__ __forceinline__ uint2 buf8(rsrc_t r, uint32_t voff, uint32_t soff) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  return uint2{v.x, v.y};
}

constexpr int kCUs = 256;

// The large-m kernel (qgemm_xl.hip), m > 32: fp32 split-k partials; the SwiGLU over interleaved gate/up tiles (one
// split; odt: CIR_F16 or CIR_F32); or the greedy head's candidates (one split; returns how many per row).
template <int FMT>
void launch_qgemm_xl(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, float* part, int M, int N, int K,
                     int splits, hipStream_t s);
template <int FMT>
void launch_qgemm_xl_swiglu(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, void* act, int odt, int M,
                            int N, int K, hipStream_t s);
template <int FMT>
int launch_qgemm_xl_argmax(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, float* cand_v, int* cand_i,
                           int M, int N, int K, hipStream_t s);

}  // namespace cir
