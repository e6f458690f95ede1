// Number formats, record geometry and paging shared by the INT2 history kernels (history.hip,
// history_chunk.hip).
#pragma once

#include "attention.h"

namespace oscar {

typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
typedef int32_t i32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i32x2* lds_i32x2_ptr_t;

constexpr int kChunk = 64;                       // tokens per wavefront iteration
constexpr int kPieces = 9;                       // 16-byte pieces staged per record
constexpr int kRec = 16 * kPieces;               // 144: LDS record stride
constexpr int kSkew = 4;                         // record base offset: V codes 8-aligned
constexpr int kStageBytes = kChunk * kRec + 16;  // 9232
constexpr int kDma = kChunk * kPieces / 64;      // 9 loads of 16 bytes per lane per chunk
constexpr int kTableCache = 256;                 // kernel blocks whose offsets live in LDS
constexpr float kTheta = 8.0f;                   // lazy-max slack, log2 units
constexpr int kQTerms = 2;
constexpr uint32_t kNoBlock = 0xffffffffu;

static_assert(kDma * 64 == kChunk * kPieces, "a chunk image is whole DMA instructions");
static_assert(kStageBytes % 16 == 0, "stages stay 16-byte aligned");

// ---------------------------------------------------------------- number formats

// Packed 2-bit codes -> FP4 nibbles: codes 0, 2, 4, .. (even) or 1, 3, 5, .. (odd) of a dword.
__device__ __forceinline__ int32_t even_codes(uint32_t w) {
  return static_cast<int32_t>(w & 0x33333333u);
}
__device__ __forceinline__ int32_t odd_codes(uint32_t w) {
  return static_cast<int32_t>((w >> 2) & 0x33333333u);
}

// S^T tile += K (FP4, A) x Q (FP8, B); K = 128 head dims.
__device__ __forceinline__ f32x4 mfma_qk(const i32x8& k4, const i32x8& q8, f32x4 c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(k4, q8, c, 4, 0, 0, 0, 0, 0);
}
// O tile += 2^(sa - 127) P (FP8, A) x V (FP4, B); K = 64 tokens x {hi, lo}.
__device__ __forceinline__ f32x4 mfma_pv(const i32x8& p8, const i32x8& v4, f32x4 c, int sa) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(p8, v4, c, 0, 4, 0, sa, 0, 127);
}

// Four floats -> four e4m3 bytes (round to nearest even).
__device__ __forceinline__ uint32_t fp8x4(float x0, float x1, float x2, float x3) {
  const int v = __builtin_amdgcn_cvt_pk_fp8_f32(x0, x1, 0, false);
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(x2, x3, v, true));
}
// Rounds x to e4m3 bytes and leaves the (exact) residual x - rounded in x.
__device__ __forceinline__ uint32_t fp8x4_take(float (&x)[4]) {
  const uint32_t b = fp8x4(x[0], x[1], x[2], x[3]);
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(b), false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(b), true);
  x[0] -= lo[0];
  x[1] -= lo[1];
  x[2] -= hi[0];
  x[3] -= hi[1];
  return b;
}

__device__ __forceinline__ float h16lo(uint32_t x) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(x & 0xffffu)));
}
__device__ __forceinline__ float h16hi(uint32_t x) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(x >> 16)));
}

// ---------------------------------------------------------------- paging

// Offset (32-byte units) of kernel block kb of this request/head, or kNoBlock
// (kernels.py:392-399: block table column -> physical page and block within the page).
__device__ __forceinline__ uint32_t kernel_block_offset(const AttnArgs& a, const Task& t, int head,
                                                        int kb) {
  if (kb < 0 || kb >= a.table_columns) return kNoBlock;
  const int blk = a.table[static_cast<int64_t>(t.req) * a.table_stride + kb];
  if (blk < 0) return kNoBlock;
  const uint32_t page = fastdiv(static_cast<uint32_t>(blk), a.L.bpp_div);
  const uint32_t inpage = static_cast<uint32_t>(blk) - page * a.L.bpp;
  const int64_t off = static_cast<int64_t>(page) * a.L.page_bytes +
                      (static_cast<int64_t>(inpage) * a.L.bk * a.L.kv_heads + head) * kSlot;
  // The whole kernel block must lie inside the history buffer.
  if (off + static_cast<int64_t>(a.L.bk) * a.L.kv_heads * kSlot > a.history_bytes) return kNoBlock;
  return static_cast<uint32_t>(off >> 5);
}

}  // namespace oscar
