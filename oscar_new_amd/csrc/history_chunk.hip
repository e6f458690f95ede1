// INT2 history branch of continuation chunks (more than 16 query tokens per request): 128
// (query, head) rows of one request and KV head per workgroup share every spread code.
//
// Reference: oscar_ascend/kernels.py:290-482 (`_attention_kernel` with IS_RAW false), split
// ranges kernels.py:368-370. Scores, masks, per-split normalization and LSE as in history.hip.
//
// The task-shaped kernel of history.hip serves the rows of four query tokens per workgroup, so
// a chunk's 2-bit codes are spread into FP4 operands once per 16 rows (a third of its vector
// instructions), a quarter of its rows are padding with six heads, and one split per request
// leaves a short chunk on a few CUs. Here eight wavefronts of 16 rows each take 128 consecutive
// rows (any number of heads, padding only in a request's last tile) and share a pipeline over
// 128-token chunks of the history:
//   * raw records arrive by direct-to-LDS DMA, four stages, three chunks ahead;
//   * each wavefront spreads an eighth of a coming chunk from its raw stage into operand images
//     (K: per 16-token tile and 128-dim half, V: per 16 output dims, transposed reads), stored
//     in lane order so that an operand is one conflict-free 16-byte read per lane;
//   * every wavefront computes the current chunk from the images: 32 QK and 32 PV MFMAs
//     (the PV k dimension holds 128 tokens; the FP8 high and low terms of P are two MFMAs over
//     the same V operand).
// One barrier per chunk. The wavefronts of a workgroup hold different rows, so no states are
// merged. 150 KB of LDS, one workgroup per CU, two wavefronts per SIMD.
//
// What bounds it: vector issue, and the waits of a wavefront for the others of its workgroup. A
// chunk takes a SIMD's two wavefronts 9100 cycles: their vector instructions (about 460 per
// wavefront, beside 64 MFMAs) hold its issue for 58 % of them, the matrix pipe is busy for 45 %, and
// a wavefront spends 38 % of its cycles at an s_waitcnt or the barrier (counters, 2048 tokens x 6
// heads over 32768). That chunk: 654 us (task-shaped kernel, one split) -> 415 us with five splits;
// 389 tokens over 20011 beside 15 decodes: 254 -> 102 us. Which steps take it:
// config.chunk_kernel_pays.
#include <type_traits>

#include "dma.h"
#include "history.h"

namespace oscar {
namespace {

constexpr int kWavesC = 8;
constexpr int kThreadsC = kWavesC * kWave;
constexpr int kRowsC = 16 * kWavesC;       // rows per workgroup
constexpr int kTokC = 128;                 // tokens per chunk: two 64-token DMA halves
constexpr int kRawC = kTokC * kRec + 16;   // raw stage: record r at kSkew + 144 r
constexpr int kRawStagesC = 4;
constexpr int kCopiesC = 2 * kDma;         // 1 KiB copies per chunk, copy i by wavefront i % 8
constexpr int kTableC = 1024;              // chunks whose record offsets live in LDS

struct ChunkLds {
  uint8_t raw[kRawStagesC][kRawC] __attribute__((aligned(16)));
  u32x4 k[2][2][8][kWave];  // [buffer][128-dim half][16-token tile][lane]
  u32x4 v[2][16][kWave];    // [buffer][2 c + parity: dims 32 c + 2 n + parity][lane]
  // [c % 4][token]: K scale and zero in units of fq (a score is two multiply-adds), V scale | zero.
  float ks[4][kTokC] __attribute__((aligned(16)));
  float kz[4][kTokC] __attribute__((aligned(16)));
  uint32_t vsz[4][kTokC] __attribute__((aligned(16)));
  uint2 off[kTableC];  // records of a chunk's two 64-token halves (32-byte units; kNoBlock: unmapped)
  int count[kWavesC], found[2];
};
static_assert(sizeof(ChunkLds) <= 160 * 1024, "one workgroup per CU");
static_assert(kRawC % 16 == 0, "raw stages stay 16-byte aligned");

// S^T tile += 2^(sb - 127) K (FP4) x Q (FP8), the scale per query row (column).
__device__ __forceinline__ f32x4 mfma_qk_scaled(u32x4 k, const i32x8& q8, f32x4 c, int sb) {
  const i32x8 k4 = {(int)k[0], (int)k[1], (int)k[2], (int)k[3], 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(k4, q8, c, 4, 0, 0, 127, 0, sb);
}

typedef int16_t i16x2 __attribute__((ext_vector_type(2)));

// Four floats / scale -> four e4m3 bytes; scale is a power of two.
__device__ __forceinline__ uint32_t fp8x4_scaled(const float (&x)[4], float scale) {
  i16x2 r = {0, 0};
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[0], x[1], scale, false);
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[2], x[3], scale, true);
  return __builtin_bit_cast(uint32_t, r);
}
// The same over the bits of x[0], dead afterwards (both halves are overwritten: no zeroed register).
__device__ __forceinline__ uint32_t fp8x4_scaled_last(const float (&x)[4], float scale) {
  i16x2 r = __builtin_bit_cast(i16x2, x[0]);
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[0], x[1], scale, false);
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(r, x[2], x[3], scale, true);
  return __builtin_bit_cast(uint32_t, r);
}
// The same, leaving the exact residual in x.
__device__ __forceinline__ uint32_t fp8x4_scaled_take(float (&x)[4], float scale) {
  const uint32_t b = fp8x4_scaled(x, scale);
  const f32x2 lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(b), scale, false);
  const f32x2 hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(b), scale, true);
  x[0] -= lo[0];
  x[1] -= lo[1];
  x[2] -= hi[0];
  x[3] -= hi[1];
  return b;
}

// max(a, b, c) without the quieting of NaN operands that fmaxf adds to selected values.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Tile `x` of the step: the tiles of 128 rows of all requests, in task order. A tile starts in
// the task whose rows hold its first row (a task holds at most 32 rows, so at most one start).
// Every thread calls it; false past the last tile.
__device__ __forceinline__ bool find_tile(const AttnArgs& a, int programs, int x, ChunkLds& lds,
                                          int& req, int& tile) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int count = max(min(a.task_count[0], programs), 0);
  const int task_rows = a.qt * a.g;
  if (threadIdx.x == 0) lds.found[0] = -1;
  __syncthreads();
  int before = 0;
  for (int c0 = 0; c0 < count && before <= x; c0 += kThreadsC) {
    const int i = c0 + static_cast<int>(threadIdx.x);
    int r = -1, b = 0;
    bool start = false;
    if (i < count) {
      r = a.tasks[2 * i];
      const int row0 = a.tasks[2 * i + 1] * a.g;
      b = (row0 + kRowsC - 1) / kRowsC;
      start = b * kRowsC < row0 + task_rows;
    }
    const uint64_t mask = __ballot(start);
    if (lane == 0) lds.count[wave] = __popcll(mask);
    __syncthreads();
    int at = before + __popcll(mask & ((1ull << lane) - 1));
    int all = 0;
#pragma unroll
    for (int w = 0; w < kWavesC; ++w) {
      at += w < wave ? lds.count[w] : 0;
      all += lds.count[w];
    }
    if (start && at == x) {
      lds.found[0] = r;
      lds.found[1] = b;
    }
    before += all;
    __syncthreads();  // counts are read, the tile is published
  }
  req = uniform(lds.found[0]);
  tile = uniform(lds.found[1]);
  return req >= 0;
}

__global__ __launch_bounds__(kThreadsC, 2) void history_chunk_kernel(const AttnArgs a,
                                                                     int32_t programs) {
  __shared__ ChunkLds lds;
  Task t;
  int tile;
  // Workgroup ((tile, kv head), split): the tiles that exist dispatch first. Their bound grows with
  // the engine's request capacity, and a workgroup past the last tile, too, holds a whole CU while
  // it looks for its tile; with the tiles varying fastest these came between the others (64 tokens
  // over 16000, capacity 256, 16 splits: 94 us, this order 49; 300 tokens and three decodes over
  // 30000, 11 splits: 182 and 108).
  const int unit = static_cast<int>(blockIdx.x) / a.splits, h = a.L.kv_heads;
  const int split = static_cast<int>(blockIdx.x) - unit * a.splits, head = unit % h;
  if (!find_tile(a, programs, unit / h, lds, t.req, tile)) return;
  t.qoff = 0;
  t.qstart = a.qstarts[t.req];
  t.qlen = min(a.qstarts[t.req + 1], a.counts[1]) - t.qstart;
  t.prefix = a.seq_lens[t.req] - t.qlen;
  t.sink_len = min(a.L.sink, t.prefix);
  t.recent_begin = max(t.sink_len, t.prefix - a.L.recent);
  const int rows = t.qlen * a.g;  // rows of this request and KV head
  const int row_base = tile * kRowsC;
  if (row_base >= rows) return;
  int begin, end;
  split_range(t.recent_begin - t.sink_len, a.block_n, a.splits, split, begin, end);
  const int p_lo = max(t.sink_len + begin, 0), p_hi = t.sink_len + end;

  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int first = p_lo >> 7;
  const int nchunk = p_lo < p_hi ? ((p_hi - 1) >> 7) - first + 1 : 0;
  // ---- copies: copy i of a chunk is DMA i % 9 of its half i / 9 (16-byte piece 64 (i % 9) +
  // lane: record piece / 9, bytes 16 (piece % 9)); this wavefront's are wave, wave + 8, wave + 16.
  const uint32_t tok_bytes = static_cast<uint32_t>(a.L.kv_heads) * kSlot;
  const uint32_t in_kb_mask = static_cast<uint32_t>(a.L.bk - 1);
  // Record offsets of chunk c's halves (of none at or past p_hi).
  auto find_records = [&](int c) -> uint2 {
    uint32_t off[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int t0 = ((first + c) << 7) + 64 * half;
      off[half] = t0 < p_hi ? kernel_block_offset(a, t, head, t0 >> a.L.bk_shift) : kNoBlock;
      // A 64-token run of records is a whole number of 32-byte units.
      if (off[half] != kNoBlock)
        off[half] += ((static_cast<uint32_t>(t0) & in_kb_mask) * tok_bytes) >> 5;
    }
    return make_uint2(off[0], off[1]);
  };
  // Chunk c's offsets, wave-uniform.
  auto records = [&](int c) -> uint2 {
    uint2 r = lds.off[min(c, kTableC - 1)];
    if (c >= kTableC) r = find_records(c);
    return make_uint2(static_cast<uint32_t>(uniform(static_cast<int>(r.x))),
                      static_cast<uint32_t>(uniform(static_cast<int>(r.y))));
  };
  uint32_t mapped = 0;  // bits 2 (c % 8) and + 1: the halves of chunk c (copied so far) have records
  auto issue = [&](int c, uint2 rec32) {
    const uint32_t stage = lds_addr(lds.raw[c % kRawStagesC]) + kSkew;
    const uint32_t bits = (rec32.x != kNoBlock ? 1u : 0u) | (rec32.y != kNoBlock ? 2u : 0u);
    mapped = (mapped & ~(3u << 2 * (c & 7))) | bits << 2 * (c & 7);
    // The lane is read anew: offsets kept across the chunk loop were spilled, and a reload between
    // the copies waits for the copies before it.
    int el;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(el));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int i = wave + 8 * k;
      if (i >= kCopiesC) break;
      const int half = i >= kDma ? 1 : 0;
      const int piece = 64 * (i - kDma * half) + el;
      const uint32_t rec = (static_cast<uint32_t>(piece) * 7282u) >> 16;  // piece / 9 (below 576)
      const uint32_t voff = rec * tok_bytes + 16 * (static_cast<uint32_t>(piece) - 9 * rec);
      const uint32_t off32 = half ? rec32.y : rec32.x;
      // An unmapped block copies the buffer's first records.
      const uint64_t at = off32 != kNoBlock ? static_cast<uint64_t>(off32) << 5 : 0;
      dma_x4(a.history + at, voff, stage + 1024 * i);
    }
  };
  for (int c = threadIdx.x; c < min(nchunk, kTableC); c += kThreadsC) lds.off[c] = find_records(c);
  __syncthreads();
  const int ahead = min(nchunk, 3);
  for (int c = 0; c < ahead; ++c) issue(c, records(c));

  // ---- this wavefront's 16 query rows as FP8 B operands (kQTerms terms, nearly exact for bf16
  // rows). Row n of lane (n, g), scaled to [128, 256) by a power of two that the MFMA takes back
  // (sb). Byte e of dword d of half h: dim 128 h + 64 (d / 4) + 16 g + sigma(4 (d % 4) + e),
  // sigma(j) = 2 (j % 8) + j / 8 (history.hip).
  const bool live = row_base + 16 * wave < rows;
  const int my_row = row_base + 16 * wave + n;
  const int qi = static_cast<int>(fastdiv(static_cast<uint32_t>(my_row), a.g_div));
  const int64_t my_token = static_cast<int64_t>(t.qstart) + qi;
  const bool valid = my_row < rows && my_token >= 0 && my_token < a.n;
  i32x8 qb[2][kQTerms];
  // The score in log2 units is fq (s acc + z qs), acc = sum_d q_d c_d / 2, qs = sum_d q_d / 2.
  float qs;
  const float fq = 2.0f * a.scale_log2;
  int sb;
  {
    const uint16_t* src = a.query + (valid ? my_token * a.qs0 +
                                                 (head * a.g + (my_row - qi * a.g)) * a.qs1
                                           : 0);
    float x[2][2][16];
    float mx = 0.f, sum = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const u32x4 w = *reinterpret_cast<const u32x4*>(src + 128 * h + 64 * b + 16 * g + 8 * q);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x0 = valid ? bf16_to_float(w[i] & 0xffffu) : 0.f;
            const float x1 = valid ? bf16_to_float(w[i] >> 16) : 0.f;
            sum += x0 + x1;
            x[h][b][8 * q + 2 * i] = x0;
            x[h][b][8 * q + 2 * i + 1] = x1;
            mx = fmaxf(mx, fmaxf(fabsf(x[h][b][8 * q + 2 * i]), fabsf(x[h][b][8 * q + 2 * i + 1])));
          }
        }
    mx = max_xor32(max_xor16(mx));
    qs = 0.5f * sum_xor32(sum_xor16(sum));
    const uint32_t eb = max((__float_as_uint(mx) >> 23) & 0xffu, 8u);
    const float scale = __uint_as_float((eb - 7) << 23);  // row max / scale in [128, 256)
    sb = static_cast<int>(eb) - 7;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = x[h][b][2 * ((4 * d + e) & 7) + ((4 * d + e) >> 3)];
#pragma unroll
          for (int term = 0; term < kQTerms; ++term)
            qb[h][term][4 * b + d] = static_cast<int>(fp8x4_scaled_take(v, scale));
        }
  }

  // ---- spreading: K images of chunk c (wavefront w takes token tile w; below 4 also the scales
  // and zeros of 64 token-vectors) and V images of chunk c (dims 32 w .. 32 w + 31). The raw
  // codes are read ahead of the scores and written as images behind them.
  uint32_t raw_k[2][2], raw_sz = 0;
  i32x2 raw_v[2];
  auto read_k = [&](int c) {
    const uint8_t* st = lds.raw[c % kRawStagesC] + kSkew;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t* kp =
          reinterpret_cast<const uint32_t*>(st + kRec * (16 * wave + n) + 8 * g + 32 * h);
      raw_k[h][0] = kp[0];
      raw_k[h][1] = kp[1];
    }
    raw_sz = *reinterpret_cast<const uint32_t*>(st + kRec * (64 * (wave & 1) + lane) + 64 +
                                                ((wave >> 1) & 1) * kVector);
  };
  auto write_k = [&](int c) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      lds.k[c & 1][h][wave][lane] =
          u32x4{(uint32_t)even_codes(raw_k[h][0]), (uint32_t)odd_codes(raw_k[h][0]),
                (uint32_t)even_codes(raw_k[h][1]), (uint32_t)odd_codes(raw_k[h][1])};
  };
  auto write_scales = [&](int c) {
    if (wave < 4) {
      // Tokens outside the split (or of an unmapped block) get a zero scale and zero: their slots
      // may hold NaN patterns; their scores are masked.
      const int tok = 64 * (wave & 1) + lane, pos = ((first + c) << 7) + tok;
      const bool in = pos >= p_lo && pos < p_hi && (mapped >> (2 * (c & 7) + (wave & 1)) & 1);
      const uint32_t sz = in ? raw_sz : 0u;
      if (wave < 2) {
        lds.ks[c & 3][tok] = h16lo(sz) * fq;
        lds.kz[c & 3][tok] = h16hi(sz) * fq;
      } else {
        lds.vsz[c & 3][tok] = sz;
      }
    }
  };
  // PV k-slot of FP8 lane group G, byte e: token 16 (e / 4) + 4 G + e % 4 (the score layout).
  // FP4 lane group g, nibble i holds that of G = 2 (g & 1) + i / 16, e = 16 (g >> 1) + i % 16:
  // lane n supplies the row of nibble n to the first read and of nibble 16 + n to the second.
  auto read_v = [&](int c) {
    const uint8_t* vp = lds.raw[c % kRawStagesC] + kSkew + kVector +
                        kRec * (64 * (g >> 1) + 16 * (n >> 2) + 8 * (g & 1) + (n & 3)) + 8 * wave;
    raw_v[0] = __builtin_amdgcn_ds_read_tr4_b64_v2i32((lds_i32x2_ptr_t)vp);
    raw_v[1] = __builtin_amdgcn_ds_read_tr4_b64_v2i32((lds_i32x2_ptr_t)(vp + 4 * kRec));
  };
  auto write_v = [&](int c) {
    lds.v[c & 1][2 * wave][lane] =
        u32x4{(uint32_t)even_codes(raw_v[0][0]), (uint32_t)even_codes(raw_v[0][1]),
              (uint32_t)even_codes(raw_v[1][0]), (uint32_t)even_codes(raw_v[1][1])};
    lds.v[c & 1][2 * wave + 1][lane] =
        u32x4{(uint32_t)odd_codes(raw_v[0][0]), (uint32_t)odd_codes(raw_v[0][1]),
              (uint32_t)odd_codes(raw_v[1][0]), (uint32_t)odd_codes(raw_v[1][1])};
  };

  float m = -INFINITY, psum = 0.f, zsum = 0.f;
  f32x4 o[16];  // o[2 c + par]: rows 4 g + v, dim 32 c + 2 n + par (units of code / 2)
#pragma unroll
  for (int j = 0; j < 16; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 acc[8];  // scores of the wavefront's chunk: token 16 tt + 4 g + v of row n
  i32x8 ph, pl;  // its P operands
  int sp = 0;    // and their E8M0 scale

  // Q K of chunk c: operand i is token tile i % 8 of the 128-dim half i / 8.
  auto qk_step = [&](int c, int i) {
    const int h = i >> 3, tt = i & 7;
    const u32x4 f = lds.k[c & 1][h][tt][lane];
#pragma unroll
    for (int term = 0; term < kQTerms; ++term)
      acc[tt] = mfma_qk_scaled(f, qb[h][term],
                               h == 0 && term == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[tt], sb);
  };
  auto pv_step = [&](int c, int j) {
    const u32x4 f = lds.v[c & 1][j][lane];
    const i32x8 v4 = {(int)f[0], (int)f[1], (int)f[2], (int)f[3], 0, 0, 0, 0};
    o[j] = mfma_pv(ph, v4, o[j], sp);
    o[j] = mfma_pv(pl, v4, o[j], sp);
  };
  // Score of chunk c's token 16 tt + 4 g + v of row n, minus `sub` (log2 units).
  float x[8][4];
  auto score_step = [&](int c, int tt, float sub) {
    const f32x4 ks = *reinterpret_cast<const f32x4*>(&lds.ks[c & 3][16 * tt + 4 * g]);
    const f32x4 kz = *reinterpret_cast<const f32x4*>(&lds.kz[c & 3][16 * tt + 4 * g]);
#pragma unroll
    for (int v = 0; v < 4; ++v) x[tt][v] = fmaf(ks[v], acc[tt][v], fmaf(kz[v], qs, -sub));
  };
  // Masks the scores of tokens outside the split or in an unmapped block; the lane's largest.
  auto visible_max = [&](int c) {
    const int t0 = (first + c) << 7;
    const bool ok0 = mapped >> 2 * (c & 7) & 1, ok1 = mapped >> 2 * (c & 7) & 2;
    if (!(ok0 && ok1 && t0 >= p_lo && t0 + kTokC <= p_hi)) {
#pragma unroll
      for (int tt = 0; tt < 8; ++tt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const bool in = (tt < 4 ? ok0 : ok1) &&
                          static_cast<uint32_t>(t0 + 16 * tt + 4 * g + v - p_lo) <
                              static_cast<uint32_t>(p_hi - p_lo);
          x[tt][v] = in ? x[tt][v] : -INFINITY;
        }
    }
    float mx = max3(x[0][0], x[0][1], x[0][2]);
#pragma unroll
    for (int e = 3; e < 31; e += 2) mx = max3(mx, x[e >> 2][e & 3], x[(e + 1) >> 2][(e + 1) & 3]);
    return fmaxf(mx, x[7][3]);
  };
  // P operands of the scores in x: p s_v as FP8 hi + lo with one E8M0 scale per row and 64-token
  // half (the MFMA reads the scale of bytes 0..15 from lane groups 0 and 1, of bytes 16..31 from
  // 2 and 3).
  auto probabilities = [&](int c, int half) {
    float amax = 0.f;
#pragma unroll
    for (int tt = 4 * half; tt < 4 * half + 4; ++tt) {
      const u32x4 sz = *reinterpret_cast<const u32x4*>(&lds.vsz[c & 3][16 * tt + 4 * g]);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float p = __builtin_amdgcn_exp2f(x[tt][v]);
        psum += p;
        zsum = fmaf(p, h16hi(sz[v]), zsum);
        x[tt][v] = fmaf(p, h16lo(sz[v]), 0.0f);
      }
      amax = max3(amax, x[tt][0], x[tt][1]);
      amax = max3(amax, x[tt][2], x[tt][3]);
    }
    amax = max_xor32(max_xor16(amax));
    const uint32_t eb = max(__float_as_uint(amax) >> 23, 7u);
    const float scale = __uint_as_float((eb - 6) << 23);  // row max / scale in [64, 128)
#pragma unroll
    for (int tt = 4 * half; tt < 4 * half + 4; ++tt) {
      ph[tt] = static_cast<int>(fp8x4_scaled_take(x[tt], scale));
      pl[tt] = static_cast<int>(fp8x4_scaled_last(x[tt], scale));
    }
    return static_cast<int>(eb) - 6;
  };

  // ---- chunk loop, one barrier per period. Period c issues the MFMAs of P V (chunk c - 1) among
  // the score arithmetic of chunk c, and those of Q K (chunk c + 1) among its probabilities, so
  // that each wavefront feeds the matrix and the vector pipe at once: 3.8 us per chunk (one phase
  // after the other 4.9 us; the two wavefronts of a SIMD taking turns 4.2 us, the waits of the
  // softmax half are then exposed). It reads the images V c - 1, K c + 1 and the scales of c, writes
  // V c and K c + 2 with its scales (each wavefront an eighth), and starts the copies of chunk
  // c + 3 (into the stage of chunk c - 1): a wavefront waits for its own copies of chunk c + 3
  // before the barrier that ends the period.
  if (nchunk > 0) {
    OSCAR_WAIT_VM(0);
    barrier_lds();
    read_k(0);
    write_k(0);
    write_scales(0);
    read_k(1);  // past the last chunk: another stage's bytes, to images nobody reads
    write_k(1);
    write_scales(1);
    barrier_lds();
    if (3 < nchunk) issue(3, records(3));
    if (live) {
#pragma unroll
      for (int i = 0; i < 16; ++i) qk_step(0, i);
    }
    barrier_lds();  // K images 0 are read: period 0 writes K images 2 in their place
    uint2 next = records(4);  // offsets of the chunk copied next, read a period ahead
    auto end_period = [&](int c) {
      write_scales(c + 2);
      if (c + 3 < nchunk) OSCAR_WAIT_VM(0);
      barrier_lds();
      if (c + 4 < nchunk) {
        issue(c + 4, next);
        next = records(c + 5);
      }
    };
    auto spread = [&](int c) {
      read_k(c + 2);  // past the last chunk: as above
      read_v(c);
      write_k(c + 2);
      write_v(c);
    };
    if (!live) {  // rows past the request's last: this wavefront only copies and spreads
#pragma unroll 1
      for (int c = 0; c < nchunk; ++c) {
        spread(c);
        end_period(c);
      }
      return;
    }
    int c = 0;
#pragma unroll 1
    for (;;) {
      // Lazy running max (history.hip): the row max moves only when a score passes it by 2^8,
      // outside the chunk loop, so that the loop holds one copy of the accumulators.
      const float base = m == -INFINITY ? 0.f : m;  // -inf: no visible token so far
#pragma unroll
      for (int tt = 0; tt < 8; ++tt) score_step(c, tt, base);
      const float mn = fmaxf(m, base + max_xor32(max_xor16(visible_max(c))));
      const float alpha = mn == -INFINITY ? 1.0f : exp2f(m - mn);
      m = mn;
      psum *= alpha;
      zsum *= alpha;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float av = __shfl(alpha, 4 * g + v, kWave);  // accumulator row 4 g + v
#pragma unroll
        for (int j = 0; j < 16; ++j) o[j][v] *= av;
      }
#pragma unroll
      for (int tt = 0; tt < 8; ++tt) score_step(c, tt, m == -INFINITY ? 0.f : m);
      visible_max(c);
      bool need = false;
#pragma unroll 1
      do {
        __builtin_amdgcn_sched_barrier(0);
        spread(c);
        const int sa0 = probabilities(c, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) qk_step(c + 1, i);  // past the last chunk: unused
        const int sa1 = probabilities(c, 1);
        sp = g < 2 ? sa0 : sa1;
        // Reads 4 operands ahead, one MFMA per 9 vector instructions.
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
        }
        // Computed here: the compiler would sink results into the next period.
        asm volatile("" : "+v"(ph), "+v"(pl), "+v"(psum), "+v"(zsum), "+v"(sp));
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) asm volatile("" : "+v"(acc[tt]));
        __builtin_amdgcn_sched_barrier(0);
        end_period(c);
        const float sub = m == -INFINITY ? 0.f : m;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 16; ++j) pv_step(c, j);
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) score_step(c + 1, tt, sub);  // as above
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) asm volatile("" : "+v"(o[j]));
#pragma unroll
        for (int tt = 0; tt < 8; ++tt)
          asm volatile("" : "+v"(x[tt][0]), "+v"(x[tt][1]), "+v"(x[tt][2]), "+v"(x[tt][3]));
        __builtin_amdgcn_sched_barrier(0);
        ++c;
        const float mx = visible_max(c);
        need = __any(mx > (m == -INFINITY ? -3.0e38f : kTheta));
      } while (c < nchunk && !need);
      if (c >= nchunk) break;
    }
  }
  if (!live) return;

  // ---- normalized rows and LSE (rows of an empty range: zeros and -inf).
  psum = sum_xor32(sum_xor16(psum));
  zsum = sum_xor32(sum_xor16(zsum));
  const float inv_n = 1.0f / fmaxf(psum, 1.0e-30f);
  // Row indices are formed again (from mbcnt lanes), so that none stays live across the loop.
  const int el = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
  const int en = el & 15, eg = el >> 4;
  const int out_row = row_base + 16 * wave + en;
  const int oqi = static_cast<int>(fastdiv(static_cast<uint32_t>(out_row), a.g_div));
  const int64_t otok = static_cast<int64_t>(t.qstart) + oqi;
  const bool ok = out_row < rows && otok >= 0 && otok < a.n;
  const int64_t my_out = ok ? (otok * a.hq + head * a.g + (out_row - oqi * a.g)) : -1;
  if (ok && eg == 0)
    a.lse[my_out * a.splits + split] = psum > 0.f ? (m + log2f(psum)) * kLn2 : -INFINITY;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int src = 4 * eg + v;
    const float inv = __shfl(inv_n, src, kWave), zs = __shfl(zsum, src, kWave);
    const int64_t row = static_cast<int64_t>(__shfl(static_cast<int>(my_out), src, kWave));
    if (row < 0) continue;
    float* out = a.partials + (row * a.splits + split) * kHeadDim + 2 * en;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      *reinterpret_cast<float2*>(out + 32 * c) =
          make_float2((2.0f * o[2 * c][v] + zs) * inv, (2.0f * o[2 * c + 1][v] + zs) * inv);
  }
}

}  // namespace

// Grid x of the launch: at least the tiles find_tile can find. A request of q query tokens holds
// ceil(q / qt) task rows of qt g <= 32 rows, x rows in all, and starts ceil(x / 128) <= (x + 127) /
// 128 tiles; over at most `reqs` requests of n tokens and `programs` task rows, x sums to at most
// the smaller of programs qt g and (n + (qt - 1) reqs) g. A task row starts at most one tile.
int64_t history_chunk_tiles(int64_t n, int64_t max_reqs, int64_t programs, int64_t qt, int64_t g) {
  const int64_t reqs = n < max_reqs ? n : max_reqs;
  const int64_t by_tasks = programs * qt * g, by_tokens = (n + (qt - 1) * reqs) * g;
  const int64_t rows = by_tasks < by_tokens ? by_tasks : by_tokens;
  const int64_t tiles = (rows + (kRowsC - 1) * reqs) / kRowsC;
  return tiles < programs ? tiles : programs;
}

}  // namespace oscar

extern "C" int64_t oscar_history_chunk_tiles(int64_t n, int64_t max_reqs, int64_t programs,
                                             int32_t query_tile, int32_t group) {
  return oscar::history_chunk_tiles(n, max_reqs, programs, query_tile, group);
}

extern "C" int oscar_history_chunk(
    const void* query, int64_t q_s0, int64_t q_s1, int64_t q_s2, const void* history,
    int64_t history_bytes, const int32_t* qstarts, const int32_t* seq_lens,
    const int32_t* block_tables, int64_t table_stride, int64_t table_columns,
    const int32_t* counts, const int32_t* tasks, const int32_t* task_count, int64_t n, int64_t hq,
    int64_t programs, int64_t max_reqs, int32_t splits, int32_t block_n, int32_t query_tile,
    float scale, const oscar_layout* layout, float* partials, float* lse, void* stream) {
  using namespace oscar;
  if (max_reqs < 1 || max_reqs > 0x7fffffffll) return OSCAR_E_SHAPE;
  AttnArgs a;
  int64_t qrows = 0;
  const int st = make_attn_args(query, q_s0, q_s1, q_s2, nullptr, 0, 0, 1, nullptr, 0, 0, 1,
                                history, history_bytes, nullptr, 0, qstarts, seq_lens,
                                block_tables, table_stride, table_columns, counts, tasks,
                                task_count, n, hq, programs, splits, block_n, query_tile, 0, scale,
                                0, 0, layout, partials, lse, &a, &qrows);
  if (st != OSCAR_OK || n == 0) return st;
  const int64_t tiles = history_chunk_tiles(n, max_reqs, programs, query_tile, a.g);
  if (tiles * a.L.kv_heads > 0x7fffffffll / splits) return OSCAR_E_SHAPE;
  const dim3 grid(static_cast<unsigned>(tiles * a.L.kv_heads * splits));
  hipLaunchKernelGGL(history_chunk_kernel, grid, dim3(kThreadsC), 0, as_stream(stream), a,
                     static_cast<int32_t>(programs));
  return static_cast<int>(hipGetLastError());
}
