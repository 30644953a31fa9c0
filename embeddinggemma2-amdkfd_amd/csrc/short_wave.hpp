// The layer of a short wave (at most kShortRows rows, a multiple of 16) in
// five kernels instead of nine:
//   residual_qkv      residual + norms + Q8_0, then the Q|K|V projection
//   short_attention   QK-norm / RoPE, scores, softmax, context, Q8_0
//   (O projection     gemm_q8_narrow_kernel)
//   residual_geglu    residual + norms + Q8_0, then gate|up + GeGLU + Q8_0
//   (down projection  gemm_q8_narrow_kernel)
// A short wave is a chain of latencies: each kernel boundary costs about 1.5
// us and empties the L2, and a 16-row residual kernel or a 3-head attention
// occupies a handful of CUs. So every workgroup of a projection repeats its
// rows' residual update and norms itself (the chip is idle anyway) while its
// weights are on their way, and one workgroup per (head, few query rows)
// takes attention from the raw projection to the quantized context with all
// keys and values in LDS. The same operations in the same order as the
// kernels they replace: the same bits. Through 24
// layers, host work included: 11 tokens 1,119 -> 650 us, 45 tokens 1,142 -> 787
// (30 tokens: 745). At 64 rows the form ends: the residual kernels'
// 320 and 288 workgroups are more than the 256 CUs, and raw rows, rotated keys and
// values no longer fit one CU's LDS at once (with the values written over the raw
// rows behind one more barrier: 1,120-1,140 us, the separate kernels 1,140-1,150).
#pragma once

#include "eg2_device.hpp"
#include "gemm_narrow.hpp"
#include "row_device.hpp"

namespace eg2 {

// Orders a wave's LDS writes before its reads of them by other lanes (the
// wave's LDS accesses execute in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// A residual + projection workgroup: 12 waves, ROWS (4 or 8) rows. Thread
// (wave w, lane) holds columns 256 (w % 3) + 4 lane .. + 3 of row w / 3 (and
// w / 3 + 4), so a norm weight vector is read once per workgroup, not once per
// row. What a CU has to read and then computes on elementwise bounds these
// kernels (with 16 rows and a row per wave, 96 KB of rows and 96 KB of norm
// weights took 5,700 cycles of 18,700 at 64 B per cycle), hence few rows per
// workgroup: 4 in a 16-row wave, 8 in a longer one, 144 to 240 workgroups
// (one 11-token query with 8: 735 us, with 4: 696; 30 tokens with 8: 767, with
// 4 for Q|K|V: 788); the MFMA tile's other rows repeat them and are not stored.
inline int short_tile(int rows) { return rows <= 16 ? 4 : 8; }
constexpr int kShortWaves = 12, kShortThreads = 64 * kShortWaves;
constexpr int kShortStride = 8 * kTPitch + 4;  // staged squares per row: the rows read at once on distinct banks

// The LDS of such a workgroup: the rows' staged squares, then the terms of
// TILES 16-column tiles, their 24 blocks split over 12 / TILES waves; the
// quantized rows [block][2][ROWS][16] and their scales [block][ROWS].
template <int TILES, int ROWS>
struct ShortLds {
  static constexpr int kSplit = kShortWaves / TILES, kPer = kBlocks / kSplit;
  static_assert(kSplit * kPer == kBlocks, "24 blocks split evenly");
  union alignas(16) {
    float squares[ROWS * kShortStride];
    float4 terms[TILES][kBlocks * 4 * ROWS];  // lanes below 4 ROWS: the rows
  };
  alignas(16) int8_t aq[kBlocks * 32 * ROWS];
  float dxs[kBlocks * ROWS];
  float inv[2][ROWS];
};

// residual_norm_quant_kernel's work on the workgroup's rows, then the
// projection onto weight columns 16 (TILES blockIdx.x + tile): x_out = x +
// rms(h) * post_w (stored by the workgroups with blockIdx.x = 0), Q8_0 of
// rms(x_out) * next_w, times W^T. Returns, for thread i < 16 ROWS TILES, output
// o = i % (16 ROWS) of tile i / (16 ROWS) (row 4 (o / 64) + o % 4, column (o /
// 4) % 16).
template <int TILES, int ROWS>
__device__ __forceinline__ float residual_project(ShortLds<TILES, ROWS>& lds, const float* __restrict__ x,
                                                  const float* __restrict__ h, const float* __restrict__ post_w,
                                                  const float* __restrict__ next_w, float eps,
                                                  const int8_t* __restrict__ wq, const float* __restrict__ wd, int ldw,
                                                  int m, float* __restrict__ x_out) {
  constexpr int kPer = ShortLds<TILES, ROWS>::kPer, kEach = ROWS / 4;  // rows per thread
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = w / 3, part = w % 3, e = 4 * (lane + 64 * part);
  float4 hv[kEach], xv[kEach];
#pragma unroll
  for (int i = 0; i < kEach; ++i)
    hv[i] = *reinterpret_cast<const float4*>(h + (size_t)(ROWS * blockIdx.y + row + 4 * i) * kEmbd + e);
#pragma unroll
  for (int i = 0; i < kEach; ++i)
    xv[i] = *reinterpret_cast<const float4*>(x + (size_t)(ROWS * blockIdx.y + row + 4 * i) * kEmbd + e);
  const float4 pw = *reinterpret_cast<const float4*>(post_w + e), nw = *reinterpret_cast<const float4*>(next_w + e);
  // The weights of this wave's blocks, on their way during the rows' work.
  const int ti = w % TILES, ks = w / TILES;
  const NarrowWeights weights(wq, wd, ldw, m, TILES * (int)blockIdx.x + ti, kBlocks);
  NarrowFrag f[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) weights.load(f[i], ks * kPer + i);

  // Squares of the thread's values into the transposed rows; wave 0 runs the
  // 64 chains of the 8 rows and leaves each row's inverse in inv.
  auto inverses = [&](const float4 (&v)[kEach], float* inv) {
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      TRow* tr = reinterpret_cast<TRow*>(lds.squares + (row + 4 * i) * kShortStride);
      const float c4[4] = {v[i].x * v[i].x, v[i].y * v[i].y, v[i].z * v[i].z, v[i].w * v[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) tr[(e + k) & 7][(e + k) >> 3] = c4[k];
    }
    __syncthreads();
    if (w == 0) {  // with 4 rows, every chain twice
      const TRow* rows = reinterpret_cast<const TRow*>(lds.squares + (lane >> 3) % ROWS * kShortStride);
      const float r = rms_inverse(sse2_combine_dpp(squares_chain(rows, lane & 7)), kEmbd, eps);
      if ((lane & 7) == 0) inv[(lane >> 3) % ROWS] = r;
    }
    __syncthreads();
  };
  inverses(hv, lds.inv[0]);
#pragma unroll
  for (int i = 0; i < kEach; ++i) {  // kernels.c:163-188
    const float inv_h = lds.inv[0][row + 4 * i];
    const float a0 = hv[i].x * inv_h, a1 = hv[i].y * inv_h, a2 = hv[i].z * inv_h, a3 = hv[i].w * inv_h;
    const float b0 = a0 * pw.x, b1 = a1 * pw.y, b2 = a2 * pw.z, b3 = a3 * pw.w;
    xv[i] = make_float4(xv[i].x + b0, xv[i].y + b1, xv[i].z + b2, xv[i].w + b3);
    if (blockIdx.x == 0)
      *reinterpret_cast<float4*>(x_out + (size_t)(ROWS * blockIdx.y + row + 4 * i) * kEmbd + e) = xv[i];
  }
  inverses(xv, lds.inv[1]);
#pragma unroll
  for (int i = 0; i < kEach; ++i) {  // kernels.c:139-151, the block over 8 lanes
    const float inv = lds.inv[1][row + 4 * i];
    const float p0 = xv[i].x * nw.x, p1 = xv[i].y * nw.y, p2 = xv[i].z * nw.z, p3 = xv[i].w * nw.w;
    const float v0 = p0 * inv, v1 = p1 * inv, v2 = p2 * inv, v3 = p3 * inv;
    const float amax = group8_max(fmaxf(fmaxf(fabsf(v0), fabsf(v1)), fmaxf(fabsf(v2), fabsf(v3))));
    const float d = div127(amax);
    const float id = amax != 0.0f ? 1.0f / d : 0.0f;
    const int kb = e / kQK, r = row + 4 * i;
    *reinterpret_cast<uint32_t*>(lds.aq + ((kb * 2 + ((e >> 4) & 1)) * ROWS + r) * 16 + (e & 15)) =
        pack_i8x4(q8_value(v0, id), q8_value(v1, id), q8_value(v2, id), q8_value(v3, id));
    if ((lane & 7) == 0) lds.dxs[kb * ROWS + r] = fp16_bits_to_fp32(fp32_to_fp16_bits(d));
  }
  __syncthreads();
  // Lane 16 g + r: row r % ROWS, values 8 g .. 8 g + 7 of the block.
  const int g = lane >> 4, aoff = ((g >> 1) * ROWS + (lane & (ROWS - 1))) * 16 + (g & 1) * 8;
  const int xoff = (4 * g + (lane & 3)) & (ROWS - 1);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int kb = ks * kPer + i;
    f[i].a = *reinterpret_cast<const uint64_t*>(lds.aq + kb * 32 * ROWS + aoff);
    f[i].dx = lds.dxs[kb * ROWS + xoff];
    const float4 t = narrow_terms(f[i]);
    if (lane < 4 * ROWS) lds.terms[ti][kb * 4 * ROWS + lane] = t;
  }
  __syncthreads();
  const int i = (int)threadIdx.x;
  float sum = 0.0f;
  if (i < 16 * ROWS * TILES) {
    const float* t = reinterpret_cast<const float*>(lds.terms[i / (16 * ROWS)]) + i % (16 * ROWS);
    float v[kBlocks];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) v[b] = t[16 * ROWS * b];
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) sum = sum + v[b];
  }
  return sum;
}

// The raw Q|K|V rows (no QK-norm / RoPE) of x_out. Grid (kQKVCols / 32, rows /
// ROWS). x_out must not be x: every workgroup reads x.
template <int ROWS>
__global__ void __launch_bounds__(kShortThreads)
residual_qkv_kernel(const float* __restrict__ x, const float* __restrict__ h, const float* __restrict__ post_w,
                    const float* __restrict__ next_w, float eps, const int8_t* __restrict__ wq,
                    const float* __restrict__ wd, int ldw, float* __restrict__ x_out, float* __restrict__ out) {
  __shared__ ShortLds<2, ROWS> lds;
  const float sum = residual_project<2, ROWS>(lds, x, h, post_w, next_w, eps, wq, wd, ldw, kQKVCols, x_out);
  const int i = (int)threadIdx.x, o = i % (16 * ROWS);
  if (i < 32 * ROWS)
    out[(size_t)(ROWS * blockIdx.y + 4 * (o >> 6) + (o & 3)) * kQKVCols + 32 * blockIdx.x + 16 * (i / (16 * ROWS)) +
        ((o >> 2) & 15)] = sum;
}

// The same rows, then gate|up (interleaved 32-row groups), GeGLU and Q8_0
// into gq / gd [kFF / 32][rows]. Grid (kFF / 32, rows / ROWS).
template <int ROWS>
__global__ void __launch_bounds__(kShortThreads)
residual_geglu_kernel(const float* __restrict__ x, const float* __restrict__ h, const float* __restrict__ post_w,
                      const float* __restrict__ next_w, float eps, const int8_t* __restrict__ wq,
                      const float* __restrict__ wd, int ldw, float* __restrict__ x_out, int8_t* __restrict__ gq,
                      float* __restrict__ gd, int rows) {
  __shared__ ShortLds<4, ROWS> lds;
  __shared__ float gu[ROWS * kGuPitch];
  const float sum = residual_project<4, ROWS>(lds, x, h, post_w, next_w, eps, wq, wd, ldw, 2 * kFF, x_out);
  const int i = (int)threadIdx.x, o = i % (16 * ROWS);
  if (i < 64 * ROWS) gu[(4 * (o >> 6) + (o & 3)) * kGuPitch + 16 * (i / (16 * ROWS)) + ((o >> 2) & 15)] = sum;
  __syncthreads();
  if (i < 32 * ROWS)
    narrow_geglu_store(gu, ROWS * (int)blockIdx.y, (int)blockIdx.x, rows, kFF / kQK, gq, gd, rows);
}

// ------------------------------------------------------------ attention

// A workgroup of 16 waves takes one head and kShortQueries query rows of a
// wave of at most kShortRows packed rows from the raw projection rows
// [q0 q1 q2 | k | v] to the quantized context: all waves normalise and rotate
// the k rows (KG each), the first kShortQueries waves also a query row each,
// which they then carry through. (With 16 query rows per workgroup the LDS
// reads of 16 score and context waves on one CU bound the kernel.) Normalised and
// rotated q and k rows are kept chain-major in LDS, [row][chain d % 4][step
// d / 4], so that a lane of chain c reads four steps with one 16-byte read
// (pitches of 68 and 272 floats: a 16-lane read group covers 4 rows x 4 chains
// on distinct banks). Scores: lane 4 k + c runs chain c of keys k + 16 i
// (kernels.c:289-294), the chains combined as (s0 + s2) + (s1 + s3); then the
// row's maximum, expf, the sum in key order and the context in key order,
// lanes over dimensions, over the row's own keys only. One form per KG groups of
// 16 rows: every row count known when compiled, no branch between the loads, and a
// 16-row wave has 16 rows' LDS (one form with the second 16 rows behind
// a branch: an 11-token query 677 us, now 650; 30 tokens 752 and 745).
constexpr int kShortRows = 48;
constexpr int kShortQueries = 4;
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kShortPitch = kHeadDim + 8;  // floats per raw row
constexpr int kChainPitch = kHeadDim / 4 + 4, kChainRow = 4 * kChainPitch;

template <int KG>  // groups of 16 key rows
struct ShortAttentionLds {
  alignas(16) float raw[kShortQueries + 16 * KG][kShortPitch];  // q rows, then k rows
  alignas(16) float q[kShortQueries][kChainRow];
  alignas(16) float k[16 * KG][kChainRow];
  alignas(16) float v[16 * KG][kHeadDim];
  alignas(16) float p[kShortQueries][16 * KG];
  uint64_t exp_tab[32];
};

template <int KG>
__global__ void __launch_bounds__(1024)
short_attention_kernel(const float* __restrict__ qkv, const uint4* __restrict__ tok, const float* __restrict__ q_w,
                       const float* __restrict__ k_w, const float* __restrict__ rope, const int32_t* __restrict__ pos,
                       float eps, int window, int rows, int8_t* __restrict__ cq, float* __restrict__ cd) {
  __shared__ ShortAttentionLds<KG> lds;
  constexpr int half = kHeadDim / 2;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hd = (int)blockIdx.x, qw = w % kShortQueries, t = kShortQueries * (int)blockIdx.y + qw;
  const bool query = w < kShortQueries;  // this wave carries query row t
  // This wave's key rows: w + 16 i.
  int pk[KG];
#pragma unroll
  for (int i = 0; i < KG; ++i) pk[i] = pos[w + 16 * i];
  const int pq = pos[t];
  const uint4 meta = tok[t];
  const float* kr = qkv + (size_t)w * kQKVCols + kHeads * kHeadDim + 4 * lane;
  const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const float4 q4 = query ? *reinterpret_cast<const float4*>(qkv + (size_t)t * kQKVCols + hd * kHeadDim + 4 * lane) : zero;
  floatx4 k4[KG], v4[KG];  // no HIP vector structs: an array of those is kept in LDS
#pragma unroll
  for (int i = 0; i < KG; ++i) k4[i] = *reinterpret_cast<const floatx4*>(kr + (size_t)16 * i * kQKVCols);
  // A row's norm weights and cos/sin for dimensions lane + 64 j.
  struct Row4 {
    float v[4];
  };
  auto row4 = [&](const float* p) { return Row4{{p[lane], p[lane + 64], p[lane + 128], p[lane + 192]}}; };
  const Row4 kw = row4(k_w), qw4 = query ? row4(q_w) : kw;
  Row4 kc[KG];
#pragma unroll
  for (int i = 0; i < KG; ++i) kc[i] = row4(rope + (size_t)pk[i] * kHeadDim);
  const Row4 cq4 = query ? row4(rope + (size_t)pq * kHeadDim) : kc[0];
#pragma unroll
  for (int i = 0; i < KG; ++i) v4[i] = *reinterpret_cast<const floatx4*>(kr + (size_t)16 * i * kQKVCols + kHeadDim);
  if (threadIdx.x < 32) lds.exp_tab[threadIdx.x] = libm::kExp2Tab.t[threadIdx.x];
  float* rawq = lds.raw[qw];
  auto rawk = [&](int i) { return lds.raw[kShortQueries + w + 16 * i]; };
  if (query) *reinterpret_cast<float4*>(rawq + 4 * lane) = q4;
#pragma unroll
  for (int i = 0; i < KG; ++i) *reinterpret_cast<floatx4*>(rawk(i) + 4 * lane) = k4[i];
  wave_lds_fence();
  // kernels.c:233-264: lanes 8 i .. 8 i + 7 run the chains of key row w + 16 i,
  // the next eight those of the query row.
  const float* chain_row = rawk(0);
#pragma unroll
  for (int i = 1; i < KG; ++i) chain_row = (lane >> 3) == i ? rawk(i) : chain_row;
  if (query && (lane >> 3) == KG) chain_row = rawq;
  const float own = rms_inverse(sse2_combine_dpp(sse2_chain<kHeadDim>(chain_row, lane & 7)), kHeadDim, eps);
  auto norm_rope = [&](const float* raw, float* dst, const Row4& g, const Row4& cs, int from, bool q) {
    const float inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(own), from));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int dd = lane + 64 * j;
      const float c = cs.v[j], s = cs.v[2 + j];
      const float x0 = raw[dd] * g.v[j] * inv;
      const float x1 = raw[dd + half] * g.v[2 + j] * inv;
      const float a0 = x0 * c, a1 = x1 * s;
      const float b0 = x0 * s, b1 = x1 * c;
      float lo = a0 - a1, hi = b0 + b1;
      if (q) {
        lo = lo * 0.0625f;
        hi = hi * 0.0625f;
      }
      dst[(dd & 3) * kChainPitch + (dd >> 2)] = lo;
      dst[(dd & 3) * kChainPitch + ((dd + half) >> 2)] = hi;
    }
  };
#pragma unroll
  for (int i = 0; i < KG; ++i) norm_rope(rawk(i), lds.k[w + 16 * i], kw, kc[i], 8 * i, false);
  if (query) norm_rope(rawq, lds.q[qw], qw4, cq4, 8 * KG, true);
#pragma unroll
  for (int i = 0; i < KG; ++i) *reinterpret_cast<floatx4*>(lds.v[w + 16 * i] + 4 * lane) = v4[i];
  __syncthreads();
  if (!query) return;
  // Scores of row t.
  const int key = lane >> 2, c = lane & 3;
  float s[KG];
  const float4* qp = reinterpret_cast<const float4*>(lds.q[qw] + c * kChainPitch);
#pragma unroll
  for (int i = 0; i < KG; ++i) {
    const float4* kp = reinterpret_cast<const float4*>(lds.k[key + 16 * i] + c * kChainPitch);
    float a = 0.0f;
#pragma unroll
    for (int st = 0; st < kHeadDim / 16; ++st) {
      const float4 qv = qp[st], kv = kp[st];
      const float p0 = qv.x * kv.x, p1 = qv.y * kv.y, p2 = qv.z * kv.z, p3 = qv.w * kv.w;
      a = a + p0;
      a = a + p1;
      a = a + p2;
      a = a + p3;
    }
    a = a + dpp<kQuad2301>(a);     // s0 + s2, s1 + s3
    s[i] = a + dpp<kQuad1032>(a);  // their sum
  }
  uint32_t first, last;
  key_range((uint32_t)t, meta.x, meta.y, window, first, last);
  auto in = [&](int i) { return (uint32_t)(key + 16 * i) >= first && (uint32_t)(key + 16 * i) < last; };
  float m = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < KG; ++i) m = fmaxf(m, in(i) ? s[i] : -__builtin_inff());
  m = fmaxf(m, dpp<kRowHalfMirror>(m));          // the other quad of each 8 lanes
  m = rows4_max(fmaxf(m, dpp<kRowMirror>(m)));  // the other 8 of the row, then the four rows
#pragma unroll
  for (int i = 0; i < KG; ++i) {
    const float e = libm::expf_tab(s[i] - m, lds.exp_tab);
    if (c == 0) lds.p[qw][key + 16 * i] = in(i) ? e : 0.0f;
  }
  wave_lds_fence();
  // The sum in key order; +0 outside the row's keys changes no sum.
  float sum = 0.0f;
  const float4* pp = reinterpret_cast<const float4*>(lds.p[qw]);
#pragma unroll
  for (int i = 0; i < 4 * KG; ++i) {
    const float4 p4 = pp[i];
    sum = sum + p4.x;
    sum = sum + p4.y;
    sum = sum + p4.z;
    sum = sum + p4.w;
  }
  const float inv = 1.0f / sum;
  float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const int kfirst = __builtin_amdgcn_readfirstlane((int)first), klast = __builtin_amdgcn_readfirstlane((int)last);
#pragma unroll 4
  for (int k = kfirst; k < klast; ++k) {
    const float wk = lds.p[qw][k] * inv;
    const float4 vv = *reinterpret_cast<const float4*>(lds.v[k] + 4 * lane);
    const float p0 = wk * vv.x, p1 = wk * vv.y, p2 = wk * vv.z, p3 = wk * vv.w;
    acc = make_float4(acc.x + p0, acc.y + p1, acc.z + p2, acc.w + p3);
  }
  // Q8_0 (quants.c:97-177): 8 lanes hold a block.
  const float amax = group8_max(fmaxf(fmaxf(fabsf(acc.x), fabsf(acc.y)), fmaxf(fabsf(acc.z), fabsf(acc.w))));
  const float d = div127(amax);
  const float id = amax != 0.0f ? 1.0f / d : 0.0f;
  const unsigned e = (unsigned)(hd * kHeadDim + 4 * lane);
  if ((lane & 7) == 0) cd[(size_t)(e / kQK) * rows + t] = fp16_bits_to_fp32(fp32_to_fp16_bits(d));
  *reinterpret_cast<uint32_t*>(cq + q8_tile_offset(t, e, kBlocks)) =
      pack_i8x4(q8_value(acc.x, id), q8_value(acc.y, id), q8_value(acc.z, id), q8_value(acc.w, id));
}

}  // namespace eg2
