// The projections of small waves: 16-row output tiles on
// v_mfma_i32_16x16x32_i8, the same arithmetic as kernels_gemm.hip (one exact
// integer dot per 32-block, ((float)dot * d_w) * d_x, terms added in block
// order), so the results are bit-identical to it.
//
// A small wave is bound by latency, not by arithmetic: 32 rows x 768 columns
// are 24 tiles of 32 x 32, so 24 waves on 1,024 SIMDs, each walking 24
// dependent block steps behind loads that miss the L2 (a kernel boundary
// empties it). These kernels shorten that chain three ways: 16 x 16 tiles
// have a quarter of the scaling work per lane and block (13 VALU operations,
// not 49) and four times the waves; the blocks of a tile are split over the
// waves of a workgroup, each of which asks for all its blocks' operands at
// once (one round trip to memory, not one per three blocks); and the waves
// only form the terms ((float)dot * d_w) * d_x, which go to LDS, from where
// one thread per output adds them in block order: the order of the sum, and
// so its bits, do not depend on the split.
#pragma once

#include "eg2_device.hpp"

namespace eg2 {

typedef int intx4 __attribute__((ext_vector_type(4)));

constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23
constexpr int kMagicBits = 0x4B400000;
constexpr int kTile = 1024;            // bytes of one 32 x 32 int8 operand block

// Operands of one 16 x 16 tile and 32-block: lane 16 g + r holds row r's
// values 8 g .. 8 g + 7 of both matrices, the weight scale of column r and
// the activation scale of row 4 g + lane % 4.
struct NarrowFrag {
  uint64_t a, b;
  float dx, dw;
};

// Byte offset of the lane's 8 values inside the 16-row half of a 1 KB block.
__device__ __forceinline__ uint32_t narrow_lane_offset() {
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  return (uint32_t)((g >> 1) * 512 + r * 16 + (g & 1) * 8);
}

// One wave's 16 weight rows 16 tc .. (rows past m repeat the last one's
// scale; the row tiles are padded to 32).
struct NarrowWeights {
  __amdgpu_buffer_rsrc_t rb, rw;
  uint32_t lane_off, woff, ldw4;
  int nb;

  __device__ __forceinline__ NarrowWeights(const int8_t* wq, const float* wd, int ldw, int m, int tc, int blocks)
      : lane_off(narrow_lane_offset()), ldw4(4u * (uint32_t)ldw), nb(blocks) {
    const uint32_t skip = (tc & 1) * 256;
    rb = buffer_rsrc(wq + (size_t)(tc >> 1) * nb * kTile + skip, (uint32_t)nb * kTile - skip);
    rw = buffer_rsrc(wd, 4u * ((uint32_t)(nb - 1) * (uint32_t)ldw + (uint32_t)m));
    woff = 4u * (uint32_t)min(16 * tc + (int)(threadIdx.x & 15), m - 1);
  }
  __device__ __forceinline__ void load(NarrowFrag& f, int kb) const {  // kb uniform; past the end: the last block
    kb = min(kb, nb - 1);
    f.b = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(rb, lane_off, kb * kTile, 0));
    f.dw = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, woff, (uint32_t)kb * ldw4, 0));
  }
};

// One wave's 16 activation rows 16 tr .., as NarrowWeights (n rows).
struct NarrowRows {
  __amdgpu_buffer_rsrc_t ra, rx;
  uint32_t lane_off, xoff, ldx4;
  int nb;

  __device__ __forceinline__ NarrowRows(const int8_t* xq, const float* xd, int ldx, int n, int tr, int blocks)
      : lane_off(narrow_lane_offset()), ldx4(4u * (uint32_t)ldx), nb(blocks) {
    const int lane = threadIdx.x & 63;
    const uint32_t skip = (tr & 1) * 256;
    ra = buffer_rsrc(xq + (size_t)(tr >> 1) * nb * kTile + skip, (uint32_t)nb * kTile - skip);
    rx = buffer_rsrc(xd, 4u * ((uint32_t)(nb - 1) * (uint32_t)ldx + (uint32_t)n));
    xoff = 4u * (uint32_t)min(16 * tr + 4 * (lane >> 4) + (lane & 3), n - 1);
  }
  __device__ __forceinline__ void load(NarrowFrag& f, int kb) const {
    kb = min(kb, nb - 1);
    f.a = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(ra, lane_off, kb * kTile, 0));
    f.dx = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, xoff, (uint32_t)kb * ldx4, 0));
  }
};

// Lane V of each aligned quad, on every lane of the quad.
template <int V>
__device__ __forceinline__ float quad_bcast(float x) {
  return dpp<V * 0x55>(x);
}

// The block's terms (dot * d_w) * d_x: element v is row 4 g + v, column r.
__device__ __forceinline__ float4 narrow_terms(const NarrowFrag& f) {
  const intx4 magic = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
  const intx4 dot =
      __builtin_amdgcn_mfma_i32_16x16x32_i8((long)f.a, (long)f.b, magic, 0, 0, 0);
  const float bias = f.dw * -kMagic;
  float t[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) t[v] = __builtin_fmaf(__int_as_float(dot[v]), f.dw, bias);
  return make_float4(t[0] * quad_bcast<0>(f.dx), t[1] * quad_bcast<1>(f.dx), t[2] * quad_bcast<2>(f.dx),
                     t[3] * quad_bcast<3>(f.dx));
}

// One chunk of a tile's blocks c0 .. c0 + SPLIT * NBW - 1: wave `ks` of SPLIT
// forms the terms of blocks c0 + ks * NBW + i from its fragments into
// terms[block of the chunk][lane] (blocks past the end repeat the last one
// and are not added).
template <int NBW>
__device__ __forceinline__ void narrow_put(const NarrowFrag (&f)[NBW], int ks, float4* terms) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < NBW; ++i) terms[(ks * NBW + i) * 64 + lane] = narrow_terms(f[i]);
}

// The ordered sum of output `o` (lane o / 4, element o % 4) over the chunk's
// first cnt blocks.
template <int CHUNK>
__device__ __forceinline__ float narrow_sum(const float* terms, int o, int cnt, float sum) {
  if (cnt == CHUNK) {
    float v[CHUNK];
#pragma unroll
    for (int b = 0; b < CHUNK; ++b) v[b] = terms[b * 256 + o];
#pragma unroll
    for (int b = 0; b < CHUNK; ++b) sum = sum + v[b];
  } else {
    for (int b = 0; b < cnt; ++b) sum = sum + terms[b * 256 + o];
  }
  return sum;
}

// y[n][m], one 16 x 16 tile per workgroup of 4 waves, NBW blocks per wave
// and chunk (4 NBW blocks: 24, 36 or 48).
template <int NBW>
__global__ void __launch_bounds__(256)
gemm_q8_narrow_kernel(const int8_t* __restrict__ xq, const float* __restrict__ xd, int ldx,
                      const int8_t* __restrict__ wq, const float* __restrict__ wd, int ldw, float* __restrict__ y,
                      int n, int m, int nb, int ldy) {
  constexpr int kChunk = 4 * NBW;
  __shared__ __align__(16) float4 terms[kChunk * 64];
  __builtin_amdgcn_s_setprio(1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tc = (int)blockIdx.x, tr = (int)blockIdx.y;
  const NarrowWeights weights(wq, wd, ldw, m, tc, nb);
  const NarrowRows rows(xq, xd, ldx, n, tr, nb);
  const int o = (int)threadIdx.x;
  float sum = 0.0f;
  for (int c0 = 0; c0 < nb; c0 += kChunk) {
    NarrowFrag f[NBW];
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
      weights.load(f[i], c0 + w * NBW + i);
      rows.load(f[i], c0 + w * NBW + i);
    }
    if (c0) __syncthreads();  // the previous chunk's terms are no longer read
    narrow_put<NBW>(f, w, terms);
    __syncthreads();
    sum = narrow_sum<kChunk>(reinterpret_cast<const float*>(terms), o, min(kChunk, nb - c0), sum);
  }
  const int row = 16 * tr + 4 * (o >> 6) + (o & 3), col = 16 * tc + ((o >> 2) & 15);
  if (row < n && col < m) y[(size_t)row * ldy + col] = sum;
}

// The GeGLU of one R x 32 tile, gu = [row][gate 0..31 | up 0..31], by the
// first 32 R threads, and its Q8_0: block tc of rows t0 .. t0 + R - 1.
constexpr int kGuPitch = 65;
__device__ __forceinline__ void narrow_geglu_store(const float* gu, int t0, int tc, int n, int nbf,
                                                   int8_t* __restrict__ gq, float* __restrict__ gd, int ldg) {
  const int row = (int)threadIdx.x >> 5, col = (int)threadIdx.x & 31, t = t0 + row;
  const Q8Lane q = q8_quantize_lane(gelu_mul(gu[row * kGuPitch + col], gu[row * kGuPitch + 32 + col]));
  if (t >= n) return;
  gq[q8_tile_offset(t, 32 * tc + col, nbf)] = (int8_t)q.q;
  if (col == 0) gd[(size_t)tc * ldg + t] = q.d;
}

// gate|up + GeGLU + Q8_0: a workgroup of 8 waves computes 16 rows x one
// 32-wide gate group and its up group (the weight rows are interleaved in
// 32-row groups, so these are 64 consecutive weight rows: four 16 x 16
// tiles, each split over two waves), then one thread per GeGLU value
// evaluates it exactly (gelu_mul: with a value per thread the certified
// approximation of the wide kernel would only lengthen the chain) and
// quantizes its block over the 32 lanes that hold it. A wave asks for its
// kNarrowGegluBlocks blocks of a chunk at once; the terms pass through LDS
// half a chunk at a time (48 KB: three workgroups per CU).
constexpr int kNarrowGegluBlocks = 12;  // blocks per wave and chunk

__global__ void __launch_bounds__(512)
gemm_q8_geglu_narrow_kernel(const int8_t* __restrict__ xq, const float* __restrict__ xd, int ldx,
                            const int8_t* __restrict__ wq, const float* __restrict__ wd, int ldw, int n, int ff,
                            int nb, int8_t* __restrict__ gq, float* __restrict__ gd, int ldg) {
  constexpr int NBW = kNarrowGegluBlocks, kHalf = NBW;
  __shared__ __align__(16) float4 terms[4][kHalf * 64];  // [tile][block of the half chunk][lane]
  __shared__ float gu[16 * kGuPitch];                    // [row][gate 0..31 | up 0..31]
  __builtin_amdgcn_s_setprio(1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ti = w & 3, ks = w >> 2;
  const int tc = (int)blockIdx.x, tr = (int)blockIdx.y;
  const NarrowWeights weights(wq, wd, ldw, 2 * ff, 4 * tc + ti, nb);
  const NarrowRows rows(xq, xd, ldx, n, tr, nb);
  const int so = (int)threadIdx.x >> 8, o = (int)threadIdx.x & 255;  // this thread adds output o of tiles so, so + 2
  float gate = 0.0f, up = 0.0f;
  for (int c0 = 0; c0 < nb; c0 += 2 * kHalf) {
    NarrowFrag f[2][NBW / 2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < NBW / 2; ++i) {
        weights.load(f[p][i], c0 + p * kHalf + ks * (NBW / 2) + i);
        rows.load(f[p][i], c0 + p * kHalf + ks * (NBW / 2) + i);
      }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (c0 + p) __syncthreads();  // the previous half's terms are no longer read
      narrow_put<NBW / 2>(f[p], ks, terms[ti]);
      __syncthreads();
      const int cnt = min(kHalf, nb - c0 - p * kHalf);
      gate = narrow_sum<kHalf>(reinterpret_cast<const float*>(terms[so]), o, cnt, gate);
      up = narrow_sum<kHalf>(reinterpret_cast<const float*>(terms[so + 2]), o, cnt, up);
    }
  }
  float* mine = gu + (4 * (o >> 6) + (o & 3)) * kGuPitch + 16 * so + ((o >> 2) & 15);
  mine[0] = gate;
  mine[32] = up;
  __syncthreads();
  narrow_geglu_store(gu, 16 * tr, tc, n, ff / kQK, gq, gd, ldg);
}

}  // namespace eg2
