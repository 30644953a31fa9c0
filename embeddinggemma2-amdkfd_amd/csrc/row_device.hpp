// Device helpers on 768-wide token rows, shared by the row kernels
// (kernels_rows.hip) and the fused kernels of short waves (short_wave.hpp).
#pragma once

#include "eg2_device.hpp"

namespace eg2 {

constexpr int kBlocks = kEmbd / kQK;                   // 24 blocks per row
constexpr int kVec = kEmbd / 256;                      // float4 per lane per row

// ---------------------------------------------------------------- 768-wide rows
// A 768-float token row is held one float4 per lane per 256 columns (lane L
// has elements 4L..4L+3 + 256r, r = 0..2). Its SSE2 sum of squares
// (kernels.c:82-94) needs chain c = the sequential sum over t of
// row[8t + c]^2: the row's squares (each rounded, as the reference's) are
// staged transposed in LDS, tr[c][t] = row[8t + c]^2, by every lane of the
// row, so the lane that runs chain c reads its 96 squares with 24
// ds_read_b128 and only adds. The 104-float pitch
// puts the eight chain rows 40 banks apart (conflict-free reads) and the
// two lanes of a pair 32 banks apart (conflict-free transposed writes).
constexpr int kChain = kEmbd / 8;  // 96
constexpr int kTPitch = kChain + 8;
typedef float TRow[kTPitch];

__device__ __forceinline__ void stage_squares(TRow* tr, const float4 (&v)[kVec]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < kVec; ++r) {
    const float c4[4] = {v[r].x * v[r].x, v[r].y * v[r].y, v[r].z * v[r].z, v[r].w * v[r].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = 4 * (lane + 64 * r) + k;
      tr[e & 7][e >> 3] = c4[k];
    }
  }
}

// Chain c of the SSE2 sum of squares from the staged squares, read in three
// groups of eight float4, each group's reads issued before its additions.
// The rolled outer loop keeps 32 registers of reads in flight, not 96: the
// residual kernel's register count (and so how many of its waves fit beside
// other streams' kernels on a CU) is set by this chain.
__device__ __forceinline__ float squares_chain(const TRow* tr, int c) {
  float s = 0.0f;
#pragma unroll 1
  for (int g = 0; g < kChain / 32; ++g) {
    float4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const float4*>(&tr[c][32 * g + 4 * j]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s = s + v[j].x;
      s = s + v[j].y;
      s = s + v[j].z;
      s = s + v[j].w;
    }
  }
  return s;
}

// DPP moves beside dpp (eg2_device.hpp), which writes every lane: `dpp_into`
// writes only the lanes of the 4-lane banks in BANKS and keeps `old`
// elsewhere. Choosing lanes by bank mask,
// not by a select on the lane index, keeps every source lane active: the
// compiler may turn a select of two DPP results into an EXEC-masked branch,
// and a DPP move reads 0 from lanes that EXEC disables.
template <int CTRL, int BANKS>
__device__ __forceinline__ float dpp_into(float old, float src) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old),
                                                               __builtin_bit_cast(int, src), CTRL, 0xf, BANKS,
                                                               false));
}
constexpr int kQuad0000 = 0x00, kQuad1111 = 0x55, kQuad2222 = 0xAA, kQuad3333 = 0xFF;
constexpr int kRowShl4 = 0x104, kRowShr4 = 0x114;  // lane i reads lane i + 4 / i - 4
constexpr int kBanks02 = 0x5, kBanks13 = 0xA;      // lanes 0-3 and 8-11 / 4-7 and 12-15 of a row

// The value of lane i ^ 4: the other 4-lane half of each aligned 8-lane group.
__device__ __forceinline__ float other_quad(float x) {
  return dpp_into<kRowShr4, kBanks13>(dpp_into<kRowShl4, kBanks02>(x, x), x);
}

// sse2_combine with DPP instead of LDS shuffles: lanes 8g..8g+7 hold chains
// 0..7 (chains 0-3 are the first 4-wide accumulator, 4-7 the second);
// v[j] = acc0[j] + acc1[j], total (v0 + v2) + (v1 + v3) (kernels.c:35-39),
// returned to every lane of the group.
__device__ __forceinline__ float sse2_combine_dpp(float s) {
  const float v = s + dpp<kRowShl4>(s);  // lanes 0-3 of the group: v[0..3]
  const float total = (dpp<kQuad0000>(v) + dpp<kQuad2222>(v)) + (dpp<kQuad1111>(v) + dpp<kQuad3333>(v));
  return dpp_into<kRowShr4, kBanks13>(total, total);  // lanes 4-7 take lanes 0-3's
}

// Maximum over each aligned group of 8 lanes, on every lane of the group.
__device__ __forceinline__ float group8_max(float m) {
  m = fmaxf(m, dpp<kQuad1032>(m));
  m = fmaxf(m, dpp<kQuad2301>(m));
  return fmaxf(m, other_quad(m));
}

// quants.c:97-177 (scalar path) on the row held as float4 per lane: block b
// (32 values) is lanes 8(b % 8)..+7 of register r = b / 8, four values per
// lane; the block maximum is combined over those 8 lanes. A group's three
// blocks get their scale computed once each: lane 8i + r takes block
// (r, i)'s maximum, computes d = amax / 127, 1/d and the fp16 scale, and
// stores the latter's float value at d[b * ld]; the group's lanes take the
// three 1/d back by swizzle broadcasts (an LDS-unit permute, no VALU work).
// Each lane stores its 4 int8 values (contiguous in the row-tile layout)
// for row t of q. v[r] must already hold the values to quantize; all 64
// lanes must be active.
template <int R>
__device__ __forceinline__ float group8_lane(float x) {
  // ds_swizzle bitmask mode within 32 lanes: source lane (lane & 0x18) | R
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), 0x18 | (R << 5)));
}
__device__ __forceinline__ void quantize_row_lanes(const float4 (&v)[kVec], int t, int8_t* __restrict__ q,
                                                   float* __restrict__ d, int ld) {
  static_assert(kVec == 3, "three blocks per 8-lane group");
  const int lane = threadIdx.x & 63, r8 = lane & 7;
  float amax[kVec];
#pragma unroll
  for (int r = 0; r < kVec; ++r)
    amax[r] = group8_max(fmaxf(fmaxf(fabsf(v[r].x), fabsf(v[r].y)), fmaxf(fabsf(v[r].z), fabsf(v[r].w))));
  const float am = r8 == 0 ? amax[0] : (r8 == 1 ? amax[1] : amax[2]);  // lanes 8i + 3 .. 7: block 2 again, unused
  const float dd = div127(am);
  const float id_own = am != 0.0f ? 1.0f / dd : 0.0f;  // 0 for an all-zero block, whose values quantize to 0
  if (r8 < kVec) d[(size_t)((lane >> 3) + 8 * r8) * ld] = fp16_bits_to_fp32(fp32_to_fp16_bits(dd));
  const float ids[kVec] = {group8_lane<0>(id_own), group8_lane<1>(id_own), group8_lane<2>(id_own)};
#pragma unroll
  for (int r = 0; r < kVec; ++r) {
    const float id = ids[r];
    const int e = 4 * (lane + 64 * r);
    const int32_t q0 = q8_value(v[r].x, id), q1 = q8_value(v[r].y, id), q2 = q8_value(v[r].z, id),
                  q3 = q8_value(v[r].w, id);
    *reinterpret_cast<uint32_t*>(q + q8_tile_offset(t, e, kBlocks)) = pack_i8x4(q0, q1, q2, q3);
  }
}

}  // namespace eg2
