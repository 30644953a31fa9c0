// The operator set of the reference's by-name kernel interface (the
// kernels/abi.h records, the kernel names and launch geometry of
// kernels/eg2.c) on this library's own gfx950 designs.
//
// Each kernel takes its record by value, so its kernarg segment has the
// record's layout and a code object built from this file can be dispatched
// by symbol name ("eg2_mm64x64.kd", ...) with the same records, grids and
// workgroup sizes the reference executor uses (src/gemma2_kfd.cpp:160-165,
// 248-336) and its operator test uses (tests/kernels.cpp:36-137). The
// results meet that test's tolerances (2e-5 absolute against exact
// references; 2e-6 between a fused operator and its unfused sequence); they
// are not the reference kernels' bits.
//
// Designs:
//  - projections (eg2_mm*): bf16 MFMA on exact bf16 parts of the operands
//    (F32 weights: fp32 MFMA), each wave over every fourth 32-deep step of the
//    tile; and a general form for any k and alignment: fp32 MFMA
//    (v_mfma_f32_16x16x4f32) on LDS-staged 32-deep K slices of the activations
//    and of the weights decoded to fp32 (F32, F16, BF16 or Q8_0 blocks over
//    the flattened matrix), zero-padded past k. There the MFMA's k index is a
//    permutation of the slice chosen so that each lane reads contiguous
//    float4s of its row: lane group g (lanes 16g .. 16g+15) feeds slice
//    elements g*KW/4 .. (g+1)*KW/4 - 1, one per MFMA. The 16x16 tile splits
//    the slice over its four waves and adds their partial tiles at the end;
//    the wider tiles give each wave its own 16x16 blocks.
//  - attention: keys in chunks of 64, one per lane: every lane computes its
//    key's whole dot product against q (broadcast from LDS), so a chunk
//    costs one wave max and one wave sum instead of one reduction per key;
//    then the softmax weights of the chunk (exp through the host libm's
//    expf restated in eg2_libm.hpp, rescaled by the running maximum between
//    chunks) go through LDS to the context, where lanes own dimensions.
//    eg2_op_launch of the whole grid of 512 tokens or more takes tiles of 16
//    tokens x one head on fp32 MFMA instead (attention_tile_kernel).
//  - row operators (norm, norm_residual, norm_rope): one wave per row with
//    the row held in registers as float4s (a single read of the row), the
//    sum of squares reduced by DPP within 16-lane rows and a 4-way add
//    across them, correctly rounded division and square root. The fused
//    forms share the helpers of the unfused ones, so fused = unfused.
//  - element-wise operators (saxpy, gathers, rope, element, pool): one
//    element per work-item, as the launch contract gives; GELU is the
//    tanh form with the host libm's tanhf restated (eg2_device.hpp).
//
// Launch contract (grid counted in workgroups, as the reference counts it):
//   eg2_saxpy, eg2_gather, eg2_rope, eg2_element, eg2_pool, eg2_gather768:
//       1-D, any workgroup size, one element per work-item
//   eg2_mm       256 work-items, grid (ceil(m/16), ceil(n/16))  16x16 tile
//   eg2_mm64     256 work-items, grid (ceil(m/64), ceil(n/16))  16x64 tile
//   eg2_mm64x64, eg2_mmstep8
//                256 work-items, grid (ceil(m/64), ceil(n/64))  64x64 tile
//   eg2_norm, eg2_norm_residual, eg2_norm_rope
//                one 64-wide wave per row, grid = rows
//   eg2_attention256, eg2_attention512
//                one wave per (token, query head), grid = 4n
//   eg2_attention256x3 (the 3 query / 1 KV head, d 256 variant)
//                one wave per (token, query head), grid = 3n
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "abi.h"
#include "eg2_device.hpp"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned flat_index() { return threadIdx.x + blockIdx.x * blockDim.x; }

// Element i of a GGML-typed weight matrix (type 0 F32, 1 F16, 30 BF16,
// otherwise Q8_0: 34-byte blocks of a little-endian fp16 scale and 32 int8
// values, running over the flattened matrix), as fp32. The Q8_0 value
// fp16(d) * q is exact in fp32.
__device__ __forceinline__ float weight_at(const void* w, size_t i, unsigned type) {
  switch (type) {
    case 0:
      return static_cast<const float*>(w)[i];
    case 1:
      return eg2::fp16_bits_to_fp32(static_cast<const uint16_t*>(w)[i]);
    case 30:
      return __uint_as_float((uint32_t)static_cast<const uint16_t*>(w)[i] << 16);
    default: {
      const unsigned char* blk = static_cast<const unsigned char*>(w) + (i >> 5) * 34;
      const float d = eg2::fp16_bits_to_fp32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
      return d * (float)reinterpret_cast<const signed char*>(blk + 2)[i & 31];
    }
  }
}

// ------------------------------------------------------------ projections

constexpr int kSlice = 32;           // K values per LDS stage
constexpr int kPitch = kSlice + 4;   // floats per staged row

// The general form: any k, any alignment, and the sums that overflow or hold
// infinities or NaN (mm_tile). out[n x m] = x[n x k] . W[m x k]^T for a
// TH x TW tile per 256-thread workgroup (4 waves), fp32 MFMA on LDS-staged
// slices of the activations and the decoded weights. With `redo` (a bit per
// output, [row][column / 16]) only those outputs are stored.
template <int TH, int TW>
__device__ __forceinline__ void mm_general(const EgMM& p, float* xs, float* ws, floatx4* part,
                                           const uint16_t (*redo)[TW / 16]) {
  static_assert((TH == 16 && (TW == 16 || TW == 64)) || (TH == 64 && TW == 64), "tile shapes of the contract");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r16 = lane & 15;
  const unsigned row0 = blockIdx.y * TH, col0 = blockIdx.x * TW;

  // Wave geometry: row blocks (16 rows) and column blocks (16 columns) it
  // owns, and the part of each slice it reads.
  constexpr bool kSplit = TH == 16 && TW == 16;  // the four waves split each slice
  constexpr int RB = TH == 64 ? 2 : 1, CB = TH == 64 ? 2 : 1;
  constexpr int KW = kSplit ? kSlice / 4 : kSlice;  // slice values per wave
  constexpr int PER = KW / 4;                       // values per lane group = MFMAs per slice
  const int rbase = TH == 64 ? 32 * (wave >> 1) : 0;
  const int cbase = TH == 64 ? 32 * (wave & 1) : (TW == 64 ? 16 * wave : 0);
  const int kbase = kSplit ? KW * wave : 0;

  floatx4 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

  for (unsigned base = 0; base < p.k; base += kSlice) {
    for (int idx = tid; idx < TH * kSlice; idx += 256) {
      const int rr = idx / kSlice, kk = idx % kSlice;
      const unsigned row = row0 + rr, kx = base + kk;
      xs[rr * kPitch + kk] = row < p.n && kx < p.k ? p.x[(size_t)row * p.k + kx] : 0.0f;
    }
    for (int idx = tid; idx < TW * kSlice; idx += 256) {
      const int cc = idx / kSlice, kk = idx % kSlice;
      const unsigned col = col0 + cc, kx = base + kk;
      ws[cc * kPitch + kk] = col < p.m && kx < p.k ? weight_at(p.weight, (size_t)col * p.k + kx, p.type) : 0.0f;
    }
    __syncthreads();
    float a[RB][PER], b[CB][PER];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < PER; ++e) a[i][e] = xs[(rbase + 16 * i + r16) * kPitch + kbase + g * PER + e];
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int e = 0; e < PER; ++e) b[j][e] = ws[(cbase + 16 * j + r16) * kPitch + kbase + g * PER + e];
#pragma unroll
    for (int e = 0; e < PER; ++e)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    __syncthreads();
  }

  if constexpr (kSplit) {
    // Waves 1-3 hand their partial tiles to wave 0, which adds them in order.
    if (wave > 0) part[(wave - 1) * 64 + lane] = acc[0][0];
    __syncthreads();
    if (wave > 0) return;
    acc[0][0] = ((acc[0][0] + part[lane]) + part[64 + lane]) + part[128 + lane];
  }
  // MFMA 16x16 output: lane holds rows 4g .. 4g + 3 of column r16.
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int tr = rbase + 16 * i + 4 * g + v, tc = cbase / 16 + j;
        const unsigned row = row0 + tr, col = col0 + 16 * tc + r16;
        if (row < p.n && col < p.m && (!redo || (redo[tr][tc] >> r16) & 1))
          p.out[(size_t)row * p.m + col] = acc[i][j][v];
      }
}

// The usual form, k a multiple of 32 and operands aligned (mm_direct_fits),
// on bf16 MFMA (v_mfma_f32_16x16x32_bf16) with fp32 sums. The activations are
// split exactly into three bf16 parts (8 + 8 + 8 of their 24 significant
// bits, by truncation; a row too small for that takes the general form); Q8_0
// values are whole numbers of at most 8 bits and BF16 weights are bf16, so
// three products per weight are exact, and a Q8_0 block's scale is one fma on
// its 32-value dot; F16 weights split exactly into two parts (six products);
// F32 weights stay on fp32 MFMA
// (v_mfma_f32_16x16x4f32). A product of 32 values takes 52 matrix cycles per
// 16 x 16 tile instead of 263, and fewer roundings: the error against a
// float64 product (2-norm) at 640 x 512 x 2048 is 7.0e-8 for Q8_0, 1.2e-7
// BF16, 1.5e-7 F16, 2.1e-7 F32, where the general form has 4.0e-7.
//
// What bounded the general form was its staging: scalar loads, a decode with
// a branch and a 64-bit address per weight, two barriers per 32 values. On one
// card inside a graph, the general form alone / this kernel, us:
//                               F32           F16           BF16          Q8_0
//   eg2_mm      40 x 512 x 512   14.4 / 3.9    14.6 / 3.9    14.3 / 3.5    16.4 / 4.1
//   eg2_mm64    40 x 768 x 1152  87.1 / 8.9    53.8 / 7.1    53.3 / 5.4    63.2 / 6.9
//   eg2_mm64x64 640 x 512 x 2048 63.4 / 27.1   62.5 / 15.1   63.3 / 12.3   68.6 / 14.5
//               2048 x 768 x 1152 158 / 62.6   151 / 32.4    152 / 24.5    158 / 28.6
// Bound by the latency of staging and splitting, F32 weights by the fp32 MFMAs
// (263 matrix cycles a step and 16 x 16 tile, 74 KB of LDS: two workgroups of 64
// x 64 per CU). Over one step (k 32) the general form is as fast: 512 x 32 x 512
// 3.1 / 3.3, 3.2 / 3.3, 3.2 / 3.2, 3.2 / 3.4, 64 x 32 x 64 in 64 x 64 tiles 5.0 / 5.7,
// 5.2 / 5.1, 5.2 / 4.6, 5.4 / 5.1, but less exact.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
struct Bf16Parts {
  uintx4 part[3];
};
// The high halves of two floats as a bf16 pair (a in the low half).
__device__ __forceinline__ uint32_t high_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302);
}
__device__ __forceinline__ float truncated(float a) { return __uint_as_float(__float_as_uint(a) & 0xffff0000u); }
// Eight floats as three bf16 parts each: a == part 0 + part 1 + part 2.
template <int PARTS>
__device__ __forceinline__ Bf16Parts split_bf16(const float (&v)[8]) {
  Bf16Parts s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
      s.part[q][i] = high_halves(a, b);
      if (q + 1 < PARTS) {
        a = a - truncated(a);
        b = b - truncated(b);
      }
    }
  }
  return s;
}
// bf16 holds whole steps of 2^-133, so a value below 2^-110 loses bits of its
// last part, at most 2^-133 in all: nothing beside a value of 2^-100 or more,
// but all of the precision in a row that has none. (One maximum per two values
// in the loop; noting the lost bits themselves costs as many instructions, but
// F16 weights lost 10% by the registers' lifetimes.)
constexpr float kSplitsFrom = 0x1p-100f;
__device__ __forceinline__ floatx4 mfma_bf16(uintx4 a, uintx4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

// One wave's operands of a step on their way through its own LDS area. A wave
// reads global memory along the rows (8 lanes a 128-byte line of x: reading
// the MFMA's order directly, 16 rows to a 16-lane group, a wave touches 64
// lines per instruction and the step took 3,100-5,200 cycles of loads alone)
// and picks the fragments up in the MFMA's order: lane 16 g + r holds row (or
// column) r, values 8 g .. 8 g + 7 of the step. A wave's LDS accesses execute
// in order and no other wave uses its area, so there is no barrier. Pitches
// keep the 16 rows of a fragment read on distinct banks.
constexpr int kStepPitch = 36;  // floats per staged fp32 row

// fp32 rows: x of every type, F32 weights.
template <int BLOCKS>  // 16-row blocks
struct StepRows {
  floatx4 v[2 * BLOCKS];
  __device__ __forceinline__ void load(const float* m, unsigned k, unsigned row0, unsigned rows, unsigned base) {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 2 * BLOCKS; ++i)
      v[i] = *reinterpret_cast<const floatx4*>(m + (size_t)min(row0 + 8 * i + (lane >> 3), rows - 1) * k + base +
                                              4 * (lane & 7));
  }
  __device__ __forceinline__ void put(float* lds) const {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < 2 * BLOCKS; ++i)
      *reinterpret_cast<floatx4*>(lds + (8 * i + (lane >> 3)) * kStepPitch + 4 * (lane & 7)) = v[i];
  }
};
__device__ __forceinline__ void step_row(const float* lds, int block, float (&f)[8]) {
  const int lane = threadIdx.x & 63;
  const floatx4* p = reinterpret_cast<const floatx4*>(lds + (16 * block + (lane & 15)) * kStepPitch + 8 * (lane >> 4));
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const floatx4 v = p[i];
    f[4 * i] = v[0], f[4 * i + 1] = v[1], f[4 * i + 2] = v[2], f[4 * i + 3] = v[3];
  }
}

// Weight columns by type: load() along the rows, put() into LDS, get() the
// lane's fragment of a 16-column block.
template <unsigned TYPE, int BLOCKS>
struct StepWeights {  // F16, BF16: 64 bytes a column and step
  static constexpr int kPitch = 80;
  uintx4 v[BLOCKS];
  __device__ __forceinline__ void load(const void* w, unsigned k, unsigned col0, unsigned m, unsigned base) {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j)
      v[j] = *reinterpret_cast<const uintx4*>(static_cast<const uint16_t*>(w) +
                                             (size_t)min(col0 + 16 * j + (lane >> 2), m - 1) * k + base + 8 * (lane & 3));
  }
  __device__ __forceinline__ void put(float* lds) const {
    const unsigned lane = threadIdx.x & 63;
    unsigned char* b = reinterpret_cast<unsigned char*>(lds);
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j)
      *reinterpret_cast<uintx4*>(b + (16 * j + (lane >> 2)) * kPitch + 16 * (lane & 3)) = v[j];
  }
  static __device__ __forceinline__ uintx4 get(const float* lds, int block) {
    const int lane = threadIdx.x & 63;
    return *reinterpret_cast<const uintx4*>(reinterpret_cast<const unsigned char*>(lds) +
                                           (16 * block + (lane & 15)) * kPitch + 16 * (lane >> 4));
  }
};
template <int BLOCKS>
struct StepWeights<8, BLOCKS> {  // Q8_0: a 34-byte block a column and step, at even addresses
  static constexpr int kPitch = 40;
  static constexpr int kScales = 16 * BLOCKS * kPitch / 4;  // floats before the scales
  uint32_t v[BLOCKS][3];
  uint32_t shift[BLOCKS];
  __device__ __forceinline__ void load(const void* w, unsigned k, unsigned col0, unsigned m, unsigned base) {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      // The lane's 8 values (and, in lane 0 of the four, the scale) lie in
      // three aligned words from 8 q bytes into the block rounded down to 4,
      // the first of which may begin two bytes before the block or the last
      // end two after it: where those are not the matrix's, kQ8Edge reads.
      // (Unaligned 8-byte loads cost 0.9 us a step.)
      const unsigned char* blk = static_cast<const unsigned char*>(w) +
                                 ((size_t)min(col0 + 16 * j + (lane >> 2), m - 1) * (k / 32) + base / 32) * 34 +
                                 8 * (lane & 3);
      shift[j] = (uint32_t)(reinterpret_cast<uintptr_t>(blk) & 2);
      const uint32_t* p = reinterpret_cast<const uint32_t*>(blk - shift[j]);
#pragma unroll
      for (int i = 0; i < 3; ++i) v[j][i] = p[i];
    }
  }
  __device__ __forceinline__ void put(float* lds) const {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const bool odd = shift[j] != 0;  // the values start 4 bytes in, not 2
      const uint32_t lo = odd ? v[j][1] : __builtin_amdgcn_alignbyte(v[j][1], v[j][0], 2);
      const uint32_t hi = odd ? v[j][2] : __builtin_amdgcn_alignbyte(v[j][2], v[j][1], 2);
      put_block(lds, 16 * j + (lane >> 2), lo, hi, odd ? v[j][0] >> 16 : v[j][0] & 0xffffu);
    }
  }
  // This lane's 8 values of its column's block; of lane 0 of the four, the scale.
  static __device__ __forceinline__ void put_block(float* lds, unsigned col, uint32_t lo, uint32_t hi, uint32_t scale) {
    const unsigned q = threadIdx.x & 3;
    *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(lds) + col * kPitch + 8 * q) = make_uint2(lo, hi);
    if (q == 0) lds[kScales + col] = eg2::fp16_bits_to_fp32(scale);
  }
  static __device__ __forceinline__ uintx4 get(const float* lds, int block, float& scale) {  // as bf16
    const int lane = threadIdx.x & 63;
    const uint2 q = *reinterpret_cast<const uint2*>(reinterpret_cast<const unsigned char*>(lds) +
                                                    (16 * block + (lane & 15)) * kPitch + 8 * (lane >> 4));
    scale = lds[kScales + 16 * block + (lane & 15)];
    float f[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = (float)(int8_t)(q.x >> (8 * e));
      f[4 + e] = (float)(int8_t)(q.y >> (8 * e));
    }
    return split_bf16<1>(f).part[0];
  }
};
// Q8_0 in a tile that holds the matrix's first block at 2 mod 4, or its last one
// at 0 mod 4: nothing outside a block is read. Lane q of a block's four reads two
// aligned words and one 16-bit value: at 0 mod 4 the words hold two bytes more
// before the lane's 8 values (lane 0: the scale) and the 16 bits their last two;
// at 2 mod 4 the words are the values and the 16 bits the scale. (For every tile
// this takes 3-20% longer: a load more per block.)
constexpr unsigned kQ8Edge = 9;
constexpr unsigned q8_words_at(unsigned q, bool odd) { return 8 * q + (odd ? 2 : 0); }
constexpr unsigned q8_half_at(unsigned q, bool odd) { return odd ? 0 : 8 * q + 8; }
static_assert(q8_words_at(3, true) + 8 == 34 && q8_words_at(3, false) + 8 == 32 && q8_half_at(3, false) + 2 == 34,
              "the last lane's reads end with the block");
template <int BLOCKS>
struct StepWeights<kQ8Edge, BLOCKS> {
  uint32_t v[BLOCKS][2];
  uint32_t half[BLOCKS];
  bool odd[BLOCKS];
  __device__ __forceinline__ void load(const void* w, unsigned k, unsigned col0, unsigned m, unsigned base) {
    const unsigned lane = threadIdx.x & 63, q = lane & 3;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const unsigned char* blk = static_cast<const unsigned char*>(w) +
                                 ((size_t)min(col0 + 16 * j + (lane >> 2), m - 1) * (k / 32) + base / 32) * 34;
      odd[j] = (reinterpret_cast<uintptr_t>(blk) & 2) != 0;
      const uint32_t* p = reinterpret_cast<const uint32_t*>(blk + q8_words_at(q, odd[j]));
      v[j][0] = p[0];
      v[j][1] = p[1];
      half[j] = *reinterpret_cast<const uint16_t*>(blk + q8_half_at(q, odd[j]));
    }
  }
  __device__ __forceinline__ void put(float* lds) const {
    const unsigned lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < BLOCKS; ++j) {
      const uint32_t lo = odd[j] ? v[j][0] : __builtin_amdgcn_alignbyte(v[j][1], v[j][0], 2);
      const uint32_t hi = odd[j] ? v[j][1] : __builtin_amdgcn_alignbyte(half[j], v[j][1], 2);
      StepWeights<8, BLOCKS>::put_block(lds, 16 * j + (lane >> 2), lo, hi, odd[j] ? half[j] : v[j][0] & 0xffffu);
    }
  }
  static __device__ __forceinline__ uintx4 get(const float* lds, int block, float& scale) {
    return StepWeights<8, BLOCKS>::get(lds, block, scale);
  }
};
template <int BLOCKS>
struct StepWeights<0, BLOCKS> {
  StepRows<BLOCKS> rows;
  __device__ __forceinline__ void load(const void* w, unsigned k, unsigned col0, unsigned m, unsigned base) {
    rows.load(static_cast<const float*>(w), k, col0, m, base);
  }
  __device__ __forceinline__ void put(float* lds) const { rows.put(lds); }
};
// LDS floats per wave: the rows, then the widest weights (F32).
template <int RB, int CB>
constexpr int kStepLds = 16 * (RB + CB) * kStepPitch;

// Accumulators per row block: one per column block; with F32 weights and one
// 16 x 16 tile four, a quarter of the products each, added at the end. The
// general form splits every step over the tile's four waves, so one chain per
// wave would be up to four times as long as its chains (one step: 1.5 times
// their rms error); four are as short at one step and shorter at more.
template <unsigned TYPE, int RB, int CB>
constexpr int kAcc = TYPE == 0 && RB * CB == 1 ? 4 : CB;

// acc[i][j] += rows 16 i .. of the step's activations times columns 16 j .. of
// its weights, from the wave's LDS area. The products run part by part over
// several tiles, so that an MFMA does not wait for the one before it. Where
// activations are split, largest[i] takes up the magnitudes of this lane's
// values of row 16 i + lane % 16 (kSplitsFrom).
template <unsigned TYPE, int RB, int CB>
__device__ __forceinline__ void mm_step(const float* xs, const float* ws, floatx4 (&acc)[RB][kAcc<TYPE, RB, CB>],
                                        float (&largest)[RB]) {
  if constexpr (TYPE == 0) {
    float a[RB][8], b[CB][8];
#pragma unroll
    for (int i = 0; i < RB; ++i) step_row(xs, i, a[i]);
#pragma unroll
    for (int j = 0; j < CB; ++j) step_row(ws, j, b[j]);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          floatx4& sum = acc[i][kAcc<TYPE, RB, CB> == CB ? j : e % 4];
          sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][e], b[j][e], sum, 0, 0, 0);
        }
  } else {
    Bf16Parts a[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      float f[8];
      step_row(xs, i, f);
      a[i] = split_bf16<3>(f);
#pragma unroll
      for (int e = 0; e < 8; e += 2) largest[i] = fmaxf(fmaxf(fabsf(f[e]), fabsf(f[e + 1])), largest[i]);
    }
    if constexpr (TYPE == 8 || TYPE == kQ8Edge) {
      constexpr int JB = RB == 1 ? CB : 1;  // column blocks at a time: RB JB = 4 independent dots
#pragma unroll
      for (int j0 = 0; j0 < CB; j0 += JB) {
        uintx4 b[JB];
        float d[JB];
        floatx4 dot[RB][JB];
#pragma unroll
        for (int j = 0; j < JB; ++j) {
          b[j] = StepWeights<8, CB>::get(ws, j0 + j, d[j]);
#pragma unroll
          for (int i = 0; i < RB; ++i) dot[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < JB; ++j) dot[i][j] = mfma_bf16(a[i].part[q], b[j], dot[i][j]);
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
          for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][j0 + j][v] = __builtin_fmaf(dot[i][j][v], d[j], acc[i][j0 + j][v]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const uintx4 raw = StepWeights<TYPE, CB>::get(ws, j);
        constexpr int kParts = TYPE == 1 ? 2 : 1;
        uintx4 b[2] = {raw, raw};
        if constexpr (TYPE == 1) {
          float f[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] = eg2::fp16_bits_to_fp32((raw[e / 2] >> (16 * (e & 1))) & 0xffffu);
          const Bf16Parts s = split_bf16<2>(f);
          b[0] = s.part[0];
          b[1] = s.part[1];
        }
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
          for (int c = kParts - 1; c >= 0; --c)
#pragma unroll
            for (int i = 0; i < RB; ++i) acc[i][j] = mfma_bf16(a[i].part[q], b[c], acc[i][j]);
      }
    }
  }
}

// One wave's 16 RB x 16 CB tile at (row0, col0): steps first, first + stride,
// ... of the k / 32, DEPTH of them in flight. Rows past n and columns past m
// repeat the last one.
template <unsigned TYPE, int RB, int CB, int DEPTH>
__device__ __forceinline__ void mm_direct(const EgMM& p, unsigned row0, unsigned col0, unsigned first, unsigned stride,
                                          float* lds, floatx4 (&acc)[RB][kAcc<TYPE, RB, CB>],
                                          float (&largest)[RB]) {
  const unsigned steps = p.k / 32;
  float *xs = lds, *ws = lds + 16 * RB * kStepPitch;
  StepRows<RB> x[DEPTH];
  StepWeights<TYPE, CB> w[DEPTH];
  auto load = [&](int slot, unsigned step) {
    if (DEPTH > 1 && step >= steps) return;  // uniform
    const unsigned base = 32 * min(step, steps - 1);  // one in flight: past the end the last step again, not used
    w[slot].load(p.weight, p.k, col0, p.m, base);
    x[slot].load(p.x, p.k, row0, p.n, base);
  };
#pragma unroll
  for (int s = 0; s < DEPTH; ++s) load(s, first + s * stride);
  for (unsigned step = first; step < steps; step += DEPTH * stride) {
#pragma unroll
    for (int s = 0; s < DEPTH; ++s) {
      if (step + s * stride >= steps) break;  // uniform
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // after the previous step's fragment reads
      w[s].put(ws);
      x[s].put(xs);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      load(s, step + (s + DEPTH) * stride);
      mm_step<TYPE, RB, CB>(xs, ws, acc, largest);
    }
  }
}

__device__ __forceinline__ bool mm_direct_fits(const EgMM& p) {
  const uintptr_t w = reinterpret_cast<uintptr_t>(p.weight), x = reinterpret_cast<uintptr_t>(p.x);
  return p.k % 32 == 0 && p.k > 0 && x % 16 == 0 && (p.type == 8 ? w % 2 == 0 : w % 16 == 0);
}

__device__ __forceinline__ bool is_finite(float v) { return fabsf(v) <= 3.40282347e38f; }

// A TH x TW tile per workgroup: each of the 4 waves takes the whole tile over
// every fourth step (so an activation is loaded and split once per workgroup,
// and a 512-deep product is 4 steps, not 16, of a wave's serial chain), and
// the four partial tiles are added through LDS, wave w finishing column block
// w. A sum that comes out infinite or NaN -- non-finite operands, or a Q8_0
// dot that overflows before its scale -- and the sums of a row too small to
// split (a lane's share of it: all zero or below kSplitsFrom, not all zero) are
// not stored but noted in `redo`, for the general form, which multiplies
// decoded weights by whole activations: an output's bits follow from its own row
// and column alone. Returns whether every output of the tile is stored.
template <unsigned TYPE, int TH, int TW>
__device__ __forceinline__ bool mm_tile_typed(const EgMM& p, float (*step)[kStepLds<TH / 16, TW / 16>],
                                              floatx4 (*part)[TW / 16][64], uint16_t (*small)[TH / 16],
                                              uint16_t (*redo)[TW / 16]) {
  constexpr int RB = TH / 16, CB = TW / 16, kDepth = TH == 64 ? 1 : 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
  const unsigned row0 = blockIdx.y * TH, col0 = blockIdx.x * TW;
  constexpr int kA = kAcc<TYPE, RB, CB>;
  floatx4 acc[RB][kA];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < kA; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  float largest[RB] = {};
  mm_direct<TYPE, RB, CB, kDepth>(p, row0, col0, __builtin_amdgcn_readfirstlane(wave), 4, step[wave], acc, largest);
  if constexpr (kA > CB) acc[0][0] = (acc[0][0] + acc[0][1]) + (acc[0][2] + acc[0][3]);
  auto too_small = [&](int i) { return TYPE != 0 && largest[i] > 0.0f && largest[i] < kSplitsFrom; };
  bool good = true;
#pragma unroll
  for (int i = 0; i < RB; ++i) good = good && !too_small(i);
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    __syncthreads();  // the waves' step areas, then the previous row block's parts, are no longer read
#pragma unroll
    for (int j = 0; j < CB; ++j) part[wave][j][lane] = acc[i][j];
    __syncthreads();
    if (wave < CB) {
      acc[i][0] = ((part[0][wave][lane] + part[1][wave][lane]) + part[2][wave][lane]) + part[3][wave][lane];
#pragma unroll
      for (int v = 0; v < 4; ++v) good = good && is_finite(acc[i][0][v]);
    }
  }
  const bool done = !__syncthreads_or(!good);
  // Stores the outputs that `bad` does not hold for.
  auto store = [&](auto bad) {
    if (wave >= CB) return;
    const unsigned col = col0 + 16 * wave + r;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const unsigned row = row0 + 16 * i + 4 * g + v;
        if (!bad(i, v) && row < p.n && col < p.m) p.out[(size_t)row * p.m + col] = acc[i][0][v];
      }
  };
  if (done) {
    store([](int, int) { return false; });
  } else {
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const uint64_t b = __ballot(too_small(i));  // lanes r, 16 + r, ..: row 16 i + r
      if (lane == 0) small[wave][i] = (uint16_t)(b | b >> 16 | b >> 32 | b >> 48);
    }
    __syncthreads();
    store([&](int i, int v) {
      const uint32_t rows = small[0][i] | small[1][i] | small[2][i] | small[3][i];
      const bool bad = (rows >> (4 * g + v)) & 1 || !is_finite(acc[i][0][v]);
      const uint64_t b = __ballot(bad);  // lanes 16 g ..: row 4 g + v
      if (r == 0) redo[16 * i + 4 * g + v][wave] = (uint16_t)(b >> (16 * g));
      return bad;
    });
    __syncthreads();
  }
  return done;
}

template <int TH, int TW>
__device__ __forceinline__ void mm_tile(const EgMM& p) {
  __shared__ union {
    alignas(16) float step[4][kStepLds<TH / 16, TW / 16>];
    floatx4 part[4][TW / 16][64];
    struct {
      floatx4 part[(TH == 16 && TW == 16) ? 3 * 64 : 1];
      alignas(16) float xs[TH * kPitch], ws[TW * kPitch];
    } general;
  } lds;
  __shared__ uint16_t small[4][TH / 16], redo[TH][TW / 16];
  if (blockIdx.y * TH >= p.n || blockIdx.x * TW >= p.m) return;
  const bool direct = mm_direct_fits(p);
  bool done = false;  // uniform
  if (direct) {
    switch (p.type) {
      case 0: done = mm_tile_typed<0, TH, TW>(p, lds.step, lds.part, small, redo); break;
      case 1: done = mm_tile_typed<1, TH, TW>(p, lds.step, lds.part, small, redo); break;
      case 30: done = mm_tile_typed<30, TH, TW>(p, lds.step, lds.part, small, redo); break;
      default: {
        const uintptr_t first = reinterpret_cast<uintptr_t>(p.weight);
        const uintptr_t end = first + (uintptr_t)p.m * (p.k / 32) * 34;
        const bool edge = (blockIdx.x == 0 && first % 4 != 0) || ((blockIdx.x + 1) * TW >= p.m && end % 4 != 0);
        done = __builtin_expect(edge, 0) ? mm_tile_typed<kQ8Edge, TH, TW>(p, lds.step, lds.part, small, redo)
                                         : mm_tile_typed<8, TH, TW>(p, lds.step, lds.part, small, redo);
        break;
      }
    }
  }
  if (!done) mm_general<TH, TW>(p, lds.general.xs, lds.general.ws, lds.general.part, direct ? redo : nullptr);
}

// -------------------------------------------------------------- row sums

// Sum over the 64 lanes: DPP exchanges within each 16-lane row (lanes
// i^1, i^2, then the mirrored half-row and row), then the four row totals
// added as (r0 + r1) + (r2 + r3). Wave-uniform result.
__device__ __forceinline__ float dpp_wave_sum(float v) {
  auto dpp = [](float x, int ctrl) -> float {
    switch (ctrl) {
      case 0:
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, false));  // quad [1,0,3,2]
      case 1:
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, false));  // quad [2,3,0,1]
      case 2:
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, false));  // row_half_mirror
      default:
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x140, 0xF, 0xF, false));  // row_mirror
    }
  };
  v = v + dpp(v, 0);
  v = v + dpp(v, 1);
  v = v + dpp(v, 2);
  v = v + dpp(v, 3);
  const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return (r0 + r1) + (r2 + r3);
}

__device__ __forceinline__ float dpp_wave_max(float v) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return v;
}

// A row of d floats held by one wave: float4 chunks c = lane + 64 j
// (elements 4c .. 4c + 3) for j < kRowChunks when d % 4 == 0 and d <=
// 256 kRowChunks; other widths are read element-wise in two passes.
constexpr int kRowChunks = 4;

struct Row {
  floatx4 v[kRowChunks];
};

__device__ __forceinline__ bool row_in_registers(unsigned d) { return d % 4 == 0 && d <= 256u * kRowChunks; }

__device__ __forceinline__ Row load_row(const float* x, unsigned d, unsigned lane) {
  Row r;
#pragma unroll
  for (int j = 0; j < kRowChunks; ++j) {
    const unsigned c = lane + 64u * j;
    r.v[j] = 4 * c < d ? *reinterpret_cast<const floatx4*>(x + 4 * c) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  return r;
}

// 1 / sqrt(mean((x * pre)^2) + 1e-6) of a row.
__device__ __forceinline__ float row_inverse_rms(const float* x, unsigned d, float pre, unsigned lane, const Row* r) {
  float ss = 0.0f;
  if (r) {
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = r->v[j][e] * pre;
        ss = __builtin_fmaf(v, v, ss);
      }
  } else {
    for (unsigned z = lane; z < d; z += 64) {
      const float v = x[z] * pre;
      ss = __builtin_fmaf(v, v, ss);
    }
  }
  return eg2::rms_inverse(dpp_wave_sum(ss), (int)d, 1.0e-6f);
}

// The normalized value of element z: ((x * pre) * inv) * w.
__device__ __forceinline__ float normed(float x, float pre, float inv, const float* w, unsigned z) {
  const float v = (x * pre) * inv;
  return w ? v * w[z] : v;
}

// NeoX rotation of the pair (a, b) by (c, s).
__device__ __forceinline__ void rotate(float a, float b, float c, float s, float& ra, float& rb) {
  const float ac = a * c, bs = b * s, as = a * s, bc = b * c;
  ra = ac - bs;
  rb = as + bc;
}

// --------------------------------------------------------------- attention

// One wave per (token t, query head h): out = softmax(q . K^T) V over the
// keys [bounds[2t], bounds[2t+1]) clipped to |t - s| <= window (window >
// 0). q rows of D floats per (t, h); K/V rows of KVS floats with head h's
// KV block at (h / GROUP) * D.
// Computed by one wave with LDS of its own (qs, ps).
__device__ __forceinline__ void wave_lds_order() {  // a wave's LDS accesses execute in order: keep the compiler to it
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int D, int HEADS, int KVS, int GROUP>
__device__ __forceinline__ void attention_chunked(const EgAttention& p, unsigned row, floatx4* qs, float* ps) {
  static_assert(D % 256 == 0, "lanes own float4s of the context");
  constexpr int CV = D / 256;  // float4 of the context per lane
  const unsigned lane = threadIdx.x & 63;
  const unsigned t = row / HEADS, h = row % HEADS, kv = (h / GROUP) * D;
  if (t >= p.n) return;
  unsigned lo = p.bounds[2 * t], hi = p.bounds[2 * t + 1];
  if (p.window) {
    if (t > p.window) lo = max(lo, t - p.window);
    hi = min(hi, t + p.window + 1);
  }
  for (unsigned c = lane; c < D / 4; c += 64) qs[c] = reinterpret_cast<const floatx4*>(p.q + (size_t)row * D)[c];
  wave_lds_order();
  float run_max = -__builtin_inff(), den = 0.0f;
  floatx4 acc[CV];
#pragma unroll
  for (int u = 0; u < CV; ++u) acc[u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  for (unsigned c0 = lo; c0 < hi; c0 += 64) {
    const unsigned key = c0 + lane;
    float score = -__builtin_inff();
    if (key < hi) {
      const floatx4* kr = reinterpret_cast<const floatx4*>(p.k + (size_t)key * KVS + kv);
      floatx4 s4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
      for (int c = 0; c < D / 4; ++c) {
        const floatx4 k4 = kr[c], q4 = qs[c];
#pragma unroll
        for (int e = 0; e < 4; ++e) s4[e] = __builtin_fmaf(q4[e], k4[e], s4[e]);
      }
      score = (s4[0] + s4[1]) + (s4[2] + s4[3]);
    }
    // A score of -inf (no key, an infinite element, a dot product past the
    // range) weighs 0, also while no other has been met and the maximum itself
    // is -inf; a row with no other score ends as 0/0.
    const float next = fmaxf(run_max, dpp_wave_max(score));
    const float alpha = run_max == -__builtin_inff() ? 0.0f : eg2::libm::expf(run_max - next);
    const float pk = score == -__builtin_inff() ? 0.0f : eg2::libm::expf(score - next);
    den = den * alpha + dpp_wave_sum(pk);
    ps[lane] = pk;
    wave_lds_order();
#pragma unroll
    for (int u = 0; u < CV; ++u) acc[u] = acc[u] * alpha;
    const unsigned count = min(64u, hi - c0);
    const float* vbase = p.v + (size_t)c0 * KVS + kv + 4 * lane;
#pragma unroll 8
    for (unsigned j = 0; j < count; ++j) {
      const float w = ps[j];
#pragma unroll
      for (int u = 0; u < CV; ++u) {
        const floatx4 v4 = *reinterpret_cast<const floatx4*>(vbase + (size_t)j * KVS + 256 * u);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[u][e] = __builtin_fmaf(w, v4[e], acc[u][e]);
      }
    }
    wave_lds_order();  // ps is rewritten by the next chunk
    run_max = next;
  }
  const float inv = hi > lo ? 1.0f / den : 0.0f;
#pragma unroll
  for (int u = 0; u < CV; ++u)
    *reinterpret_cast<floatx4*>(p.out + (size_t)row * D + 4 * lane + 256 * u) = acc[u] * inv;
}

// The same attention over tiles of 16 tokens x one head, which eg2_op_launch
// takes for the contract's whole grid from kTileTokens tokens on (the
// by-symbol kernel's one wave per (token, head) reads every key and value row
// once per token and head: 17 GB from the L2 for one 2048-token sequence). A
// workgroup of kTileWaves waves shares the 16 queries in LDS; wave w takes
// every kTileWaves-th 16-key block of the keys that any of its tokens has,
// with its own running maximum, sum and context (the softmax recurrence of the
// form above), and the waves' results are rescaled to the common maximum and
// added at the end. Both products run on fp32 MFMA (v_mfma_f32_16x16x4f32):
//  - scores: lane 16 g + r feeds key r; one float4 of its row, dimensions
//    16 E + 4 g .., is four MFMAs (q from LDS in the same order). The key rows
//    come through the wave's LDS 64 dimensions at a time, read along the rows
//    (in the MFMA's order a load touches 64 lines, which alone took twice the
//    MFMAs' time), the next 64 on their way meanwhile;
//  - context: the 16 x 16 weights go through LDS to the operand order (lane
//    16 g + r: query r, keys 4 g .. 4 g + 3), and a lane's float4 of a value
//    row, dimensions 64 T + 4 r .., feeds four output tiles.
// A key outside a token's range weighs 0 there. The 2-norm error to a float64
// softmax is that of the form above or less (2.2e-7 against 2.8e-7 at 1021
// tokens in 9 texts, 3.8e-7 against 8.4e-7 on one of 2048); a row's rounding
// depends on the tile and wave its keys fall to, so on the packing. Bound by the
// MFMAs (128 of 33 cycles per 16 x 16 scores) and, over few keys, by the
// chain of one block. eg2_attention256 inside a graph, that form / this one in
// us: 1021 tokens in texts of 113 67 / 21, 2048 in texts of 128 145 / 27, one of
// 2048 2,240 / 212; eg2_attention512 130 / 39, 285 / 50, 4,460 / 425.
//
// The host knows the token count and the window but not the ranges, so a tile
// chooses by the keys that its tokens reach: few keys close together
// (attention_few_keys), few keys far apart (row by row), else by keys. At 512
// tokens, that form / this one: texts of one token 6.9 / 6.3, of 8 8.4 / 6.3, of
// 16 10.3 / 6.3, of 24 12.1 / 10.2, of 64 21.5 / 11.4; window 4 8.7 / 8.1, 16
// 14.2 / 10.4; at 2048 texts of one token 20.4 / 13.7. (By keys alone 10.0-11.4
// at 512 whatever the texts, 22 at 2048.) Slower than one wave per row is only
// what no packing has, neighbours whose keys lie far apart: 8 keys anywhere, 512
// tokens 8.4 / 16.5, 2048 25.8 / 32.6; 100 keys, 1040 tokens 66 / 99, 2048 122 / 165;
// the rows of a tile share its CU.
constexpr int kTileWaves = 8;
// From here the tiles fill half of the CUs; fewer tokens were not looked into.
constexpr unsigned kTileTokens = 512;

template <int D>
struct AttentionTileLds {
  alignas(16) float q[16][D + 4];
  alignas(16) float p[kTileWaves][16][20];
  float m[kTileWaves][16], l[kTileWaves][16];
  // 64 dimensions of a wave's 16 keys; at the end, of its 16 rows' context.
  alignas(16) float part[kTileWaves][16][68];
  uint64_t exp_tab[32];
};

// Reductions over the 16 lanes of a DPP row, on every lane of it.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, eg2::dpp<eg2::kQuad1032>(v));
  v = fmaxf(v, eg2::dpp<eg2::kQuad2301>(v));
  v = fmaxf(v, eg2::dpp<eg2::kRowHalfMirror>(v));
  return fmaxf(v, eg2::dpp<eg2::kRowMirror>(v));
}
__device__ __forceinline__ float row16_sum(float v) {
  v = v + eg2::dpp<eg2::kQuad1032>(v);
  v = v + eg2::dpp<eg2::kQuad2301>(v);
  v = v + eg2::dpp<eg2::kRowHalfMirror>(v);
  return v + eg2::dpp<eg2::kRowMirror>(v);
}

// A tile whose tokens reach at most kFewKeys keys [first, last) between them:
// texts of a few tokens, or a narrow window. Split by keys such a tile would
// have work for one wave or a few; here every wave takes all the keys over an
// eighth of the dimensions, its keys and values on their way at once, the
// waves' partial scores are added through LDS, and each wave carries the whole
// softmax and the context of its own dimensions. (With a fourth block of keys
// the split by keys is faster: texts of 64, 512 tokens, 12.9 us against 11.4,
// of three blocks 10.2 against 10.6.) lo, hi: the key ranges of the
// lane's rows 4 g + v. Returns whether the tile needs the per-row form (as the
// kernel's `polluted`); it has stored nothing then.
constexpr int kFewBlocks = 3;
constexpr unsigned kFewKeys = 16 * kFewBlocks;

template <int D, int HEADS, int KVS>
__device__ __forceinline__ bool attention_few_keys(const EgAttention& p, AttentionTileLds<D>& lds, unsigned t0,
                                                   unsigned h, unsigned kv, const unsigned (&lo)[4],
                                                   const unsigned (&hi)[4], unsigned first, unsigned last) {
  constexpr int kDims = D / kTileWaves, kPer = kDims / 16;  // a wave's dimensions; float4s of a key, outputs per lane
  typedef float floatxp __attribute__((ext_vector_type(kPer)));
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const unsigned nb = (last - first + 15) / 16;
  floatx4 kf[kFewBlocks][kPer];  // key r of each block, dimensions 16 e + 4 g ..
  floatxp vf[kFewBlocks][4];     // keys 4 g + j, dimensions kPer r ..
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
      const float* row = p.k + (size_t)min(first + 16 * b + r, last - 1) * KVS + kv + kDims * w + 4 * g;
#pragma unroll
      for (int e = 0; e < kPer; ++e) kf[b][e] = *reinterpret_cast<const floatx4*>(row + 16 * e);
    }
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        vf[b][j] = *reinterpret_cast<const floatxp*>(p.v + (size_t)min(first + 16 * b + 4 * g + j, last - 1) * KVS +
                                                     kv + kDims * w + kPer * r);
    }
  __syncthreads();  // the queries and the exp table are in LDS
  floatx4 qf[kPer];
#pragma unroll
  for (int e = 0; e < kPer; ++e) qf[e] = *reinterpret_cast<const floatx4*>(&lds.q[r][kDims * w + 16 * e + 4 * g]);
  floatx4 s[kFewBlocks];
  floatx4* partial = reinterpret_cast<floatx4*>(lds.part[w][0]);
  bool polluted = false;
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
      s[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int e = 0; e < kPer; ++e)
#pragma unroll
        for (int c = 0; c < 4; ++c) s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[e][c], kf[b][e][c], s[b], 0, 0, 0);
      partial[64 * b + lane] = s[b];
    }
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
      bool all_in = true;
#pragma unroll
      for (int v = 0; v < 4; ++v) all_in = all_in && lo[v] <= first + 16 * b && first + 16 * b + 16 <= hi[v];
      if (!__all(all_in)) {
        float probe = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < kPer; ++i) probe = __builtin_fmaf(vf[b][j][i], 0.0f, probe);
        polluted = polluted || !(probe == 0.0f);
      }
    }
  if (__syncthreads_or(polluted)) return true;
  float m[4], l[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) m[v] = -__builtin_inff(), l[v] = 0.0f;
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
      s[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < kTileWaves; ++i)
        s[b] = s[b] + reinterpret_cast<const floatx4*>(lds.part[i][0])[64 * b + lane];
      const unsigned key = first + 16 * b + r;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[b][v] = key >= lo[v] && key < hi[v] ? s[b][v] : -__builtin_inff();
        m[v] = fmaxf(m[v], s[b][v]);
      }
    }
#pragma unroll
  for (int v = 0; v < 4; ++v) m[v] = row16_max(m[v]);
  floatx4 acc[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) acc[i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int b = 0; b < kFewBlocks; ++b)
    if (b < nb) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float pk = s[b][v] == -__builtin_inff() ? 0.0f : eg2::libm::expf_tab(s[b][v] - m[v], lds.exp_tab);
        l[v] = l[v] + pk;
        lds.p[w][4 * g + v][r] = pk;
      }
      wave_lds_order();
      const floatx4 pf = *reinterpret_cast<const floatx4*>(&lds.p[w][r][4 * g]);  // query r, keys 4 g ..
      wave_lds_order();  // p is rewritten by the next block
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < kPer; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[j], vf[b][j][i], acc[i], 0, 0, 0);
    }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float den = row16_sum(l[v]);  // every lane active
    const float inv = hi[v] > lo[v] ? 1.0f / den : 0.0f;
    const unsigned t = t0 + 4 * g + v;
    floatxp o;
#pragma unroll
    for (int i = 0; i < kPer; ++i) o[i] = acc[i][v] * inv;
    if (t < p.n) *reinterpret_cast<floatxp*>(p.out + ((size_t)t * HEADS + h) * D + kDims * w + kPer * r) = o;
  }
  return false;
}

template <int D, int HEADS, int KVS, int GROUP>
__global__ void __launch_bounds__(64 * kTileWaves)
attention_tile_kernel(EgAttention p) {
  constexpr int T = D / 64;  // 64-dimension parts of the context
  __shared__ AttentionTileLds<D> lds;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15;
  const unsigned t0 = 16 * blockIdx.x, h = blockIdx.y, kv = (h / GROUP) * D;
  for (int c = tid; c < 16 * D / 4; c += 64 * kTileWaves) {
    const int row = c / (D / 4), e = c % (D / 4);
    *reinterpret_cast<floatx4*>(&lds.q[row][4 * e]) =
        *reinterpret_cast<const floatx4*>(p.q + ((size_t)min(t0 + row, p.n - 1) * HEADS + h) * D + 4 * e);
  }
  if (tid < 32) lds.exp_tab[tid] = eg2::libm::kExp2Tab.t[tid];
  auto exp_ = [&](float x) { return eg2::libm::expf_tab(x, lds.exp_tab); };
  // Key ranges: of token t0 + r in every lane (for the union), of the lane's
  // output rows 4 g + v.
  auto range = [&](unsigned t, unsigned& lo, unsigned& hi) {
    lo = hi = 0;
    if (t >= p.n) return;
    lo = p.bounds[2 * t];
    hi = p.bounds[2 * t + 1];
    if (p.window) {
      if (t > p.window) lo = max(lo, t - p.window);
      hi = min(hi, t + p.window + 1);
    }
    if (hi <= lo) lo = hi = 0;
  };
  unsigned lo[4], hi[4], first = 0xffffffffu, last = 0;
#pragma unroll
  for (int v = 0; v < 4; ++v) range(t0 + 4 * g + v, lo[v], hi[v]);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const unsigned a = __builtin_amdgcn_readlane(lo[i & 3], 16 * (i >> 2)), b = __builtin_amdgcn_readlane(hi[i & 3], 16 * (i >> 2));
    if (b > a) {
      first = min(first, a);
      last = max(last, b);
    }
  }
  first = min(first, last);
  // The keys split over the waves; whether the tile needs the per-row form.
  auto by_keys = [&]() -> bool {
    float m[4], l[4];
    floatx4 acc[4 * T];
#pragma unroll
    for (int v = 0; v < 4; ++v) m[v] = -__builtin_inff(), l[v] = 0.0f;
#pragma unroll
    for (int i = 0; i < 4 * T; ++i) acc[i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // Rows 4 i + lane / 16 of a key block, dimensions 64 part + 4 (lane % 16) ..
    // (rows past the last repeat it; their scores are masked).
    floatx4 kr[4];
    auto load_k = [&](unsigned k0, int part) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        kr[i] = *reinterpret_cast<const floatx4*>(p.k + (size_t)min(k0 + 4 * i + g, last - 1) * KVS + kv + 64 * part +
                                                 4 * r);
    };
    bool polluted = false;
    if (first + 16 * w < last) load_k(first + 16 * w, 0);
    __syncthreads();  // the queries and the exp table are in LDS
    for (unsigned k0 = first + 16 * w; k0 < last; k0 += 16 * kTileWaves) {
      // Scores of keys k0 .. + 15, in four chains.
      floatx4 s[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) s[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int part = 0; part < T; ++part) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<floatx4*>(&lds.part[w][4 * i + g][4 * r]) = kr[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (part + 1 < T)
          load_k(k0, part + 1);
        else if (k0 + 16 * kTileWaves < last)
          load_k(k0 + 16 * kTileWaves, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const floatx4 kf = *reinterpret_cast<const floatx4*>(&lds.part[w][r][16 * e + 4 * g]);
          const floatx4 qf = *reinterpret_cast<const floatx4*>(&lds.q[r][64 * part + 16 * e + 4 * g]);
#pragma unroll
          for (int c = 0; c < 4; ++c) s[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[c], kf[c], s[c], 0, 0, 0);
        }
      }
      // The block's first value rows, on their way during the softmax: keys
      // k0 + 4 g + j, kAhead j in flight (one at 512 dimensions, whose context
      // takes half of the registers).
      constexpr int kAhead = D == 256 ? 2 : 1;
      floatx4 vr[kAhead][T];
      auto load_v = [&](int slot, int j) {
        const float* vrow = p.v + (size_t)min(k0 + 4 * g + j, last - 1) * KVS + kv + 4 * r;
#pragma unroll
        for (int part = 0; part < T; ++part) vr[slot][part] = *reinterpret_cast<const floatx4*>(vrow + 64 * part);
      };
#pragma unroll
      for (int j = 0; j < kAhead; ++j) load_v(j, j);
      float score[4], next[4];
      bool grown = false;
#pragma unroll
      for (int v = 0; v < 4; ++v) {  // row 4 g + v, key k0 + r
        const bool in = k0 + r >= lo[v] && k0 + r < hi[v];
        score[v] = in ? (s[0][v] + s[1][v]) + (s[2][v] + s[3][v]) : -__builtin_inff();
        next[v] = fmaxf(m[v], row16_max(score[v]));
        grown = grown || next[v] != m[v];
      }
      if (__any(grown)) {
        float alpha[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          alpha[v] = next[v] == -__builtin_inff() ? 0.0f : exp_(m[v] - next[v]);  // no key of this row yet: all zero
          l[v] = l[v] * alpha[v];
          m[v] = next[v];
        }
#pragma unroll
        for (int i = 0; i < 4 * T; ++i)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][v] = acc[i][v] * alpha[v];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float pk = score[v] == -__builtin_inff() ? 0.0f : exp_(score[v] - m[v]);
        l[v] = l[v] + row16_sum(pk);
        lds.p[w][4 * g + v][r] = pk;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const floatx4 pf = *reinterpret_cast<const floatx4*>(&lds.p[w][r][4 * g]);  // query r, keys 4 g ..
      // A key outside a row's range weighs +0, but +0 times an infinite or NaN
      // value is NaN: where some row does not have all 16 keys, such values send
      // the whole tile to the per-row form below.
      bool all_in = true;
#pragma unroll
      for (int v = 0; v < 4; ++v) all_in = all_in && lo[v] <= k0 && k0 + 16 <= hi[v];
      const bool partial = !__all(all_in);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (partial) {  // uniform
          float probe = 0.0f;
#pragma unroll
          for (int part = 0; part < T; ++part)
#pragma unroll
            for (int i = 0; i < 4; ++i) probe = __builtin_fmaf(vr[j % kAhead][part][i], 0.0f, probe);
          polluted = polluted || !(probe == 0.0f);
        }
#pragma unroll
        for (int part = 0; part < T; ++part)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc[4 * part + i] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(pf[j], vr[j % kAhead][part][i], acc[4 * part + i], 0, 0, 0);
        if (j + kAhead < 4) load_v(j % kAhead, j + kAhead);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // p is rewritten by the next block
    }
    // The waves' contexts brought to the rows' common maximum and added; thread
    // 16 i + row computes wave i's factor for the row.
    if (__syncthreads_or(polluted)) return true;
    if (r == 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) lds.m[w][4 * g + v] = m[v], lds.l[w][4 * g + v] = l[v];
    }
    __syncthreads();
    if (tid < 16 * kTileWaves) {
      const int row = tid & 15;
      const float own = lds.m[tid >> 4][row];
      float top = own;
#pragma unroll
      for (int i = 0; i < kTileWaves; ++i) top = fmaxf(top, lds.m[i][row]);
      lds.p[tid >> 4][row][0] = own == -__builtin_inff() ? 0.0f : exp_(own - top);
    }
    __syncthreads();
    float scale[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 4 * g + v;
      float den = 0.0f;
#pragma unroll
      for (int i = 0; i < kTileWaves; ++i) den = den + lds.l[i][row] * lds.p[i][row][0];
      scale[v] = hi[v] > lo[v] ? lds.p[w][row][0] / den : 0.0f;
    }
#pragma unroll
    for (int part = 0; part < T; ++part) {
      if (part) __syncthreads();
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        floatx4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = acc[4 * part + i][v] * scale[v];
        *reinterpret_cast<floatx4*>(&lds.part[w][4 * g + v][4 * r]) = o;
      }
      __syncthreads();
      const int row = tid >> 5, e = 2 * (tid & 31);  // 512 threads x 2 outputs
      float a = 0.0f, b = 0.0f;
#pragma unroll
      for (int i = 0; i < kTileWaves; ++i) {
        a = a + lds.part[i][row][e];
        b = b + lds.part[i][row][e + 1];
      }
      if (t0 + row < p.n) {
        float* dst = p.out + ((size_t)(t0 + row) * HEADS + h) * D + 64 * part + e;
        dst[0] = a;
        dst[1] = b;
      }
    }
    return false;
  };
  // Tokens whose few keys lie far apart go one by one: a row costs about 15 us +
  // 0.7 a key where the tile costs 3 + 6.5 per 128 keys of the whole reach
  // (2048 tokens with 8 keys each anywhere: 182 us by keys, 32 by row).
  const unsigned reach = last - first;
  const unsigned longest = max(max(hi[0] - lo[0], hi[1] - lo[1]), max(hi[2] - lo[2], hi[3] - lo[3]));  // of four rows
  bool rows = reach > 256 && !__any(longest + 17 >= 9 * ((reach + 127) / 128));
  if (!rows)
    rows = reach <= kFewKeys ? attention_few_keys<D, HEADS, KVS>(p, lds, t0, h, kv, lo, hi, first, last) : by_keys();
  if (!rows) return;
  __syncthreads();
  for (unsigned i = w; i < 16 && t0 + i < p.n; i += kTileWaves)
    attention_chunked<D, HEADS, KVS, GROUP>(p, (t0 + i) * HEADS + h, reinterpret_cast<floatx4*>(lds.q[w]),
                                            lds.part[w][0]);
}

}  // namespace

// y = a x + y.
extern "C" __global__ void eg2_saxpy(float* y, const float* x, float a, unsigned n) {
  const unsigned i = flat_index();
  if (i < n) y[i] = __builtin_fmaf(a, x[i], y[i]);
}

// Rows of 512 values of a Q8_0 table: (fp16(d) * q) * sqrt(512)
// (kernels/eg2.c:36-39 semantics).
extern "C" __global__ void eg2_gather(EgGather p) {
  const unsigned i = flat_index();
  if (i >= p.n * 512u) return;
  const unsigned r = i >> 9, z = i & 511;
  p.out[i] = weight_at(p.weight, (size_t)p.ids[r] * 512 + z, 8) * 22.62741699796952f;
}

// Rows of 768 values with the 768-wide CPU path's order (engine.c:288-295,
// quants.c:67,86-88): (fp16(d) * sqrt(768)) * q.
extern "C" __global__ void eg2_gather768(EgGather p) {
  const unsigned i = flat_index();
  if (i >= p.n * 768u) return;
  const unsigned r = i / 768u, z = i - 768u * r;
  const unsigned char* blk = static_cast<const unsigned char*>(p.weight) + ((size_t)p.ids[r] * 24 + z / 32) * 34;
  const float d = eg2::fp16_bits_to_fp32((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
  p.out[i] = (d * 27.712812921102035f) * (float)reinterpret_cast<const signed char*>(blk + 2)[z & 31];
}

// kernels/eg2.c:41-119 semantics, four tile shapes.
extern "C" __global__ void __launch_bounds__(256) eg2_mm(EgMM p) { mm_tile<16, 16>(p); }
extern "C" __global__ void __launch_bounds__(256) eg2_mm64(EgMM p) { mm_tile<16, 64>(p); }
extern "C" __global__ void __launch_bounds__(256) eg2_mm64x64(EgMM p) { mm_tile<64, 64>(p); }
extern "C" __global__ void __launch_bounds__(256) eg2_mmstep8(EgMM p) { mm_tile<64, 64>(p); }

// out = ((x * scale) * inv) * w, inv = 1/sqrt(mean((x * scale)^2) + 1e-6);
// w may be NULL (= 1); out == x is valid (kernels/eg2.c:121-133 semantics).
extern "C" __global__ void __launch_bounds__(64) eg2_norm(EgNorm p) {
  const unsigned row = blockIdx.x, lane = threadIdx.x;
  if (row >= p.rows) return;
  const float* x = p.x + (size_t)row * p.d;
  float* out = p.out + (size_t)row * p.d;
  if (row_in_registers(p.d)) {
    const Row r = load_row(x, p.d, lane);
    const float inv = row_inverse_rms(x, p.d, p.scale, lane, &r);
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j) {
      const unsigned c = lane + 64u * j;
      if (4 * c >= p.d) break;
      floatx4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = normed(r.v[j][e], p.scale, inv, p.weight, 4 * c + e);
      *reinterpret_cast<floatx4*>(out + 4 * c) = o;
    }
  } else {
    const float inv = row_inverse_rms(x, p.d, p.scale, lane, nullptr);
    for (unsigned z = lane; z < p.d; z += 64) out[z] = normed(x[z], p.scale, inv, p.weight, z);
  }
}

// NeoX rotation of pairs (z, z + d/2), table row of token row/heads =
// [cos(d/2) | sin(d/2)] (kernels/eg2.c:135-143 semantics).
extern "C" __global__ void eg2_rope(EgRope p) {
  const unsigned i = flat_index(), half = p.d / 2;
  if (i >= p.n * p.heads * half) return;
  const unsigned z = i % half, row = i / half, t = row / p.heads;
  const float* tab = p.table + (size_t)t * p.d;
  float* x = p.x + (size_t)row * p.d;
  rotate(x[z], x[half + z], tab[z], tab[half + z], x[z], x[half + z]);
}

// kernels/eg2.c:145-170 semantics: 4 query heads per token; d 256 reads KV
// head h/2 of two, d 512 the single KV head (K/V rows of 512 floats).
extern "C" __global__ void __launch_bounds__(64) eg2_attention256(EgAttention p) {
  __shared__ __align__(16) floatx4 qs[64];
  __shared__ float ps[64];
  attention_chunked<256, 4, 512, 2>(p, blockIdx.x, qs, ps);
}
extern "C" __global__ void __launch_bounds__(64) eg2_attention512(EgAttention p) {
  __shared__ __align__(16) floatx4 qs[128];
  __shared__ float ps[64];
  attention_chunked<512, 4, 512, 4>(p, blockIdx.x, qs, ps);
}
// 3 query heads sharing one KV head of 256 (K/V rows of 256 floats).
extern "C" __global__ void __launch_bounds__(64) eg2_attention256x3(EgAttention p) {
  __shared__ __align__(16) floatx4 qs[64];
  __shared__ float ps[64];
  attention_chunked<256, 3, 256, 3>(p, blockIdx.x, qs, ps);
}

// Mode 0: (x + other) * scale; 1: gelu(x) * other; 2: gelu(x) * the
// per-layer gate other[(i/512 * 24 + layer) * 512 + i % 512]
// (kernels/eg2.c:172-179 semantics). Both loads come before the mode
// branch: with the x load inside a three-way branch, hipcc (ROCm 7.2, -O3)
// left the mode-2 path's x address undefined.
extern "C" __global__ void eg2_element(EgElement p) {
  const unsigned i = flat_index();
  if (i >= p.n) return;
  const size_t o = p.mode == 2 ? ((size_t)(i >> 9) * 24 + p.layer) * 512 + (i & 511) : (size_t)i;
  const float xv = p.x[i], ov = p.other[o];
  p.out[i] = p.mode == 0 ? (xv + ov) * p.scale : eg2::gelu_mul(xv, ov);
}

// Mean over rows [offsets[s], offsets[s+1]) of width 768, in row order
// (kernels/eg2.c:181-188 semantics); four rows' loads in flight at a time.
extern "C" __global__ void eg2_pool(EgPool p) {
  const unsigned i = flat_index(), seq = i / 768u, z = i - 768u * seq;
  if (seq >= p.batch) return;
  const unsigned lo = p.offsets[seq], hi = p.offsets[seq + 1];
  const float* col = p.x + z;
  float sum = 0.0f;
  unsigned t = lo;
  for (; t + 4 <= hi; t += 4) {
    const float a = col[(size_t)t * 768], b = col[(size_t)(t + 1) * 768];
    const float c = col[(size_t)(t + 2) * 768], d = col[(size_t)(t + 3) * 768];
    sum = sum + a;
    sum = sum + b;
    sum = sum + c;
    sum = sum + d;
  }
  for (; t < hi; ++t) sum = sum + col[(size_t)t * 768];
  p.out[i] = sum / (float)(hi - lo);
}

// out = (out + (x * inv) * w) * scale (kernels/eg2.c:190-202 semantics):
// the normalized values of eg2_norm with scale 1, added to the residual.
extern "C" __global__ void __launch_bounds__(64) eg2_norm_residual(EgNormResidual p) {
  const unsigned row = blockIdx.x, lane = threadIdx.x;
  if (row >= p.rows) return;
  const float* x = p.x + (size_t)row * p.d;
  float* out = p.out + (size_t)row * p.d;
  if (row_in_registers(p.d)) {
    const Row r = load_row(x, p.d, lane);
    const float inv = row_inverse_rms(x, p.d, 1.0f, lane, &r);
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j) {
      const unsigned c = lane + 64u * j;
      if (4 * c >= p.d) break;
      floatx4 o = *reinterpret_cast<const floatx4*>(out + 4 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (o[e] + normed(r.v[j][e], 1.0f, inv, p.weight, 4 * c + e)) * p.scale;
      *reinterpret_cast<floatx4*>(out + 4 * c) = o;
    }
  } else {
    const float inv = row_inverse_rms(x, p.d, 1.0f, lane, nullptr);
    for (unsigned z = lane; z < p.d; z += 64) out[z] = (out[z] + normed(x[z], 1.0f, inv, p.weight, z)) * p.scale;
  }
}

// Per-row RMS with the row weight, then the NeoX rotation with the table
// row of token row/heads, in place (kernels/eg2.c:204-217 semantics): the
// normalized row goes through LDS so that each lane can take its pairs.
extern "C" __global__ void __launch_bounds__(64) eg2_norm_rope(EgNormRope p) {
  constexpr unsigned kMaxD = 4096;
  __shared__ float nrow[kMaxD];
  const unsigned row = blockIdx.x, lane = threadIdx.x, half = p.d / 2;
  if (row >= p.rows || p.d > kMaxD) return;
  float* x = p.x + (size_t)row * p.d;
  if (row_in_registers(p.d)) {
    const Row r = load_row(x, p.d, lane);
    const float inv = row_inverse_rms(x, p.d, 1.0f, lane, &r);
#pragma unroll
    for (int j = 0; j < kRowChunks; ++j) {
      const unsigned c = lane + 64u * j;
      if (4 * c >= p.d) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) nrow[4 * c + e] = normed(r.v[j][e], 1.0f, inv, p.weight, 4 * c + e);
    }
  } else {
    const float inv = row_inverse_rms(x, p.d, 1.0f, lane, nullptr);
    for (unsigned z = lane; z < p.d; z += 64) nrow[z] = normed(x[z], 1.0f, inv, p.weight, z);
  }
  __syncthreads();
  const float* tab = p.table + (size_t)(row / p.heads) * p.d;
  for (unsigned z = lane; z < half; z += 64) rotate(nrow[z], nrow[half + z], tab[z], tab[half + z], x[z], x[half + z]);
}

// ---------------------------------------------------------------- dispatch

#include <cstring>

#include "eg2_ops.h"

namespace {

enum class Block { kAny, k64, k256 };

struct OpEntry {
  const char* name;
  const void* fn;
  size_t record_size;
  Block block;
  bool (*valid)(const void* record);
  const void* tile = nullptr;  // attention: the tiled kernel for the whole grid of heads x n
  unsigned heads = 0;
};

template <class R>
const R& as(const void* r) {
  return *static_cast<const R*>(r);
}

bool valid_saxpy(const void* r) { return as<EgSaxpy>(r).y && as<EgSaxpy>(r).x; }
bool valid_gather(const void* r) { return as<EgGather>(r).out && as<EgGather>(r).weight && as<EgGather>(r).ids; }
bool valid_mm(const void* r) {
  const EgMM& p = as<EgMM>(r);
  return p.out && p.x && p.weight && (p.type == 0 || p.type == 1 || p.type == 8 || p.type == 30);
}
bool valid_norm(const void* r) { return as<EgNorm>(r).out && as<EgNorm>(r).x && as<EgNorm>(r).d > 0; }
bool valid_rope(const void* r) {
  const EgRope& p = as<EgRope>(r);
  return p.x && p.table && p.d > 0 && p.d % 2 == 0;
}
bool valid_attention(const void* r) {
  const EgAttention& p = as<EgAttention>(r);
  return p.out && p.q && p.k && p.v && p.bounds;
}
bool valid_element(const void* r) {
  const EgElement& p = as<EgElement>(r);
  return p.out && p.x && p.other && p.mode <= 2;
}
bool valid_pool(const void* r) { return as<EgPool>(r).out && as<EgPool>(r).x && as<EgPool>(r).offsets; }
bool valid_norm_residual(const void* r) {
  const EgNormResidual& p = as<EgNormResidual>(r);
  return p.out && p.x && p.weight && p.d > 0;
}
bool valid_norm_rope(const void* r) {
  const EgNormRope& p = as<EgNormRope>(r);
  return p.x && p.weight && p.table && p.d > 0 && p.d % 2 == 0 && p.d <= 4096 && p.heads > 0;
}

const OpEntry kOps[] = {
    {"eg2_saxpy", reinterpret_cast<const void*>(&eg2_saxpy), sizeof(EgSaxpy), Block::kAny, valid_saxpy},
    {"eg2_gather", reinterpret_cast<const void*>(&eg2_gather), sizeof(EgGather), Block::kAny, valid_gather},
    {"eg2_gather768", reinterpret_cast<const void*>(&eg2_gather768), sizeof(EgGather), Block::kAny, valid_gather},
    {"eg2_mm", reinterpret_cast<const void*>(&eg2_mm), sizeof(EgMM), Block::k256, valid_mm},
    {"eg2_mm64", reinterpret_cast<const void*>(&eg2_mm64), sizeof(EgMM), Block::k256, valid_mm},
    {"eg2_mm64x64", reinterpret_cast<const void*>(&eg2_mm64x64), sizeof(EgMM), Block::k256, valid_mm},
    {"eg2_mmstep8", reinterpret_cast<const void*>(&eg2_mmstep8), sizeof(EgMM), Block::k256, valid_mm},
    {"eg2_norm", reinterpret_cast<const void*>(&eg2_norm), sizeof(EgNorm), Block::k64, valid_norm},
    {"eg2_rope", reinterpret_cast<const void*>(&eg2_rope), sizeof(EgRope), Block::kAny, valid_rope},
    {"eg2_attention256", reinterpret_cast<const void*>(&eg2_attention256), sizeof(EgAttention), Block::k64,
     valid_attention, reinterpret_cast<const void*>(&attention_tile_kernel<256, 4, 512, 2>), 4},
    {"eg2_attention512", reinterpret_cast<const void*>(&eg2_attention512), sizeof(EgAttention), Block::k64,
     valid_attention, reinterpret_cast<const void*>(&attention_tile_kernel<512, 4, 512, 4>), 4},
    {"eg2_attention256x3", reinterpret_cast<const void*>(&eg2_attention256x3), sizeof(EgAttention), Block::k64,
     valid_attention, reinterpret_cast<const void*>(&attention_tile_kernel<256, 3, 256, 3>), 3},
    {"eg2_element", reinterpret_cast<const void*>(&eg2_element), sizeof(EgElement), Block::kAny, valid_element},
    {"eg2_pool", reinterpret_cast<const void*>(&eg2_pool), sizeof(EgPool), Block::kAny, valid_pool},
    {"eg2_norm_residual", reinterpret_cast<const void*>(&eg2_norm_residual), sizeof(EgNormResidual), Block::k64,
     valid_norm_residual},
    {"eg2_norm_rope", reinterpret_cast<const void*>(&eg2_norm_rope), sizeof(EgNormRope), Block::k64,
     valid_norm_rope},
};
constexpr unsigned kOpCount = sizeof(kOps) / sizeof(kOps[0]);

}  // namespace

extern "C" int eg2_op_launch(const char* name, const void* record, size_t record_size, unsigned grid_x,
                             unsigned grid_y, unsigned block, void* stream) {
  if (!name || !record || grid_x == 0 || grid_y == 0 || block == 0 || block > 1024) return (int)hipErrorInvalidValue;
  for (const OpEntry& op : kOps) {
    if (std::strcmp(op.name, name) != 0) continue;
    if (record_size != op.record_size) return (int)hipErrorInvalidValue;
    if ((op.block == Block::k64 && block != 64) || (op.block == Block::k256 && block != 256))
      return (int)hipErrorInvalidValue;
    if (!op.valid(record)) return (int)hipErrorInvalidValue;
    if (op.tile && grid_y == 1) {
      const EgAttention& p = as<EgAttention>(record);
      if (p.n >= kTileTokens && (uint64_t)op.heads * p.n == grid_x) {
        EgAttention rec = p;
        void* args[] = {&rec};
        return (int)hipLaunchKernel(op.tile, dim3((p.n + 15) / 16, op.heads), dim3(64 * kTileWaves), args, 0,
                                    reinterpret_cast<hipStream_t>(stream));
      }
    }
    // The kernarg segment is the record itself: copy it so the caller's
    // buffer may be reused as soon as this returns.
    alignas(16) unsigned char kernarg[64];
    std::memcpy(kernarg, record, record_size);
    if (op.fn == reinterpret_cast<const void*>(&eg2_saxpy)) {
      EgSaxpy s;
      std::memcpy(&s, kernarg, sizeof(s));
      void* args[] = {&s.y, &s.x, &s.a, &s.n};
      return (int)hipLaunchKernel(op.fn, dim3(grid_x, grid_y), dim3(block), args, 0,
                                  reinterpret_cast<hipStream_t>(stream));
    }
    void* args[] = {kernarg};
    return (int)hipLaunchKernel(op.fn, dim3(grid_x, grid_y), dim3(block), args, 0,
                                reinterpret_cast<hipStream_t>(stream));
  }
  return (int)hipErrorInvalidValue;
}

extern "C" unsigned eg2_op_count(void) { return kOpCount; }

extern "C" const char* eg2_op_name(unsigned index) { return index < kOpCount ? kOps[index].name : nullptr; }
