// Building blocks of the feature-split chain kernels (nerf_fused.hip,
// dlrm_fused.hip): a dense chain over a tile of 64 rows, for calls of fewer
// rows than the 256-row kernels need to fill the chip.
//
// The 256-row kernels give each of eight waves 32 rows and all features: no
// activation crosses a wave, but a call of 4,096 rows is 16 workgroups.  Here
// the eight waves split the features instead -- wave w computes features 32 w
// .. 32 w + 31 of every 256-wide layer for all 64 rows -- and hand their
// outputs on through LDS.  A wave then needs only its own eighth of a layer's
// weights, straight from L2 into registers about a layer ahead (14 fragments),
// and the LDS holds activations only: as finished B operands ("images": the 1
// KiB fragment of k-block kb and row block rb at ((kb RB) + rb) KiB, 16 bytes a
// lane), written by the wave that computed them and read by all, both without
// bank conflicts.  One barrier a layer.
//
// What bounds a tile: the weight feed (128 KiB a 256 x 256 layer at 64 bytes a
// clock and CU), the image reads (256 KiB at 128 bytes a clock) and the MFMAs
// (2 x 16 a wave) all take about 2,048 cycles a layer at 64 rows, which is why
// a tile has two row blocks: with one the feed alone binds, with four the
// image reads do.
//
// Measured (NeRF full chain, fp16, kernel time): up to 4,096 rows 53.9 -> 17.9
// us, 16,384 rows 56.6 -> 23.4, 32,768 rows 60.2 -> 42.9; at 65,536 rows the
// 256-row kernel is ahead, 73 against 82.  The B operands are read three
// k-blocks ahead of their MFMAs.
//
// Every accumulator adds the same MFMA products in the same order as in the
// 256-row kernels, from the same packed fragments: the results are the same
// bits.
#pragma once

#include <type_traits>
#include <utility>

#include "gp_device.hpp"

namespace gp {
namespace rows_split {

constexpr int RB = 2;           // 32-row blocks per tile
constexpr int ROWS = 32 * RB;   // rows per tile
constexpr int NW = 8;           // waves per workgroup, two per SIMD
constexpr int NT = NW * kWave;
constexpr int FRAG = 1024;      // one operand fragment: 64 lanes x 16 bytes

template <int... I, class F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

// 16-bit pair of an accumulator block with an optional ReLU: lo holds elements
// 0-7, hi 8-15 -- in the accumulator lane layout, the B operands of the next
// layer's k-blocks 2 fb and 2 fb + 1.  In bf16 the ReLU is a signed 16-bit
// integer max on the rounded bits (a bf16 value with its sign bit set becomes
// +0).
template <typename E>
__device__ __forceinline__ void to_operands(const f16x& a, bool relu, h8& lo, h8& hi) {
  if constexpr (std::is_same_v<E, F16>) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      lo[r] = (half_t)a[r];
      hi[r] = (half_t)a[8 + r];
    }
    if (relu) {
      lo = __builtin_elementwise_max(lo, h8{});
      hi = __builtin_elementwise_max(hi, h8{});
    }
  } else {
    lo = __builtin_shufflevector(E::cvt4(f4{a[0], a[1], a[2], a[3]}), E::cvt4(f4{a[4], a[5], a[6], a[7]}), 0, 1, 2, 3,
                                 4, 5, 6, 7);
    hi = __builtin_shufflevector(E::cvt4(f4{a[8], a[9], a[10], a[11]}), E::cvt4(f4{a[12], a[13], a[14], a[15]}), 0, 1,
                                 2, 3, 4, 5, 6, 7);
    if (relu) {
      lo = __builtin_bit_cast(h8, __builtin_elementwise_max(__builtin_bit_cast(s8, lo), s8{}));
      hi = __builtin_bit_cast(h8, __builtin_elementwise_max(__builtin_bit_cast(s8, hi), s8{}));
    }
  }
}

// Byte offset of the fragment of k-block kb, row block rb in an image.
__device__ __forceinline__ constexpr int img(int kb, int rb) { return (kb * RB + rb) * FRAG; }

__device__ __forceinline__ h8 img_read(GP_LDS const char* p) { return *(GP_LDS const h8*)p; }

__device__ __forceinline__ h8 load_frag(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// B operand of k-block kb for row `row` of a [rows][K] input behind descriptor
// r (rows K values long): columns 16 kb + 8 lh .. +7 in natural order, zero at
// and past column K and past the last row.
__device__ __forceinline__ h8 input_frag(__amdgpu_buffer_rsrc_t r, int row, int K, int kb, int lh) {
  const int c = 16 * kb + 8 * lh;
  const int n = min(max(K - c, 0), 8);  // valid columns of this lane's 8
  u32x4 w;
  if ((K & 7) == 0) {
    w = __builtin_amdgcn_raw_buffer_load_b128(r, (row * K + c) * 2, 0, 0);
  } else {
    unsigned short e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = __builtin_amdgcn_raw_buffer_load_b16(r, (row * K + c + i) * 2, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (unsigned)e[2 * i] | (unsigned)e[2 * i + 1] << 16;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] &= n >= 2 * i + 2 ? 0xffffffffu : n == 2 * i + 1 ? 0xffffu : 0u;
  return __builtin_bit_cast(h8, w);
}

}  // namespace rows_split
}  // namespace gp
