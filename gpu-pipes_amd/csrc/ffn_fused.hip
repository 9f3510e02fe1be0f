// The FFN blocks of the BERT apps at their width (H = 128, FF = 512) as one
// kernel each, and the packing of their weights:
//
//   bert_ffn        out = LN(act(x W1 + b1) W2 + b2 + x)
//                   (apps/bert_ffn/torch/model.py:3-14)
//   bert_addln_ffn  h0 = LN0(attn W0 + b0 + x),
//                   out = LN2(act(h0 W1 + b1) W2 + b2 + h0)
//                   (apps/bert_addln_ffn/torch/model.py:3-20)
//
// As GEMM launches with the LayerNorms in their epilogues these blocks move
// the 512-wide activations through memory and their K of 128 leaves each
// launch little but prologue and epilogue: three launches of 10 to 16 us for a
// block of 32,768 rows whose inputs and output are 25 MB.  Here a workgroup
// takes a tile of 32 rows through the whole block: four waves split the
// features as in rows_split.hpp, the activations pass through LDS as finished B
// operands (the fragment of k-block kb at kb KiB of an image), and the weights
// (288 KiB, packed once per call in the order they are consumed) stream from L2
// straight into registers.
//
//  * 128-wide layers: wave w computes feature block w; the 512-wide one:
//    blocks w, w + 4, w + 8 and w + 12.
//  * The images hold k in natural order: v_permlane32_swap turns a wave's
//    accumulator layout (four features, alternating between the wave halves)
//    into eight consecutive features a lane, which is the B operand layout and
//    the layout of a row in memory at once.
//  * LayerNorm: one wave reads the 16-bit rows back from their image, a row in
//    two lanes, sums in the order of the GEMM epilogue (gemm.hip) and writes the
//    normalised rows to the next image or to memory.
// Products, biases, residuals and statistics are added in the GEMM chain's
// order, so results agree with it bit for bit.
//
// What bounds it: one tile is a serial chain (six barriers, two LayerNorms of a
// few hundred dependent instructions on one wave, about 2 us of its 6), so two
// workgroups share a CU and one's LayerNorm runs under the other's MFMAs; which
// wave computes it rotates with the workgroup, since wave w of every workgroup
// sits on one SIMD.  With the weights left in registers (wrong results) 16,384
// rows take 13.5 instead of 15.2 us, so the feed is not it.  Kernel time of
// bert_addln_ffn (fp16, ReLU): 100 rows 8.2 us, 16,384 rows 13.9, 32,768 rows
// 21.6.  It is the faster way at large row counts too; us a call with the packing
// launch, this kernel / the chain of GEMM launches (fp16):
//   rows         FFN ReLU       FFN GELU       add + LN + FFN, ReLU / GELU
//      32,768    19.9 / 31.3    21.1 / 31.8    24.1 / 41.1    26.5 / 42.0
//     131,072    60.6 / 90.7    70.2 / 95.8    78.3 /  174    90.0 /  183
//     300,000     131 /  245                    174 /  320
//   1,048,576     460 /  763     581 /  831     601 / 1147     737 / 1241  Tried and
// slower at 32,768 rows: three workgroups a CU with half the weights in flight
// (23.4), eight waves on 64 rows (24.8).
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "../../include/gpipes.h"
#include "gp_device.hpp"
#include "gp_kernels.hpp"
#include "rows_split.hpp"
#include "stages.hpp"

namespace gp {
namespace ffn128 {

using rows_split::img_read;
using rows_split::load_frag;
using rows_split::static_for;
constexpr int NW = 4, NT = NW * kWave;  // waves per workgroup, one per SIMD
constexpr int ROWS = 32, FRAG = rows_split::FRAG;
constexpr int H = 128, FF = 512;
constexpr int KBH = H / 16, KBF = FF / 16, FBH = H / 32, FBF = FF / 32;  // k-blocks, feature blocks
constexpr int NF = FBF / NW;  // feature blocks per wave of the 512-wide layer
static_assert(FBH == NW, "one feature block per wave of a 128-wide layer");
constexpr int LB = 3;  // B operands are read from LDS this many k-blocks ahead
// Packed weights: fragment (kb, fb) of a layer at its base + (kb FB + fb) FRAG.
constexpr int O_W0 = 0, O_W1 = O_W0 + KBH * FBH * FRAG, O_W2 = O_W1 + KBH * FBF * FRAG,
              PACK_BYTES = O_W2 + KBF * FBH * FRAG;

struct Args {
  const half_t* a;     // [M][128]: attn (ADDLN) or x
  const half_t* x;     // [M][128]: residual of the first LayerNorm (ADDLN)
  const char* pack;    // PACK_BYTES
  const half_t *b0, *b1, *b2;              // biases or null
  const half_t *ga0, *be0, *ga2, *be2;     // LayerNorm affines or null (1 / 0)
  half_t* out;         // [M][128]
  int64_t M;
  float eps;
};

template <typename E, int ACT, bool ADDLN>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void ffn_kernel(Args p) {
  // Streamed fragments per wave and tile: first layer (ADDLN), 128 -> 512, 512 -> 128.
  constexpr int J1 = ADDLN ? KBH : 0, J2 = J1 + NF * KBH, T = J2 + KBF;
  constexpr int PF = ADDLN ? 24 : 16;  // fragments in flight per wave
  static_assert(T % PF == 0, "a tile's first fragment takes register set 0");
  // LDS: image S (attn, then the rows before the last LayerNorm), image H (the
  // FFN's input), image F (512 wide; first the rows before LN0), then the
  // vectors ga0, be0, ga2, be2, b0, b2 and b1.
  constexpr int L_S = 0, L_H = KBH * FRAG, L_F = 2 * KBH * FRAG, L_P = L_F + KBF * FRAG, L_B1 = L_P + 6 * H * 2;
  __shared__ __attribute__((aligned(1024))) char smem[L_B1 + FF * 2];

  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool ln_wave = wave == (int)(blockIdx.x & (NW - 1));
  GP_LDS char* const lds = (GP_LDS char*)smem;
  GP_LDS char* const mine = lds + 16 * lane;
  const int ntiles = (int)((p.M + ROWS - 1) / ROWS);

  const __amdgpu_buffer_rsrc_t rp = make_rsrc(p.pack, PACK_BYTES), none = make_rsrc(p.pack, 0);
  const int vw = 16 * lane + wave * FRAG;
  h8 wf[PF];
  auto fetch = [&](auto jc, __amdgpu_buffer_rsrc_t r) {
    constexpr int j = decltype(jc)::value;
    constexpr int off = j < J1   ? O_W0 + j * FBH * FRAG
                        : j < J2 ? O_W1 + ((j - J1) % KBH * FBF + (j - J1) / KBH * NW) * FRAG
                                 : O_W2 + (j - J2) * FBH * FRAG;
    wf[j % PF] = load_frag(r, vw, off);
  };
  // Elements 4 g .. 4 g + 3 of feature block fb of an LDS vector, as this lane's
  // accumulators hold them (feature 32 fb + 8 g + 4 lh + e).
  auto vec = [&](int base, int fb, int g) { return *(GP_LDS const h4*)(lds + base + (32 * fb + 8 * g + 4 * lh) * 2); };

  // Input fragments of a tile: k-blocks w and w + 4; with ADDLN also this
  // lane's residual values.
  h8 in[2];
  h4 res[4];
  auto load_tile = [&](int t) {
    const int64_t r0 = (int64_t)t * ROWS;
    const int64_t left = t < ntiles ? p.M - r0 : 0;
    const int rows = left < ROWS ? (int)left : ROWS;
    const int64_t base = t < ntiles ? r0 * H : 0;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a + base, rows * H * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) in[i] = load_frag(ra, (lr * H + 16 * (wave + NW * i) + 8 * lh) * 2, 0);
    if constexpr (ADDLN) {
      const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x + base, rows * H * 2);
#pragma unroll
      for (int g = 0; g < 4; ++g) res[g] = buf_load_h4(rx, (lr * H + 32 * wave + 8 * g + 4 * lh) * 2);
    }
  };

  // Accumulator block as 16-bit values o[g] (features 8 g + 4 lh ..) into
  // k-blocks 2 f, 2 f + 1 of the image at `base`.
  auto to_image = [&](const h4 (&o)[4], int base, int f) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const u32x2 u = __builtin_bit_cast(u32x2, o[2 * q]), v = __builtin_bit_cast(u32x2, o[2 * q + 1]);
      const auto x = __builtin_amdgcn_permlane32_swap(u[0], v[0], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(u[1], v[1], false, false);
      *(GP_LDS u32x4*)(mine + base + (2 * f + q) * FRAG) =
          u32x4{(unsigned)x[0], (unsigned)y[0], (unsigned)x[1], (unsigned)y[1]};
    }
  };
  // LayerNorm of the rows in image `src` (one wave); affine pair i of the LDS
  // vectors; each normalised 16-byte chunk goes to put(c, w).  The 16-bit
  // values are read as they are by v_fma_mix_f32: fma(x, one, y) with a `one`
  // the compiler cannot see stays an fma and rounds x + y once.
  float one = 1.f;
  asm volatile("" : "+v"(one));
  auto layer_norm = [&](int src, int i, auto put) {
    h8 v[KBH];  // features 16 c + 4 lh + (0..3), 16 c + 8 + 4 lh + (0..3)
#pragma unroll
    for (int c = 0; c < KBH; ++c) {
      const u32x4 w = *(GP_LDS const u32x4*)(mine + src + c * FRAG);
      const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      v[c] = __builtin_bit_cast(h8, u32x4{(unsigned)x[0], (unsigned)y[0], (unsigned)x[1], (unsigned)y[1]});
    }
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int c = 0; c < KBH; ++c)
#pragma unroll
      for (int k = 0; k < 8; ++k) s = __builtin_fmaf(E::val(v[c][k]), one, s);
    const float mean = sum_lane_halves(s) * (1.f / H);
#pragma unroll
    for (int c = 0; c < KBH; ++c)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float d = __builtin_fmaf(E::val(v[c][k]), one, -mean);
        q = __builtin_fmaf(d, d, q);
      }
    const float rstd = rsqrtf(sum_lane_halves(q) * (1.f / H) + p.eps);
    GP_LDS const char* const ga = lds + L_P + 2 * i * H * 2 + 8 * lh;
    GP_LDS const char* const be = ga + H * 2;
#pragma unroll
    for (int c = 0; c < KBH; ++c) {
      u32x2 o[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const h4 g4 = *(GP_LDS const h4*)(ga + (16 * c + 8 * hh) * 2), b4 = *(GP_LDS const h4*)(be + (16 * c + 8 * hh) * 2);
        f4 z;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          z[e] = __builtin_fmaf(__builtin_fmaf(E::val(v[c][4 * hh + e]), one, -mean) * rstd, E::val(g4[e]), E::val(b4[e]));
        o[hh] = __builtin_bit_cast(u32x2, E::cvt4(z));
      }
      const auto x = __builtin_amdgcn_permlane32_swap(o[0][0], o[1][0], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(o[0][1], o[1][1], false, false);
      put(c, u32x4{(unsigned)x[0], (unsigned)y[0], (unsigned)x[1], (unsigned)y[1]});
    }
  };

  // The first tile's inputs, the first weights and the vectors: everything is
  // requested before anything is waited for.
  load_tile(blockIdx.x);
  static_for(std::make_integer_sequence<int, PF>{}, [&](auto j) { fetch(j, rp); });
  {
    // (An absent vector is read through an empty descriptor: zeros.)
    const half_t one16 = __builtin_bit_cast(half_t, E::kOne);
    auto load = [&](const half_t* v, int n, int i) {
      return __builtin_bit_cast(
          half_t, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(make_rsrc(v ? v : p.out, v ? n * 2 : 0), i * 2, 0, 0));
    };
    const int f = threadIdx.x & (H - 1), odd = wave >> 1;  // 256 threads: two vectors of 128 at a time
    half_t v[3], w[FF / NT];
    v[0] = load(odd ? p.be0 : p.ga0, H, f);
    v[1] = load(odd ? p.be2 : p.ga2, H, f);
    v[2] = load(odd ? p.b2 : p.b0, H, f);
#pragma unroll
    for (int i = 0; i < FF / NT; ++i) w[i] = load(p.b1, FF, threadIdx.x + i * NT);
    if (!odd && !p.ga0) v[0] = one16;
    if (!odd && !p.ga2) v[1] = one16;
#pragma unroll
    for (int i = 0; i < 3; ++i) *(GP_LDS half_t*)(lds + L_P + ((2 * i + odd) * H + f) * 2) = v[i];
#pragma unroll
    for (int i = 0; i < FF / NT; ++i) *(GP_LDS half_t*)(lds + L_B1 + (threadIdx.x + i * NT) * 2) = w[i];
  }

  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int64_t r0 = (int64_t)t * ROWS;
    const int vrows = p.M - r0 < ROWS ? (int)(p.M - r0) : ROWS;
    // Past the last tile the next tile's fragments come through an empty
    // descriptor.
    const __amdgpu_buffer_rsrc_t rnext = t + (int)gridDim.x < ntiles ? rp : none;
    // W . B over fragments J0 .. J0 + KB - 1 and the image at `base`; each
    // register set is refilled with the fragment PF further on.
    auto mmas = [&](auto j0c, auto kbc, int base) {
      constexpr int J0 = decltype(j0c)::value, KB = decltype(kbc)::value;
      f16x acc = {};
      h8 x[LB];
      static_for(std::make_integer_sequence<int, LB>{}, [&](auto kc) { x[kc] = img_read(mine + base + kc * FRAG); });
      static_for(std::make_integer_sequence<int, KB>{}, [&](auto kc) {
        constexpr int kb = decltype(kc)::value, j = J0 + kb;
        acc = E::mma(wf[j % PF], x[kb % LB], acc);
        fetch(std::integral_constant<int, (j + PF) % T>{}, j + PF < T ? rp : rnext);
        if constexpr (kb + LB < KB) x[kb % LB] = img_read(mine + base + (kb + LB) * FRAG);
        __builtin_amdgcn_sched_barrier(0);
      });
      return acc;
    };
    using KH = std::integral_constant<int, KBH>;
    using KF = std::integral_constant<int, KBF>;

#pragma unroll
    for (int i = 0; i < 2; ++i) *(GP_LDS h8*)(mine + (ADDLN ? L_S : L_H) + (wave + NW * i) * FRAG) = in[i];
    lds_barrier();
    if constexpr (ADDLN) {
      const f16x acc = mmas(std::integral_constant<int, 0>{}, KH{}, L_S);
      h4 o[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const h4 b = vec(L_P + 4 * H * 2, wave, g);
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[4 * g + e] + E::val(b[e]) + E::val(res[g][e]);
        o[g] = E::cvt4(v);
      }
      to_image(o, L_F, wave);
      lds_barrier();
      if (ln_wave) layer_norm(L_F, 0, [&](int c, u32x4 w) { *(GP_LDS u32x4*)(mine + L_H + c * FRAG) = w; });
      lds_barrier();
    }
    load_tile(t + gridDim.x);  // the next tile's inputs, over the rest of this one
    // 128 -> 512
    static_for(std::make_integer_sequence<int, NF>{}, [&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const f16x acc = mmas(std::integral_constant<int, J1 + i * KBH>{}, KH{}, L_H);
      h4 o[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const h4 b = vec(L_B1, wave + NW * i, g);
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = apply_act(acc[4 * g + e] + E::val(b[e]), ACT);
        o[g] = E::cvt4(v);
      }
      to_image(o, L_F, wave + NW * i);
    });
    lds_barrier();
    // 512 -> 128, residual from the FFN's input image
    {
      const f16x acc = mmas(std::integral_constant<int, J2>{}, KF{}, L_F);
      h4 o[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const h4 b = vec(L_P + 5 * H * 2, wave, g);
        const h4 r = *(GP_LDS const h4*)(lds + L_H + (2 * wave + (g >> 1)) * FRAG + (lr + 32 * (g & 1)) * 16 + 8 * lh);
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[4 * g + e] + E::val(b[e]) + E::val(r[e]);
        o[g] = E::cvt4(v);
      }
      to_image(o, L_S, wave);
    }
    lds_barrier();
    if (ln_wave) {
      const __amdgpu_buffer_rsrc_t ro = make_rsrc(p.out + r0 * H, vrows * H * 2);
      layer_norm(L_S, 1, [&](int c, u32x4 w) { buf_store_u4(ro, (lr * H + 16 * c + 8 * lh) * 2, w); });
    }
    // The next tile's attn overwrites image S: the LayerNorm wave first.
    if constexpr (ADDLN) lds_barrier();
  }
  wait_vmcnt<0>();  // the fragments fetched past the last tile
}

struct PackArgs {
  const half_t *w0, *w1, *w2;  // [128][128] (null: left out), [128][512], [512][128]
  char* pack;
};

// One thread per 16-byte lane chunk of a fragment: W[16 kb + 8 h + e][32 fb + i]
// for lane (i, h).  A block lies within one matrix.
__global__ __launch_bounds__(256) void ffn_pack_kernel(PackArgs a) {
  const int gid = blockIdx.x * 256 + threadIdx.x + (a.w0 ? 0 : O_W1 / 16);
  const int f = gid / kWave, lane = gid % kWave;
  constexpr int F1 = O_W1 / FRAG, F2 = O_W2 / FRAG;
  const bool one = f >= F1 && f < F2;
  const half_t* const w = f < F1 ? a.w0 : one ? a.w1 : a.w2;
  const int fi = f - (f < F1 ? 0 : one ? F1 : F2), FB = one ? FBF : FBH, n = one ? FF : H;
  const int kb = fi / FB, fb = fi % FB;
  const half_t* const src = w + (int64_t)(16 * kb + 8 * (lane >> 5)) * n + 32 * fb + (lane & 31);
  h8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = src[e * n];
  *(h8*)(a.pack + (size_t)gid * 16) = v;
}

template <typename E, bool ADDLN>
static hipError_t launch(const Args& a, int act, int grid, hipStream_t s) {
  switch (act) {
    case ACT_NONE: hipLaunchKernelGGL((ffn_kernel<E, ACT_NONE, ADDLN>), dim3(grid), dim3(NT), 0, s, a); break;
    case ACT_RELU: hipLaunchKernelGGL((ffn_kernel<E, ACT_RELU, ADDLN>), dim3(grid), dim3(NT), 0, s, a); break;
    case ACT_GELU_TANH: hipLaunchKernelGGL((ffn_kernel<E, ACT_GELU_TANH, ADDLN>), dim3(grid), dim3(NT), 0, s, a); break;
    case ACT_SIGMOID: hipLaunchKernelGGL((ffn_kernel<E, ACT_SIGMOID, ADDLN>), dim3(grid), dim3(NT), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace ffn128

size_t ffn_fused_workspace() { return ffn128::PACK_BYTES; }

hipError_t ffn_fused_launch(const BertAddlnArgs& f, void* ws, int num_cus, hipStream_t s, int dtype) {
  using namespace ffn128;
  if (!ffn_fused_supported(f.H, f.FF) || f.M <= 0 || f.M > (int64_t(1) << 31) - 1) return hipErrorInvalidValue;
  const bool addln = f.w0 != nullptr;
  const PackArgs pa{(const half_t*)f.w0, (const half_t*)f.w1, (const half_t*)f.w2, (char*)ws};
  hipLaunchKernelGGL(ffn_pack_kernel, dim3((PACK_BYTES - (addln ? 0 : O_W1)) / 16 / 256), dim3(256), 0, s, pa);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  const Args a{(const half_t*)f.attn, (const half_t*)f.x, (const char*)ws, (const half_t*)f.b0, (const half_t*)f.b1,
               (const half_t*)f.b2, (const half_t*)f.ga0, (const half_t*)f.be0, (const half_t*)f.ga2,
               (const half_t*)f.be2, (half_t*)f.out, f.M, f.eps};
  const int64_t tiles = (f.M + ROWS - 1) / ROWS;
  const int64_t slots = (int64_t)num_cus * 2;
  const int grid = (int)(tiles < slots ? tiles : slots);
  if (dtype == GP_DTYPE_BF16)
    return addln ? launch<BF16, true>(a, f.act, grid, s) : launch<BF16, false>(a, f.act, grid, s);
  return addln ? launch<F16, true>(a, f.act, grid, s) : launch<F16, false>(a, f.act, grid, s);
}

}  // namespace gp
