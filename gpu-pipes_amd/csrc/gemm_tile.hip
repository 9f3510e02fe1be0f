// Small-tile form of the wide GEMM stage (gemm.hip), for calls whose 256-row
// tiles would leave most of the chip idle:
//
//   C[M][N] = act(A[M][K] . B[K][N] + bias[N]) (+ R[M][N])      fp32 accumulate
//
// and the LayerNorm over finished rows that follows such a GEMM.
//
// What bounds it: with few rows the chip is filled by tiles, not by work per
// tile, so a launch takes about as long as one tile's walk over K, and that
// walk is a serial chain of one wave per SIMD: barrier, fragment reads, MFMAs,
// copy issue.  So a workgroup owns one small tile (64 x 64 or 128 x 128),
// nothing is persistent, the next slab's fragments are read while this slab's
// MFMAs run, and the loop is unrolled over the four ring slots, which leaves
// about 45 instructions a slab at 64 x 64 (75 with the slot in a register:
// 0.21 against 0.27 us a slab).  A ring of nine slabs ahead instead of three
// changed nothing.  Two workgroups share a CU (64 KiB of LDS each), one's waits
// under the other's MFMAs: at 128 x 128 that takes slabs of 32 k, and beats one
// workgroup with slabs of 64 on every shape measured (2048 x 4096 x 1024 27.1
// -> 23.6 us, 4096 x 1024 x 4096 40.4 -> 39.0).  A 256 x 128 tile of 32-k slabs,
// two a CU, was behind the persistent kernel where that one fills the chip and
// behind 128 x 128 where it does not.  Measured, 509 x 1024 x 4096 (fp16): 82 us on the
// persistent kernel's 8 tiles, 16.3 on 128 tiles of 64 x 64; the calls
// bert_ffn 509 x 1024 x 4096 134 -> 33 us, DLRM bottom + top at 2,048 rows 118
// -> 69 us.
//
// Every accumulator adds the same MFMA products in the same order as the
// persistent kernel's (32x32x16, k ascending from zero, bias added last), so a
// row's result does not depend on which kernel computed it: small batches are
// bit-identical to the same rows of large ones.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "../../include/gpipes.h"
#include "gemm_common.hpp"

namespace gp {
namespace gemm {
namespace tile {

constexpr int NW = 4;  // waves per workgroup
constexpr int NT = NW * kWave;

template <int... I, class F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int NB, int BK_, int NS_, int OCC_>
struct Cfg {
  static constexpr int NBW = NB, MBW = NB, WN = 2, WM = 2;       // 32-feature / 32-row blocks per wave, waves
  static constexpr int BN = 32 * NBW * WN, BM = 32 * MBW * WM;   // features and rows per tile
  static constexpr int BK = BK_, KS = BK / 16;                   // k and MFMA steps per slab
  static constexpr int ROWB = 2 * BK, CPR = ROWB / 16, RPC = 64 / CPR;  // bytes and chunks of a slab row, rows per copy
  static constexpr int NS = NS_;                                 // slabs in the LDS ring
  static constexpr int OCC = OCC_;                               // workgroups per CU
  static constexpr int ABYTES = BM * ROWB, BBYTES = BN * ROWB;   // bytes of a slab's A and B part
  static constexpr int STAGE = ABYTES + BBYTES;
  static constexpr int UA = ABYTES / 1024 / NW, UB = BBYTES / 1024 / NW;  // copies per wave of each part
  static_assert(UA * 1024 * NW == ABYTES && UB * 1024 * NW == BBYTES, "copy split must be uniform per wave");
  static_assert(NS >= 3 && OCC * NS * STAGE <= 160 * 1024, "LDS");
  static_assert((NS - 1) * (UA + UB) <= 63, "copies in flight exceed the counter field");
};
using T64 = Cfg<1, 64, 4, 2>;
using T128 = Cfg<2, 32, 4, 2>;

// Byte offset of 16-byte chunk c of row r in an operand slab of ROWB-byte rows:
// XOR-swizzled so that 16 consecutive rows read at one chunk cover all of the
// 16-byte bank groups (128-byte rows: unit_off; 64-byte rows lie four to a
// 256-byte bank window).
template <class C>
__device__ __forceinline__ int row_swz(int r) {
  return C::ROWB == 128 ? (r >> 1) & 7 : (r >> 2) & 3;
}
template <class C>
__device__ __forceinline__ int row_off(int r, int c) {
  return r * C::ROWB + ((c ^ row_swz<C>(r)) << 4);
}

// Chunk swizzle of row r of a weight slab kept in its own [k][feature] layout
// (16-byte chunks; BN = 64: eight to a row, two rows to a 256-byte bank
// window; BN = 128: sixteen, one row): the four rows that a transposing read
// takes 64 bytes from fall into four different quarters of the window.
template <int BN>
__host__ __device__ constexpr int brow_swz(int r) {
  return BN == 64 ? 4 * ((r >> 1) & 1) : 4 * (r & 3);
}

// BROW: the weights are read in their own [K][N] layout (see gemm.hip).
template <class C, int ACT, bool RESID, bool BROW, typename E>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(C::OCC, C::OCC))) void tile_kernel(Args p) {
  __shared__ __attribute__((aligned(1024))) char ring[C::NS * C::STAGE];
  constexpr int NS = C::NS, CPS = C::UA + C::UB;  // ring slabs, copies per wave and slab
  constexpr int BK = C::BK, KS = C::KS, ROWB = C::ROWB, CPR = C::CPR, RPC = C::RPC;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int lr = lane & 31, lh = lane >> 5;
  const int wn = wave % C::WN, wm = wave / C::WN;
  const int K = p.K;
  const int nslab = K / BK;

  // Workgroup b is taken to run on XCD b % 8; each XCD gets a contiguous range
  // of the tile list.  The list runs along the dimension with fewer operand
  // bytes first (rows when M < N), so that an XCD's L2 holds an eighth of the
  // larger operand and all of the smaller.
  const int tiles_n = p.N / C::BN;
  const int tiles_m = (int)((p.M + C::BM - 1) / C::BM);
  const int ntiles = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7, wid = blockIdx.x >> 3;
  const int lo = (int)((int64_t)ntiles * xcd / 8), hi = (int)((int64_t)ntiles * (xcd + 1) / 8);
  const int t = lo + wid;
  if (t >= hi) return;
  int tn, tm;
  if (p.M < p.N) {
    tn = t / tiles_m;
    tm = t - tn * tiles_m;
  } else {
    tm = t / tiles_n;
    tn = t - tm * tiles_n;
  }
  const int n0 = tn * C::BN;
  const int64_t m0 = (int64_t)tm * C::BM;
  const int64_t left = p.M - m0;
  const int rows = (int)(left < C::BM ? left : C::BM);

  // Copies.  A (and a transposed weight slab): copy j of a wave fills rows
  // 8 (NW j + wave) + lane / 8 of the part at chunk position lane % 8, which
  // holds the logical chunk that the unit_off swizzle maps there; rows of
  // consecutive j are 32 apart, which leaves the swizzle unchanged.  A weight
  // slab in its own layout: 64 rows of BN features, RB rows to a copy.
  const int vrow = RPC * wave + lane / CPR;
  const int vswz = ((lane % CPR) ^ row_swz<C>(vrow)) << 4;
  const int voffa = vrow * p.lda * 2 + vswz;
  constexpr int CB = C::BN / 8, RB = 64 / CB;
  const int rq = RB * wave + lane / CB;
  static_assert(brow_swz<C::BN>(RB * NW) == brow_swz<C::BN>(0), "copies of one lane share a swizzle");
  const int voffb = BROW ? rq * p.ldw * 2 + (((lane % CB) ^ brow_swz<C::BN>(rq)) << 4) : vrow * K * 2 + vswz;
  const int lck = (vswz >> 4) * 8;      // the lane's first column within an A slab
  constexpr int kBeyond = 0x40000000;   // past every descriptor's range: the copy writes zeros
  const int jstra = RPC * NW * p.lda * 2, jstrb = BROW ? RB * NW * p.ldw * 2 : RPC * NW * K * 2;
  const int slabb = BROW ? BK * p.ldw * 2 : ROWB;
  const half_t* const abase = p.a + m0 * p.lda;
  const half_t* const bbase = BROW ? p.w + n0 : p.bt + (int64_t)n0 * K;
  const int abytes = rows * p.lda * 2;
  const int bbytes = BROW ? (int)((int64_t)p.kw * p.ldw * 2 - (int64_t)n0 * 2) : C::BN * K * 2;
  GP_LDS char* const lds = (GP_LDS char*)ring + wave * 1024;
  // Slab kt into ring slot s.  Past the last slab the descriptors are empty:
  // the copies touch no memory and zero a dead slot, so that every wait below
  // finds the same number of copies in flight.
  auto issue = [&](int kt, int s) {
    const bool in = kt < nslab;
    const __amdgpu_buffer_rsrc_t da = make_rsrc(abase, in ? abytes : 0), db = make_rsrc(bbase, in ? bbytes : 0);
    const int k0 = kt * BK;
    const int vo = k0 + BK <= p.ka || k0 + lck < p.ka ? voffa : kBeyond;
    const int sob = kt * slabb, soa = kt * ROWB;
#pragma unroll
    for (int j = 0; j < C::UB; ++j)
      dma16_buf_so(db, voffb, j * jstrb + sob, lds + s * C::STAGE + C::ABYTES + j * NW * 1024);
#pragma unroll
    for (int j = 0; j < C::UA; ++j) dma16_buf_so(da, vo, j * jstra + soa, lds + s * C::STAGE + j * NW * 1024);
  };

  // Fragment addresses (see gemm.hip): row blocks 32 apart share the swizzle.
  const int frow = 32 * C::NBW * wn + lr, arow = 32 * C::MBW * wm + lr;
  int lb[C::NBW];
#pragma unroll
  for (int nb = 0; nb < C::NBW; ++nb) {
    const int m = lane & 15, r4 = m >> 2;
    const int f = 32 * (C::NBW * wn + nb) + 16 * ((lane >> 4) & 1) + 4 * (m & 3);
    lb[nb] = (8 * lh + r4) * (C::BN * 2) + (((f >> 3) ^ brow_swz<C::BN>(r4)) << 4) + (f & 7) * 2;
  }

  // Bias and residual of this lane's outputs (see the epilogue), requested
  // before the first copies, so that the wait for slab 0 covers them.
  const __amdgpu_buffer_rsrc_t rr = make_rsrc(RESID ? p.r + m0 * p.ldr : p.c, RESID ? rows * p.ldr * 2 : 0);
  h4 bias[C::NBW][4], res[RESID ? C::NBW : 1][C::MBW][4];
#pragma unroll
  for (int nb = 0; nb < C::NBW; ++nb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int col = n0 + 32 * (C::NBW * wn + nb) + 8 * g + 4 * lh;
      bias[nb][g] = p.bias ? *(const h4*)(p.bias + col) : h4{};
      if constexpr (RESID) {
#pragma unroll
        for (int mb = 0; mb < C::MBW; ++mb) res[nb][mb][g] = buf_load_h4(rr, ((arow + 32 * mb) * p.ldr + col) * 2);
      }
    }

  // Operand fragments of one slab, in two register sets: slab kt + 1 is read
  // while slab kt's MFMAs run, so neither the LDS latency nor the barrier
  // stands between two slabs' products.
  struct Frags {
    h8 a[KS][C::NBW], b[KS][C::MBW];
  };
  Frags f[2];
  // Per-lane addresses in slot 0; a slot is a constant offset away (the loop
  // below is unrolled over the slots, so the reads need no address arithmetic).
  GP_LDS const char* pa[KS];
  GP_LDS const char* pb[BROW ? C::NBW : KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    pa[ks] = (GP_LDS const char*)ring + row_off<C>(arow, 2 * ks + lh);
    if constexpr (!BROW) pb[ks] = (GP_LDS const char*)ring + C::ABYTES + row_off<C>(frow, 2 * ks + lh);
  }
  if constexpr (BROW) {
#pragma unroll
    for (int nb = 0; nb < C::NBW; ++nb) pb[nb] = (GP_LDS const char*)ring + C::ABYTES + lb[nb];
  }
  auto load = [&](Frags& q, int s) {
    const int o = s * C::STAGE;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int nb = 0; nb < C::NBW; ++nb) {
        if constexpr (BROW) {
          GP_LDS const char* const w = pb[nb] + (o + ks * 16 * (C::BN * 2));
          q.a[ks][nb] = __builtin_bit_cast(
              h8, __builtin_shufflevector(lds_tr16(w), lds_tr16(w + 4 * (C::BN * 2)), 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
          q.a[ks][nb] = *(GP_LDS const h8*)(pb[ks] + (o + 32 * nb * ROWB));
        }
      }
#pragma unroll
      for (int mb = 0; mb < C::MBW; ++mb) q.b[ks][mb] = *(GP_LDS const h8*)(pa[ks] + (o + 32 * mb * ROWB));
    }
  };

  f16x acc[C::NBW][C::MBW];
#pragma unroll
  for (int nb = 0; nb < C::NBW; ++nb)
#pragma unroll
    for (int mb = 0; mb < C::MBW; ++mb) acc[nb][mb] = f16x{};

#pragma unroll
  for (int i = 0; i < NS; ++i) issue(i, i);
  wait_vmcnt<(NS - 1) * CPS>();
  lds_barrier();
  load(f[0], 0);
  // Slab kt, which lives in ring slot kt % NS and register set kt % 2; U is kt
  // modulo the unrolling, a multiple of both.
  constexpr int UNROLL = NS % 2 ? 2 * NS : NS;
  auto step = [&](int kt, auto uc) {
    constexpr int U = decltype(uc)::value, S = U % NS, S1 = (U + 1) % NS;
    // This wave's copies of slab kt + 1 have landed once at most the NS - 2
    // slabs issued after it are in flight; past the barrier every wave's have,
    // and every wave holds slab kt in registers, so its slot takes slab kt + NS.
    wait_vmcnt<(NS - 2) * CPS>();
    lds_barrier();
    load(f[(U + 1) % 2], S1);
    issue(kt + NS, S);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nb = 0; nb < C::NBW; ++nb)
#pragma unroll
        for (int mb = 0; mb < C::MBW; ++mb) acc[nb][mb] = E::mma(f[U % 2].a[ks][nb], f[U % 2].b[ks][mb], acc[nb][mb]);
  };
  for (int kt = 0; kt < nslab; kt += UNROLL)
    static_for(std::make_integer_sequence<int, UNROLL>{}, [&](auto uc) {
      if (uc == 0 || kt + uc < nslab) step(kt + uc, uc);
    });

  // Epilogue: lane (lr, lh) holds, in elements 4 g + e of block (nb, mb), row
  // arow + 32 mb and feature n0 + 32 (NBW wn + nb) + 8 g + 4 lh + e.  The
  // exchange of feature groups between the wave halves and the 16-byte stores
  // are the persistent kernel's.
  const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.c + m0 * p.ldc, rows * p.ldc * 2);
#pragma unroll
  for (int nb = 0; nb < C::NBW; ++nb) {
    const int col = n0 + 32 * (C::NBW * wn + nb);
#pragma unroll
    for (int mb = 0; mb < C::MBW; ++mb) {
      u32x2 o[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = apply_act(acc[nb][mb][4 * g + e] + E::val(bias[nb][g][e]), ACT);
          if constexpr (RESID) v[e] += E::val(res[nb][mb][g][e]);
        }
        o[g] = __builtin_bit_cast(u32x2, E::cvt4(v));
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const auto x = __builtin_amdgcn_permlane32_swap(o[2 * q][0], o[2 * q + 1][0], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(o[2 * q][1], o[2 * q + 1][1], false, false);
        const u32x4 w = {(unsigned)x[0], (unsigned)y[0], (unsigned)x[1], (unsigned)y[1]};
        buf_store_u4(rc, ((arow + 32 * mb) * p.ldc + col + 16 * q + 8 * lh) * 2, w);
      }
    }
  }
  wait_vmcnt<0>();  // the empty copies past the last slab have landed before the waves exit
}

// LayerNorm of finished rows, with the statistics of the GEMM's LayerNorm
// epilogue (gemm.hip) bit for bit: per 128 features two lanes sum 64 values
// each in the epilogue's order (feature groups of four alternate between
// them), mean and M2 of the 128, then the N / 128 partials combined in order.
// A pair of lanes loads whole 16-byte chunks and trades halves; a row is N /
// 64 lanes.  In place when out == x: a row is read whole before it is written.
template <int N, typename E>
__global__ __launch_bounds__(256) void ln_rows_kernel(const half_t* x, const half_t* gamma, const half_t* beta,
                                                      float eps, half_t* out, int64_t M) {
  constexpr int P = N / 128, LPR = 2 * P, RPW = kWave / LPR;
  const int lane = threadIdx.x & 63;
  const int lh = lane & 1, g = (lane % LPR) >> 1;
  const int64_t row = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + lane / LPR;
  const bool ok = row < M;
  // Trades halves between the lanes of a pair: chunk c (lane 0) and c + 1
  // (lane 1) in, the lower (upper) four features of both out, and back.
  auto trade = [&](u32x4 v) {
    const u32x2 keep = lh ? u32x2{v[2], v[3]} : u32x2{v[0], v[1]};
    const u32x2 give = lh ? u32x2{v[0], v[1]} : u32x2{v[2], v[3]};
    u32x2 got;
#pragma unroll
    for (int i = 0; i < 2; ++i) got[i] = (unsigned)__builtin_amdgcn_mov_dpp((int)give[i], 0xB1, 0xF, 0xF, false);
    return lh ? u32x4{got[0], got[1], keep[0], keep[1]} : u32x4{keep[0], keep[1], got[0], got[1]};
  };
  const half_t* const xr = x + (ok ? row : 0) * N + 128 * g;
  h8 v[8];  // [chunk pair c]: features 16 c + 4 lh + (0..3) and 16 c + 8 + 4 lh + (0..3) of the 128
#pragma unroll
  for (int c = 0; c < 8; ++c) v[c] = __builtin_bit_cast(h8, trade(*(const u32x4*)(xr + 16 * c + 8 * lh)));
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += E::val(v[c][e]);
  auto pair_sum = [](float a) {
    return a + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0xB1, 0xF, 0xF, false));
  };
  float mean = pair_sum(s) * (1.f / 128);
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = E::val(v[c][e]) - mean;
      q = __builtin_fmaf(d, d, q);
    }
  q = pair_sum(q);
  float mp[P], qp[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    mp[i] = __shfl(mean, 2 * i, LPR);
    qp[i] = __shfl(q, 2 * i, LPR);
  }
  mean = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) mean += mp[i];
  mean /= (float)P;
  float m2 = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const float d = mp[i] - mean;
    m2 += __builtin_fmaf(128.f * d, d, qp[i]);
  }
  const float rstd = rsqrtf(m2 / (float)N + eps);
  half_t* const orow = out + row * N + 128 * g;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    h8 o;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int f = 128 * g + 16 * c + 8 * hh + 4 * lh;
      const half_t one = __builtin_bit_cast(half_t, E::kOne);
      const h4 ga = gamma ? *(const h4*)(gamma + f) : h4{one, one, one, one};
      const h4 be = beta ? *(const h4*)(beta + f) : h4{};
      f4 z;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        z[e] = __builtin_fmaf((E::val(v[c][4 * hh + e]) - mean) * rstd, E::val(ga[e]), E::val(be[e]));
      const h4 h = E::cvt4(z);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[4 * hh + e] = h[e];
    }
    const u32x4 w = trade(__builtin_bit_cast(u32x4, o));
    if (ok) *(u32x4*)(orow + 16 * c + 8 * lh) = w;
  }
}

template <class C, int ACT, bool RESID, bool BROW, typename E>
static hipError_t launch(const Args& a, hipStream_t s) {
  const int64_t tiles = ((a.M + C::BM - 1) / C::BM) * (a.N / C::BN);
  // XCD x runs tiles [x T / 8, (x + 1) T / 8): at most ceil(T / 8) of them.
  const int64_t grid = (tiles + 7) / 8 * 8;
  if (grid > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((tile_kernel<C, ACT, RESID, BROW, E>), dim3((unsigned)grid), dim3(NT), 0, s, a);
  return hipGetLastError();
}

template <class C, bool BROW, typename E>
static hipError_t dispatch(const Args& g, int act, hipStream_t s) {
  if constexpr (BROW) {
    if (g.r) return act == ACT_NONE ? launch<C, ACT_NONE, true, BROW, E>(g, s) : hipErrorInvalidValue;
  }
  if (g.r) return hipErrorInvalidValue;
  switch (act) {
    case ACT_NONE: return launch<C, ACT_NONE, false, BROW, E>(g, s);
    case ACT_RELU: return launch<C, ACT_RELU, false, BROW, E>(g, s);
    case ACT_GELU_TANH: return launch<C, ACT_GELU_TANH, false, BROW, E>(g, s);
    case ACT_SIGMOID: return launch<C, ACT_SIGMOID, false, BROW, E>(g, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename E>
static hipError_t launch_typed(const Args& g, int act, int size, bool brow, hipStream_t s) {
  if (size == 64) return brow ? dispatch<T64, true, E>(g, act, s) : dispatch<T64, false, E>(g, act, s);
  return brow ? dispatch<T128, true, E>(g, act, s) : dispatch<T128, false, E>(g, act, s);
}

template <typename E>
static hipError_t ln_typed(int64_t M, int64_t N, const half_t* x, const half_t* g, const half_t* b, float eps,
                           half_t* out, hipStream_t s) {
  const int64_t rows = 4 * kWave / (N / 64);  // rows per block
  const dim3 grid((unsigned)((M + rows - 1) / rows)), block(256);
  switch (N) {
    case 256: hipLaunchKernelGGL((ln_rows_kernel<256, E>), grid, block, 0, s, x, g, b, eps, out, M); break;
    case 512: hipLaunchKernelGGL((ln_rows_kernel<512, E>), grid, block, 0, s, x, g, b, eps, out, M); break;
    case 1024: hipLaunchKernelGGL((ln_rows_kernel<1024, E>), grid, block, 0, s, x, g, b, eps, out, M); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace tile

hipError_t tile_launch(const Args& g, int act, int size, int dtype, hipStream_t s) {
  const bool brow = g.w != nullptr;
  return dtype == GP_DTYPE_BF16 ? tile::launch_typed<BF16>(g, act, size, brow, s)
                                : tile::launch_typed<F16>(g, act, size, brow, s);
}

}  // namespace gemm

hipError_t gemm_ln_rows_launch(int64_t M, int64_t N, const void* x, const void* gamma, const void* beta, float eps,
                               void* out, int dtype, hipStream_t s) {
  using namespace gemm::tile;
  if (M <= 0) return hipSuccess;
  if ((((uintptr_t)x | (uintptr_t)out) & 15) || (((uintptr_t)gamma | (uintptr_t)beta) & 7)) return hipErrorInvalidValue;
  return dtype == GP_DTYPE_BF16
             ? ln_typed<BF16>(M, N, (const half_t*)x, (const half_t*)gamma, (const half_t*)beta, eps, (half_t*)out, s)
             : ln_typed<F16>(M, N, (const half_t*)x, (const half_t*)gamma, (const half_t*)beta, eps, (half_t*)out, s);
}

}  // namespace gp
