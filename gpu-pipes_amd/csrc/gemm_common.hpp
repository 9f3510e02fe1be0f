// What the wide GEMM kernels share (gemm.hip: persistent 256-row tiles;
// gemm_tile.hip: one small tile per workgroup): the launch arguments and the
// 128-byte-row LDS layout of an operand slab.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/gpipes.h"
#include "gp_device.hpp"
#include "gp_kernels.hpp"
#include "stages.hpp"

namespace gp {
namespace gemm {

constexpr int BK = 64;              // k per slab
constexpr int ROWB = BK * 2;        // bytes per unit row (one 128-byte L2 line)
constexpr int CPR = ROWB / 16;      // 16-byte chunks per row
constexpr int RPC = 1024 / ROWB;    // rows per 1 KiB copy instruction
constexpr int KS = BK / 16;         // MFMA k-steps per slab

struct Args {
  const half_t* a;     // [M][lda], the first K columns used
  const half_t* bt;    // [N][K] (transposed weights), or
  const half_t* w;     // [kw][ldw] (the weights in their own layout, BROW kernels)
  int ldw, kw;         // row stride and rows of w; rows [kw, K) read as zero
  const half_t* bias;  // [N] or null
  const half_t* r;     // [M][ldr] residual or null
  half_t* c;           // [M][ldc], the first N columns written
  int64_t M;
  int N;
  int K;
  int ka;              // columns of A read (a multiple of 8, <= K); columns [ka, K) read as zero
  int lda, ldc, ldr;   // row strides in elements
  // LayerNorm epilogue (LNM kernels): gamma / beta [N] or null (1 / 0), eps.
  const half_t* gamma;
  const half_t* beta;
  float eps;
  // LNM 2: per-row partial statistics [M][N / 128] ((mean, M2) of one wave's
  // 128 features, as 64-bit words), per-row-block commit counters, and the
  // launch context (epoch, status word, poll bound).
  unsigned long long* stats;
  QCounter* cnt;
  QueueCtx ctx;
  uint32_t ln_target;  // count of a row block's counter once this launch's waves have all committed
  int fresh_out;       // LNM 2: zeros for the rows of a failed wait
};

// Small-tile kernels (gemm_tile.hip): one `size` x `size` output tile per
// workgroup (64 or 128); p.bt or p.w as in gemm_launch (a residual with p.w
// only), no LayerNorm epilogue.
hipError_t tile_launch(const Args& p, int act, int size, int dtype, hipStream_t s);

// Byte offset of logical 16-byte chunk c of unit row r: the chunk position is
// XOR-swizzled with (r / 2) so 16 consecutive rows (two per 256-byte bank
// window) read at one logical chunk cover 16 distinct 16-byte bank groups.
__device__ __forceinline__ int unit_off(int r, int c) { return r * ROWB + ((c ^ ((r >> 1) & 7)) << 4); }

}  // namespace gemm
}  // namespace gp
