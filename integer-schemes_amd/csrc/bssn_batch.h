// Batched form of the fused RHS / RK stage kernels: every block of a block-structured
// hierarchy (blocks of different extents and spacings in one pool) in one launch.
//
// Replaces, on the reference side, the slot-batched step of the block-AMR solver
// (2D/src/mcs2d/amr/evolve.py:659-775): there every level is a fixed-shape slot array and the
// RHS is vmapped over all slots, inactive ones included (:710-717). Here the work is a list of
// bricks over the blocks that exist, of any extent, and each brick is evaluated by the
// same wave program as the single-grid kernel (bssn_fused.h), so a block's result is
// bit-identical to running the single-grid kernel on that block alone.
//
// Scheduling: the brick list is split into one chunk per XCD. Either one workgroup per brick
// (workgroup w -> chunk w mod 8, matching the round-robin placement of workgroups on XCDs), or
// a persistent grid whose waves pull bricks from their XCD's queue and then from the others'
// until every queue is drained; each wave takes one brick per atomic, so every wave exits once
// the counters pass the chunk ends.
#pragma once

#include <hip/hip_runtime.h>

#include <math.h>

#include "bssn_algebra.h"
#include "bssn_brick.h"
#include "bssn_group.h"
#include "bssn_hip.h"
#include "bssn_kernels.h"
#include "bssn_params.h"
#include "bssn_stage.h"

namespace bssn {


__device__ __forceinline__ const double* shifted(const double* p, long off) {
  return p ? p + off : p;
}
__device__ __forceinline__ double* shifted(double* p, long off) { return p ? p + off : p; }

// next brick of this wave: -1 when every chunk it may serve is drained
__device__ __forceinline__ int next_item(const BatchArgs& b, int* chunk, int* round) {
  if (!b.persistent) {
    if (*round) return -1;
    *round = 1;
    const int w = (int)blockIdx.x;
    const int c = w & (BATCH_CHUNKS - 1);
    const int i = b.list.cb[c] + (w >> 3);
    return i < b.list.cb[c + 1] ? i : -1;
  }
  while (*round < BATCH_CHUNKS) {
    const int c = (*chunk + *round) & (BATCH_CHUNKS - 1);
    int k = 0;
    if (threadIdx.x == 0) k = atomicAdd(&b.ctr[c], 1);
    k = __builtin_amdgcn_readfirstlane(k);
    const int i = b.list.cb[c] + k;
    if (i < b.list.cb[c + 1]) return i;
    ++*round;
  }
  return -1;
}

// A block of the batch as one launch's grid: extents, per-block scales and scalars (formed on the
// device in the host's rounding) and the stage's buffers at the block's offset. What is the same
// for the whole brick is moved to scalar registers: the block table is read by vector loads, and
// as vector values the six buffer pointers and the extents would live through the whole kernel.
template <int ORD>
struct BatchBlock {
  Dims d;
  Scales w;
  Scal sc;
  StageArgs a;
  long off;             // pool offset of the block

  __device__ __forceinline__ BatchBlock(const StageArgs& args, const BatchArgs& b,
                                        const BlockDesc& blk) {
    d.ng = uniform(blk.ng);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      d.S[a] = uniform(blk.S[a]);
      d.lo[a] = b.interior ? d.ng : 0;
      d.n[a] = b.interior ? d.S[a] - 2 * d.ng : d.S[a];
    }
    d.P = (long)d.S[0] * d.S[1] * d.S[2];
    off = uniform(blk.off);
    w = make_scales(blk.h, ORD, b.sigma);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      w.s1[a] = uniform(w.s1[a]);
      w.s2[a] = uniform(w.s2[a]);
      w.sm[a] = uniform(w.sm[a]);
      w.sko[a] = uniform(w.sko[a]);
    }
    sc = with_ssl(b.base, args.tdev, args.toff);
    sc.cahd = uniform(cahd_factor(b.cahd_c, blk.h[0], b.dt));
    a = args;
    a.Yin = shifted(args.Yin, off);
    a.U = shifted(args.U, off);
    a.Y = shifted(args.Y, off);
    a.K1 = shifted(args.K1, off);
    a.FP = shifted(args.FP, off);
    a.Uout = shifted(args.Uout, off);
  }
};

// one brick of one block, by the single-grid wave program
template <int ORD, bool KO, int MODE, int KIND>
__device__ __forceinline__ void batch_brick(double* lds, const StageArgs& args,
                                            const BatchArgs& b, int it, int lane) {
  using G = Geo<ORD, KO>;
  const BrickItem item = b.list.items[it];
  const BlockDesc blk = b.blk[item.blk];
  const BatchBlock<ORD> B(args, b, blk);
  const int org = uniform(item.org);
  const int ox = org & 1023, oy = (org >> 10) & 1023, oz = (org >> 20) & 1023;
  using Src = WaveSrc<ORD, KO, MODE, RhsOrder, fused_depth<KIND, ORD>()>;
  if constexpr (MODE == LINK) {
    Src src(lds, args.Yin, B.off, b.link + 2 * blk.moff, b.pool_n, B.w, B.d, ox, oy, oz, lane);
    StageOut<KIND> out(B.a, B.d.P, src.gp, lane_valid<G>(B.d, ox, oy, oz, lane), true);
    bssn_rhs_point<KO>(src, B.sc, out);
  } else {
    Src src(lds, B.a.Yin, B.w, B.d, ox, oy, oz, lane);
    StageOut<KIND> out(B.a, B.d.P, src.gp, lane_valid<G>(B.d, ox, oy, oz, lane), true);
    bssn_rhs_point<KO>(src, B.sc, out);
  }
}

template <int ORD, bool KO, int MODE, bool PERSIST, int KIND>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(fused_waves<KIND>(), fused_waves<KIND>())))
void k_fused_batch(StageArgs args, BatchArgs b) {
  using G = Geo<ORD, KO>;
  __shared__ double lds[G::VOL];
  const int lane = (int)threadIdx.x;
  int chunk = (int)blockIdx.x & (BATCH_CHUNKS - 1), round = 0;
  if (!PERSIST) {
    const int it = next_item(b, &chunk, &round);
    if (it >= 0) batch_brick<ORD, KO, MODE, KIND>(lds, args, b, it, lane);
    return;
  }
#pragma unroll 1
  for (int it = next_item(b, &chunk, &round); it >= 0; it = next_item(b, &chunk, &round)) {
    batch_brick<ORD, KO, MODE, KIND>(lds, args, b, it, lane);
    // the next brick restages the box: keep its writes behind this brick's reads
    __builtin_amdgcn_wave_barrier();
  }
}

// The same on bricks shared by four waves (bssn_group.h), one workgroup per brick of the list;
// equal results.
template <int ORD, bool KO, int MODE, int KIND>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2, 2)))
void k_fused_batch_group(StageArgs args, BatchArgs b) {
  using G = GroupGeo<ORD, KO>;
  static_assert(G::NT == 256, "launch bounds");
  __shared__ double mem[G::LDS_DOUBLES];
  int chunk = 0, round = 0;
  const int it = next_item(b, &chunk, &round);   // b.persistent is 0: the same for every lane
  if (it < 0) return;
  const BrickItem item = b.list.items[it];
  const BlockDesc blk = b.blk[item.blk];
  const BatchBlock<ORD> B(args, b, blk);
  const int org = uniform(item.org);
  const int ox = org & 1023, oy = (org >> 10) & 1023, oz = (org >> 20) & 1023;
  const int t = (int)threadIdx.x;
  using Src = GroupSrc<ORD, KO, MODE>;
  if constexpr (MODE == LINK) {
    Src src(mem, args.Yin, B.off, b.link + 2 * blk.moff, b.pool_n, B.w, B.d, ox, oy, oz, t);
    StageOut<KIND, true> out(B.a, B.d.P, src.gp, lane_valid<G>(B.d, ox, oy, oz, t), true);
    bssn_rhs_point<KO>(src, B.sc, out);
  } else {
    Src src(mem, B.a.Yin, B.w, B.d, ox, oy, oz, t);
    StageOut<KIND, true> out(B.a, B.d.P, src.gp, lane_valid<G>(B.d, ox, oy, oz, t), true);
    bssn_rhs_point<KO>(src, B.sc, out);
  }
}

template <int ORD, bool KO, int MODE, int KIND>
static hipError_t launch_batch_t(const StageArgs& a, const BatchArgs& b, int grid,
                                 hipStream_t st) {
  using G = Geo<ORD, KO>;
  if (b.shared)
    hipLaunchKernelGGL((k_fused_batch_group<ORD, KO, MODE, KIND>), dim3(grid), dim3(256), 0, st,
                       a, b);
  else if (b.persistent)
    hipLaunchKernelGGL((k_fused_batch<ORD, KO, MODE, true, KIND>), dim3(grid), dim3(G::NT), 0,
                       st, a, b);
  else
    hipLaunchKernelGGL((k_fused_batch<ORD, KO, MODE, false, KIND>), dim3(grid), dim3(G::NT), 0,
                       st, a, b);
  return hipGetLastError();
}

// every (KO, MODE, kind) instance of one FD order (RHS and RK4 kinds)
template <int ORD>
static hipError_t launch_batch_ord(const StageArgs& a, const BatchArgs& b, int grid, bool ko,
                                   int mode, hipStream_t st) {
  return with_kind<false>(a.kind, [&](auto k) -> hipError_t {
    constexpr int K = decltype(k)::value;
    if (ko)
      return mode == WRAP   ? launch_batch_t<ORD, true, WRAP, K>(a, b, grid, st)
             : mode == LINK ? launch_batch_t<ORD, true, LINK, K>(a, b, grid, st)
                            : launch_batch_t<ORD, true, CLAMP, K>(a, b, grid, st);
    return mode == WRAP   ? launch_batch_t<ORD, false, WRAP, K>(a, b, grid, st)
           : mode == LINK ? launch_batch_t<ORD, false, LINK, K>(a, b, grid, st)
                          : launch_batch_t<ORD, false, CLAMP, K>(a, b, grid, st);
  });
}

}  // namespace bssn
