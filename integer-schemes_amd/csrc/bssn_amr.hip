// Block hierarchy transfers: node-centred 2:1 prolongation and the refinement indicator.
//
// Prolongation (3D/src/multipatch/amr/kernels.py:53-108): the 1D refinement keeps coarse node k
// at fine index 2k and puts at 2k+1 the 6-point Lagrange midpoint
//     fine[2k+1] = sum_{j=-2..3} w_j coarse[k + j],  w = (3, -25, 150, 150, -25, 3) / 256
// (the reference forms w with its Lagrange product in float64, which gives these dyadic values
// exactly), with the coarse reads edge-clamped to the parent's padded block; 3D is the tensor
// product applied x, then y, then z. One thread evaluates one destination point for all 24
// fields directly from the parent: per field the x sums are formed first, then the y sum over
// them, then the z sum, each sum left to right from 0.0 and with contraction off -- the
// rounding of the reference's three sequential passes. Even axes are copies.
//
// Indicator (kernels.py:143-158): the largest undivided difference |u(p + e_a) - u(p)| over the
// interior plus one ring, per (block, field), NaN-propagating like a max over an array.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "bssn_entries.h"
#include "bssn_hip.h"
#include "bssn_kernels.h"

namespace bssn {

namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

struct Taps {
  int n;          // 1 (coincident node) or 6 (midpoint)
  int idx[6];     // parent node indices along the axis, clamped
};

__device__ __forceinline__ Taps taps(int fine, int S) {
  Taps t;
  const int k = fine >> 1;
  if ((fine & 1) == 0) {
    t.n = 1;
    t.idx[0] = clampi(k, 0, S - 1);
  } else {
    t.n = 6;
#pragma unroll
    for (int j = 0; j < 6; ++j) t.idx[j] = clampi(k - 2 + j, 0, S - 1);
  }
  return t;
}

__constant__ double kWMid[6] = {3.0 / 256.0, -25.0 / 256.0, 150.0 / 256.0,
                                150.0 / 256.0, -25.0 / 256.0, 3.0 / 256.0};

}  // namespace

// one field of one destination point, with the tap counts of its parity class fixed at compile
// time (OX: x fine index odd, ...)
template <bool OX, bool OY, bool OZ>
__device__ __forceinline__ void prolong_field(double* __restrict__ pool,
                                              const bssn_prolong_point& m, int f) {
#pragma clang fp contract(off)
  constexpr int NY = OY ? 6 : 1, NZ = OZ ? 6 : 1;
  const Taps tx = taps(m.fine[0], m.pS[0]);
  const Taps ty = taps(m.fine[1], m.pS[1]);
  const Taps tz = taps(m.fine[2], m.pS[2]);
  const long sy = m.pS[2], sx = (long)m.pS[1] * m.pS[2];
  const long P = sx * m.pS[0];
  const double* c = pool + m.parent + (long)f * P;
  double vz = 0.0;
#pragma unroll
  for (int kz = 0; kz < NZ; ++kz) {
    double vy = 0.0;
#pragma unroll
    for (int ky = 0; ky < NY; ++ky) {
      const double* row = c + (long)ty.idx[ky] * sy + tz.idx[kz];
      double vx;
      if constexpr (OX) {
        vx = 0.0;
#pragma unroll
        for (int kx = 0; kx < 6; ++kx) vx = vx + kWMid[kx] * row[(long)tx.idx[kx] * sx];
      } else {
        vx = row[(long)tx.idx[0] * sx];
      }
      if constexpr (OY) vy = vy + kWMid[ky] * vx; else vy = vx;
    }
    if constexpr (OZ) vz = vz + kWMid[kz] * vy; else vz = vy;
  }
  pool[m.dst + (long)f * m.dst_stride] = vz;
}

// One thread per entry and field (blockIdx.y = field): the up to 6^3 taps of a point are
// independent loads, and 24 threads per point keep many more of them in flight than one thread
// looping over the fields. Entries sorted by parity class keep a wave on one branch. An entry
// that would reach outside the pool (pool_n doubles) is skipped.
__global__ __launch_bounds__(256) void k_prolong(double* __restrict__ pool,
                                                 const bssn_prolong_point* __restrict__ pts,
                                                 long n, long long pool_n) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int f = (int)blockIdx.y;
  if (e >= n) return;
  const bssn_prolong_point m = pts[e];
  if (!prolong_entry_ok(m, pool_n)) return;
  const int cls = (m.fine[0] & 1) << 2 | (m.fine[1] & 1) << 1 | (m.fine[2] & 1);
  switch (cls) {
    case 0: prolong_field<false, false, false>(pool, m, f); break;
    case 1: prolong_field<false, false, true>(pool, m, f); break;
    case 2: prolong_field<false, true, false>(pool, m, f); break;
    case 3: prolong_field<false, true, true>(pool, m, f); break;
    case 4: prolong_field<true, false, false>(pool, m, f); break;
    case 5: prolong_field<true, false, true>(pool, m, f); break;
    case 6: prolong_field<true, true, false>(pool, m, f); break;
    default: prolong_field<true, true, true>(pool, m, f); break;
  }
}

// One 4x4x4 fine tile and PT_FIELDS consecutive fields per 64-lane workgroup (blockIdx.y =
// field group). Per field, the 7^3 coarse window of the tile (clamped into the parent, as the
// point kernel's taps) is written to LDS, then the x pass X[fx][cy][cz], the y pass
// Y[fx][fy][cz] and, at the tile's points only, the z pass -- each sum over its taps in the
// point kernel's order, so every point gets the value of its bssn_prolong_point entry bit for
// bit. The window's parent offsets and the lane's tile point are formed once per tile; the next
// field's window is loaded into registers while the current field's passes run. A tile or point
// that would reach outside the pool or the point array is skipped (the tile test is uniform
// over the group). Four fields per group: on the 640-block hierarchy's fill, 2 / 3 / 4 / 6 / 8 /
// 24 fields per group take 1.134 / 1.124 / 1.121 / 1.124 / 1.133 / 1.179 ms per fill, one field
// per group 1.352 ms.
#ifndef BSSN_PT_FIELDS
#define BSSN_PT_FIELDS 4
#endif
constexpr int PT_FIELDS = BSSN_PT_FIELDS;
static_assert(BSSN_NF % PT_FIELDS == 0, "field groups must tile the 24 fields");

__global__ __launch_bounds__(64) void k_prolong_tile(double* __restrict__ pool,
                                                     const bssn_prolong_tile* __restrict__ tiles,
                                                     long ntiles,
                                                     const bssn_prolong_tile_point* __restrict__ tp,
                                                     long long ntp, long long pool_n) {
#pragma clang fp contract(off)
  constexpr int NW = 343, NS = (NW + 63) / 64;     // window cells; per-lane slots
  __shared__ double W[NW];
  __shared__ double X[4 * 49];
  __shared__ double Y[16 * 7];
  // XCD-aware: the dispatcher deals workgroups round-robin over the 8 XCDs (gridDim.x is a
  // multiple of 8, so x % 8 picks the XCD); each XCD takes a contiguous run of tiles, whose
  // coarse windows (tiles are sorted by parent and position) share cache lines
  const long G8 = (long)gridDim.x, w = (long)blockIdx.x;
  const long ti = (w & 7) * (G8 >> 3) + (w >> 3);
  if (ti >= ntiles) return;
  const bssn_prolong_tile T = tiles[ti];
  const int lane = (int)threadIdx.x;
  if (!prolong_tile_ok(T, pool_n) || T.first + T.count > ntp) return;
  const int f0 = (int)blockIdx.y * PT_FIELDS;
  const long sy = T.pS[2], sx = (long)T.pS[1] * T.pS[2];
  const long P = sx * T.pS[0];
  const int c0[3] = {(T.origin[0] >> 1) - 2, (T.origin[1] >> 1) - 2, (T.origin[2] >> 1) - 2};
  long woff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int i = lane + 64 * s;
    const int x = clampi(c0[0] + i / 49, 0, T.pS[0] - 1);
    const int y = clampi(c0[1] + (i / 7) % 7, 0, T.pS[1] - 1);
    const int z = clampi(c0[2] + i % 7, 0, T.pS[2] - 1);
    woff[s] = x * sx + y * sy + z;
  }
  // the lane's point of the tile's first 64 (a tile holds each of its 64 fine points once)
  bssn_prolong_tile_point q0{};
  bool ok0 = false;
  if (lane < T.count) {
    q0 = tp[T.first + lane];
    ok0 = prolong_tile_point_ok(q0, pool_n);
  }
  double wv[NS];
  {
    const double* c = pool + T.parent + (long)f0 * P;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (lane + 64 * s < NW) wv[s] = c[woff[s]];
  }
#pragma unroll 1
  for (int f = f0; f < f0 + PT_FIELDS; ++f) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (lane + 64 * s < NW) W[lane + 64 * s] = wv[s];
    __syncthreads();
    if (f + 1 < f0 + PT_FIELDS) {                     // next field's window, in flight
      const double* c = pool + T.parent + (long)(f + 1) * P;
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (lane + 64 * s < NW) wv[s] = c[woff[s]];
    }
    for (int i = lane; i < 4 * 49; i += 64) {        // x pass
      const int fx = i / 49, jk = i % 49;
      const int fine = T.origin[0] + fx, kx = (fine >> 1) - c0[0];
      double v;
      if (fine & 1) {
        v = 0.0;
#pragma unroll
        for (int t = 0; t < 6; ++t) v = v + kWMid[t] * W[(kx - 2 + t) * 49 + jk];
      } else {
        v = W[kx * 49 + jk];
      }
      X[i] = v;
    }
    __syncthreads();
    for (int i = lane; i < 16 * 7; i += 64) {        // y pass
      const int fx = i / 28, fy = (i / 7) % 4, k = i % 7;
      const int fine = T.origin[1] + fy, ky = (fine >> 1) - c0[1];
      double v;
      if (fine & 1) {
        v = 0.0;
#pragma unroll
        for (int t = 0; t < 6; ++t) v = v + kWMid[t] * X[fx * 49 + (ky - 2 + t) * 7 + k];
      } else {
        v = X[fx * 49 + ky * 7 + k];
      }
      Y[i] = v;
    }
    __syncthreads();
    auto zpass = [&](const bssn_prolong_tile_point& q) {
      const int fz = q.local & 3;
      const double* yr = Y + (q.local >> 2) * 7;
      const int fine = T.origin[2] + fz, kz = (fine >> 1) - c0[2];
      double v;
      if (fine & 1) {
        v = 0.0;
#pragma unroll
        for (int t = 0; t < 6; ++t) v = v + kWMid[t] * yr[kz - 2 + t];
      } else {
        v = yr[kz];
      }
      pool[q.dst + (long)f * q.dst_stride] = v;
    };
    if (ok0) zpass(q0);
    for (long long e = T.first + 64 + lane; e < T.first + T.count; e += 64) {
      const bssn_prolong_tile_point q = tp[e];
      if (prolong_tile_point_ok(q, pool_n)) zpass(q);
    }
  }
}

hipError_t launch_prolong_tiles(double* pool, long long pool_n, const void* tiles, long n,
                                const void* tp, long long ntp, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const long g = (n + 7) & ~7L;
  if (g > 0x7fffffffL) return hipErrorInvalidValue;       // beyond one grid dimension
  hipLaunchKernelGGL(k_prolong_tile, dim3((unsigned)g, BSSN_NF / PT_FIELDS), dim3(64), 0, st,
                     pool, (const bssn_prolong_tile*)tiles, n, (const bssn_prolong_tile_point*)tp,
                     ntp, pool_n);
  return hipGetLastError();
}

hipError_t launch_prolong(double* pool, long long pool_n, const void* pts, long n,
                          hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const long blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_prolong, dim3((unsigned)blocks, BSSN_NF), dim3(256), 0, st, pool,
                     (const bssn_prolong_point*)pts, n, pool_n);
  return hipGetLastError();
}

// Separable whole-block prolongation: one workgroup per (job, field group, x slab), a slab being
// PB_SLABS-th of the padded block's fine x planes. The x pass fills X[rx][ky][kz] (the slab's
// fine x planes, coarse y and z window) from the parent, the y pass Y[rx][ry][kz] from X, and
// the z sums are formed only at the points the job writes. Every fine x plane depends only on
// its own coarse taps, so slabs share no work. Window index k stands for parent node kmin + k,
// read clamped, so the taps of every sum are the clamped nodes of the per-point kernel, summed
// in the same order. A job that is not a valid block of at most PB_WMAX padded nodes per axis
// inside the pool (pool_n doubles) is skipped (the test is uniform across the workgroup, so no
// thread reaches a barrier alone). What bounds it is instruction issue, not its bytes: most of
// it was turning indices into coordinates by integer division, for every field anew. A workgroup
// now takes PB_FIELDS fields of a slab, a thread forms its columns, rows and points once, the next
// field's coarse nodes are loaded while the current one's passes run, and a plane whose points
// are all supplied but its ghost rows forms only those. 384-block hierarchy (16^3 blocks), the two
// launches of a fill: 0.310 + 0.210 -> 0.144 + 0.102 ms (2 / 4 / 24 fields 0.189 + 0.129 / 0.153
// + 0.106 / 0.167 + 0.097; 8 or 5 slabs 0.178 / 0.186 for the larger one at 4 fields; 384 / 512
// threads 0.155 / 0.152).
constexpr int PB_SLABS = 6;
constexpr int PB_THREADS = 256;
constexpr int PB_FIELDS = 8;
static_assert(BSSN_NF % PB_FIELDS == 0, "field groups must tile the 24 fields");
constexpr int PB_SW = (PB_WMAX + PB_SLABS - 1) / PB_SLABS;   // fine x planes per slab, at most

// Quotient of 0 <= i < 2^20 / PB_WMAX by a divisor known only at run time, 1 <= d <= PB_WMAX,
// with a quotient below 2^11: m = 2^20 / d rounded up exceeds it by less than 1, so i m 2^-20
// exceeds i / d by less than i 2^-20 < 1 / PB_WMAX and rounds down to the quotient. Two
// instructions instead of about 40.
struct SmallDiv {
  unsigned m;
  __device__ __forceinline__ explicit SmallDiv(int d) : m(((1u << 20) + d - 1) / d) {}
  __device__ __forceinline__ int quot(int i) const { return (int)(((unsigned)i * m) >> 20); }
};
static_assert(PB_SW * PB_WMAX * PB_WMAX < (1 << 20) / PB_WMAX && PB_SW * PB_WMAX < (1 << 11),
              "SmallDiv's range");

// sum of the six taps at u[0], u[stride], ..., left to right from 0.0 (odd fine index), or the
// coarse node itself (even)
__device__ __forceinline__ double refine_1d(const double* u, int stride, bool odd) {
#pragma clang fp contract(off)
  double v = 0.0;
#pragma unroll
  for (int j = 0; j < 6; ++j) v = v + kWMid[j] * u[j * stride];
  return odd ? v : u[2 * stride];
}

__global__ __launch_bounds__(PB_THREADS) void k_prolong_block(
    double* __restrict__ pool, const bssn_prolong_block* __restrict__ jobs, long long pool_n) {
#pragma clang fp contract(off)
  constexpr int NX = (PB_KMAX * PB_KMAX + PB_THREADS - 1) / PB_THREADS;
  constexpr int NY = (PB_SW * PB_WMAX * PB_KMAX + PB_THREADS - 1) / PB_THREADS;
  constexpr int NZ = (PB_SW * PB_WMAX * PB_WMAX + PB_THREADS - 1) / PB_THREADS;
  constexpr int NV = 6 + (PB_SW + 1) / 2;         // coarse nodes under a slab's planes, at most
  __shared__ double X[PB_SW * PB_KMAX * PB_KMAX];
  __shared__ double Y[PB_SW * PB_WMAX * PB_KMAX];
  const int slab = (int)(blockIdx.x % PB_SLABS);
  const long jf = blockIdx.x / PB_SLABS;
  constexpr int NG = BSSN_NF / PB_FIELDS;
  const bssn_prolong_block jb = jobs[jf / NG];
  if (!block_job_ok(jb, pool_n)) return;
  const int f0 = (int)(jf % NG) * PB_FIELDS;
  const int W = jb.BS + 2 * jb.ng;
  const int sw = (W + PB_SLABS - 1) / PB_SLABS;
  const int x0 = slab * sw, nx = min(W, x0 + sw) - x0;
  if (nx <= 0) return;
  const int sy = W, sx = W * W;
  const long P = (long)sx * W;
  int r0[3], kmin[3], K[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    r0[a] = jb.ng + jb.corner[a] * jb.BS;
    kmin[a] = (r0[a] >> 1) - 2;
    K[a] = ((r0[a] + W - 1) >> 1) + 3 - kmin[a] + 1;
  }
  const int lo = jb.ng, hi = jb.ng + jb.BS, t = (int)threadIdx.x;
  const SmallDiv dK2(K[2]), dW(W), dG(max(1, 2 * lo));

  // What a thread does in the three passes is the same for every field: formed once.
  // x pass: window columns (ky, kz), their offset in a parent plane and their place in X
  int xsrc[NX], xdst[NX];
#pragma unroll
  for (int k = 0; k < NX; ++k) {
    const int i = min(t + k * PB_THREADS, K[1] * K[2] - 1);
    const int ky = dK2.quot(i), kz = i - ky * K[2];
    xsrc[k] = clampi(kmin[1] + ky, 0, W - 1) * sy + clampi(kmin[2] + kz, 0, W - 1);
    xdst[k] = ky * PB_KMAX + kz;
  }
  // The y rows a plane needs: all of them, or, for a plane inside the block whose z face slabs
  // come from neighbours, its 2 ng ghost rows only. Planes [0, a) and [a + ns, nx) of the slab are
  // of the first kind, [a, a + ns) of the second.
  const bool thin = lo > 0 && (jb.skip & (48 | 64)) == 48;
  const int a = thin ? min(nx, max(0, lo - x0)) : nx;
  const int ns = thin ? max(0, min(nx, hi - x0) - a) : 0;
  const int full_rows = (nx - ns) * W, rows = full_rows + ns * 2 * lo;
  auto row_at = [&](int r, int* xl, int* y) {
    if (r < full_rows) {
      const int p = dW.quot(r);
      *y = r - p * W;
      *xl = p < a ? p : p + ns;
    } else {
      const int p = dG.quot(r - full_rows), q = r - full_rows - p * 2 * lo;
      *y = q < lo ? q : q + jb.BS;
      *xl = a + p;
    }
  };
  // y pass: first tap in X | place in Y << 12 | odd << 24; -1: none
  int yitem[NY];
#pragma unroll
  for (int k = 0; k < NY; ++k) {
    const int i = t + k * PB_THREADS, r = dK2.quot(i), kz = i - r * K[2];
    yitem[k] = -1;
    if (i < rows * K[2]) {
      int xl, y;
      row_at(r, &xl, &y);
      const int ry = r0[1] + y;
      yitem[k] = ((xl * PB_KMAX + (ry >> 1) - 2 - kmin[1]) * PB_KMAX + kz) |
                 ((xl * PB_WMAX + y) * PB_KMAX + kz) << 12 | (ry & 1) << 24;
    }
  }
  // z pass: first tap in Y | point of the block << 12 | odd << 26; -1: not written
  int zitem[NZ];
#pragma unroll
  for (int k = 0; k < NZ; ++k) {
    const int i = t + k * PB_THREADS, r = dW.quot(i), z = i - r * W;
    zitem[k] = -1;
    if (i < rows * W) {
      int xl, y;
      row_at(r, &xl, &y);
      const int x = x0 + xl, rz = r0[2] + z;
      const bool ix = x >= lo && x < hi, iy = y >= lo && y < hi, iz = z >= lo && z < hi;
      // the interior only if asked for; a face slab (ghost along exactly one axis, interior along
      // the other two) unless a neighbour supplies it
      const bool skip = (ix && iy && iz) ? !(jb.skip & 64)
                        : (iy && iz)     ? (jb.skip & (x < lo ? 1 : 2)) != 0
                        : (ix && iz)     ? (jb.skip & (y < lo ? 4 : 8)) != 0
                        : (ix && iy)     ? (jb.skip & (z < lo ? 16 : 32)) != 0
                                         : false;
      if (!skip)
        zitem[k] = ((xl * PB_WMAX + y) * PB_KMAX + (rz >> 1) - 2 - kmin[2]) |
                   ((x * W + y) * W + z) << 12 | (rz & 1) << 26;
    }
  }
  const int k0 = ((r0[0] + x0) >> 1) - 2;
  int plane[NV];                                   // offsets of the coarse planes
#pragma unroll
  for (int j = 0; j < NV; ++j) plane[j] = clampi(k0 + j, 0, W - 1) * sx;

  auto run = [&](auto odd) {
    constexpr int ODD = decltype(odd)::value;      // parity of the slab's first plane
    double u[NX][NV];
    auto load = [&](int f) {
      const double* c = pool + jb.parent + (long)f * P;
#pragma unroll
      for (int k = 0; k < NX; ++k)
#pragma unroll
        for (int j = 0; j < NV; ++j)
          if (k == 0 || t + k * PB_THREADS < K[1] * K[2]) u[k][j] = c[xsrc[k] + plane[j]];
    };
    load(f0);
#pragma unroll 1
    for (int f = f0; f < f0 + PB_FIELDS; ++f) {
#pragma unroll
      for (int k = 0; k < NX; ++k)
        if (t + k * PB_THREADS < K[1] * K[2]) {
#pragma unroll
          for (int xl = 0; xl < PB_SW; ++xl)
            if (xl < nx)
              X[xl * PB_KMAX * PB_KMAX + xdst[k]] =
                  refine_1d(u[k] + ((ODD + xl) >> 1), 1, (ODD + xl) & 1);
        }
      __syncthreads();
      if (f + 1 < f0 + PB_FIELDS) load(f + 1);     // in flight during the y and z passes
#pragma unroll
      for (int k = 0; k < NY; ++k)
        if (yitem[k] >= 0)
          Y[(yitem[k] >> 12) & 4095] = refine_1d(X + (yitem[k] & 4095), PB_KMAX, yitem[k] >> 24);
      __syncthreads();
      double* out = pool + jb.dst + (long)f * P;
#pragma unroll
      for (int k = 0; k < NZ; ++k)
        if (zitem[k] >= 0)
          out[(zitem[k] >> 12) & 16383] = refine_1d(Y + (zitem[k] & 4095), 1, zitem[k] >> 26);
    }
  };
  if ((r0[0] + x0) & 1)
    run(std::integral_constant<int, 1>());
  else
    run(std::integral_constant<int, 0>());
}
static_assert(PB_SW * PB_KMAX * PB_KMAX <= 4096 && PB_SW * PB_WMAX * PB_KMAX <= 4096 &&
                  PB_WMAX * PB_WMAX * PB_WMAX <= 16384,
              "packed items");

hipError_t launch_prolong_blocks(double* pool, long long pool_n, const void* jobs, long n,
                                 hipStream_t st) {
  constexpr long per_job = (BSSN_NF / PB_FIELDS) * PB_SLABS;
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffffL / per_job) return hipErrorInvalidValue;   // grid too large
  hipLaunchKernelGGL(k_prolong_block, dim3((unsigned)(n * per_job)), dim3(PB_THREADS), 0, st,
                     pool, (const bssn_prolong_block*)jobs, pool_n);
  return hipGetLastError();
}

namespace {

__device__ __forceinline__ double nanmax(double m, double v) {
  return (v > m || v != v) ? v : m;     // a NaN, once in, stays
}

}  // namespace

// one workgroup of 256 per (block, field): blockIdx.x = 24 b + f
__global__ __launch_bounds__(256) void k_indicator(const double* __restrict__ pool,
                                                   const BlockDesc* __restrict__ blks,
                                                   double* __restrict__ out) {
  const int b = (int)blockIdx.x / BSSN_NF, f = (int)blockIdx.x % BSSN_NF;
  const BlockDesc blk = blks[b];
  const int lo = blk.ng - 1;
  const int C[3] = {blk.S[0] - 2 * blk.ng + 2, blk.S[1] - 2 * blk.ng + 2,
                    blk.S[2] - 2 * blk.ng + 2};
  const long sy = blk.S[2], sx = (long)blk.S[1] * blk.S[2];
  const double* u = pool + blk.off + (long)f * sx * blk.S[0];
  const long total = (long)C[0] * C[1] * C[2];
  double m = 0.0;
  for (long i = threadIdx.x; i < total; i += blockDim.x) {
    const int z = (int)(i % C[2]);
    const int y = (int)((i / C[2]) % C[1]);
    const int x = (int)(i / ((long)C[2] * C[1]));
    const long p = (long)(lo + x) * sx + (long)(lo + y) * sy + (lo + z);
    const double v = u[p];
    if (x + 1 < C[0]) m = nanmax(m, fabs(u[p + sx] - v));
    if (y + 1 < C[1]) m = nanmax(m, fabs(u[p + sy] - v));
    if (z + 1 < C[2]) m = nanmax(m, fabs(u[p + 1] - v));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = nanmax(m, __shfl_xor(m, o, 64));
  __shared__ double red[4];
  const int wave = (int)threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) red[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int w = 1; w < (int)blockDim.x / 64; ++w) r = nanmax(r, red[w]);
    out[blockIdx.x] = r;
  }
}

hipError_t launch_indicator(const double* pool, const BlockDesc* blk, int nblk, double* out,
                            hipStream_t st) {
  if (nblk <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_indicator, dim3((unsigned)(nblk * BSSN_NF)), dim3(256), 0, st, pool, blk,
                     out);
  return hipGetLastError();
}

}  // namespace bssn
