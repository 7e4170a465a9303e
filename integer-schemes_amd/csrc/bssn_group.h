// Bricks shared by the waves of a workgroup, for the fused kernels.
//
// One workgroup is four waves owning a 4 x 4 x 16 brick of output points (one point per lane, z
// fastest). The four waves stage one field at a time into a common LDS box (the brick plus H on
// every side), so a point costs about half the staged cells of a wave-private 4 x 4 x 4 brick
// (FD order 4 with KO: 5.9 instead of 8.5 loads per point for the fields with mixed derivatives,
// 4.4 instead of 5.5 for the others), and its rows are runs of 16 to 22 doubles instead of 4 to
// 10, both in the loads and in the stores.
//
// What bounds the fused stage kernels is unhidden latency: at one wave per SIMD (the
// wave-private form needs 374-438 registers) the 256^3 FD4 RK4 step takes 37.4 ms, of which 21.4
// ms remain with every staging load, write-back operand and store left out. Two waves per SIMD
// cover each other, but must fit 256 registers:
//   * fewer staged cells per lane (6 instead of 9) and one in-flight set of them;
//   * the write-back operands of a field are loaded shortly before its put (StageOut NEAR);
//   * 18 long-lived values per point are parked in LDS (bssn_rhs_point's keep/kept), which the
//     shared box leaves room for: 2 boxes of 17.2 KB and 36 KB of slots, two workgroups per CU.
//   * fields are addressed by 32-bit byte offsets from their uniform base (fields below 4 GiB):
//     with 64-bit indices the address pairs of 9 fields lived, spilled, from the first loads to
//     the last stores, 1.1 GB of scratch written per stage (step 26.0, bare RHS 4.81 ms).
// Measured at 256^3, FD4 with KO 6, RK4 step / bare RHS: wave-private 37.37 / 5.96, shared 24.1 /
// 4.52 ms (FD order 4 does not spill). Other shapes, with 64-bit indices: 4x4x16 26.0 / 4.64,
// 4x8x8 27.8 / 4.65, 2x8x16 27.0 / 4.86, 8x8x8 29.0 / 5.06, 4x8x16 27.1 / 5.00, 8x4x16 27.3 /
// 5.12, 8x2x16 28.3 / 4.90, 4x4x8 (two waves) 31.5 / 4.84 ms.
//
// The boxes alternate, so one barrier per field is enough: the box written for field i was last
// read for field i - 2, and a wave passes the barrier of field i - 1 only after those reads.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bssn_brick.h"

namespace bssn {

template <int ORD, bool KO>
struct GroupGeo {
  static constexpr int R = Coef<ORD>::R;                  // FD reach
  static constexpr int RK = KO ? Coef<ORD>::RK : 0;       // KO reach
  static constexpr int H = R > RK ? R : RK;               // box halo
  static constexpr int BX = BSSN_GROUP_X, BY = BSSN_GROUP_Y, BZ = BSSN_GROUP_Z;  // brick
  static constexpr int NT = BX * BY * BZ;                 // lanes (four waves)
  static constexpr int NX = BX + 2 * H, NY = BY + 2 * H, NZ = BZ + 2 * H;   // box extents
  // dense rows and planes: the 16 lanes of one LDS access phase read one z row of the brick, 16
  // distinct bank pairs whatever the pitch
  static constexpr int SY = NZ, SX = NY * NZ, VOL = NX * SX;
  static_assert(NX < 32 && NY < 32 && NZ < 32, "box coordinates are packed in 5 bits");
  static constexpr int NCORE = BX * BY * BZ;
  static constexpr int NFACE = 2 * H * (BY * BZ + BX * BZ + BX * BY);
  static constexpr int NEDGE = 4 * R * R * (BX + BY + BZ);
  __host__ __device__ static constexpr int lx(int t) { return t / (BY * BZ); }
  __host__ __device__ static constexpr int ly(int t) { return (t / BZ) % BY; }
  __host__ __device__ static constexpr int lz(int t) { return t % BZ; }
  static constexpr int NCELL = NCORE + NFACE + NEDGE;
  static constexpr int PER = (NCELL + NT - 1) / NT;       // staged cells per lane
  static constexpr int PER_FACES = (NCORE + NFACE + NT - 1) / NT;
  // parked values per point: all 18, or as many as let two workgroups share a CU's 160 KB of LDS
  // (13 with the wider boxes of FD orders 6 and 8)
  static constexpr int ROOM = (80 * 1024 / 8 - 2 * VOL) / NT;
  static constexpr int SLOTS = ROOM < 18 ? ROOM : 18;
  static_assert(SLOTS >= 12, "the gt and At rates must fit");
  static constexpr int LDS_DOUBLES = 2 * VOL + SLOTS * NT;
};

// Points of a field from which its bytes no longer fit 32-bit offsets (4 GiB).
constexpr long kGroupPoints = 1L << 29;

// Barrier of the workgroup that orders its LDS accesses (global loads and stores stay in
// flight across it).
__device__ __forceinline__ void group_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Source of fields and derivatives for bssn_rhs_point over shared boxes: as WaveSrc with one
// field in flight, with a workgroup barrier where WaveSrc relies on a wave's LDS order. Every
// lane of the workgroup must run the whole stage sequence (lanes without a point of their own
// stage cells for the others). WIDE: 64-bit addresses, for fields of 4 GiB and more.
template <int ORD, bool KO, int MODE, class ORDER = RhsOrder, bool WIDE = false>
struct GroupSrc : BoxStencil<GroupGeo<ORD, KO>, Coef<ORD>> {
  using G = GroupGeo<ORD, KO>;
  using Box = BoxStencil<G, Coef<ORD>>;
  using Box::c;
  using Box::lds;
  double* boxes;        // two boxes
  double* slots;        // this lane's parked values, NT apart
  const double* F;      // stencil source state (LINK: the pool)
  const double* Fc;     // the block's state (centre values)
  long P;
  unsigned off[G::PER]; // byte offsets of this lane's staged cells in a field (LINK: pool
                        // offsets in doubles, WIDE: offsets in doubles)
  int psrc[MODE == LINK ? G::PER : 1];   // LINK: field stride of each staged cell's block
  int cel[G::PER];      // box indices of this lane's staged cells
  double pf[G::PER];    // the next field's cells, in flight
  // the lane's point, clamped into the grid, and the place of its centre value (the point, or its
  // periodic image): byte offsets in a field (WIDE: indices)
  std::conditional_t<WIDE, long, unsigned> gp, gc;
  static constexpr int kParkSlots = G::SLOTS;

  __device__ __forceinline__ GroupSrc(double* mem, const double* F_, const Scales& sc_,
                                      const Dims& d, int ox, int oy, int oz, int t,
                                      int first = ORDER::at(0))
      : Box(mem, sc_), boxes(mem), slots(mem + 2 * G::VOL + t), F(F_), Fc(F_), P(d.P) {
    static_assert(MODE != LINK, "LINK sources take the pool and the link map");
    place(d, ox, oy, oz, t);
    const int o[3] = {ox, oy, oz};
#pragma unroll
    for (int k = 0; k < G::PER; ++k) {
      const int e = kCells<G>.c[t + k * G::NT];
      const int cc[3] = {e & 31, (e >> 5) & 31, (e >> 10) & 31};
      cel[k] = cc[0] * G::SX + cc[1] * G::SY + cc[2];
      int g[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) g[a] = map_axis<MODE>(o[a] + cc[a] - G::H, d.S[a], d.ng);
      off[k] = (unsigned)((g[0] * d.S[1] + g[1]) * d.S[2] + g[2]);
      if constexpr (!WIDE) off[k] <<= 3;
    }
    fetch(first);
  }

  // LINK: a block of a batch, as WaveSrc's (ng >= H; pool below 2^29 doubles).
  __device__ __forceinline__ GroupSrc(double* mem, const double* pool, long boff,
                                      const int* lmap, long long pool_n, const Scales& sc_,
                                      const Dims& d, int ox, int oy, int oz, int t)
      : Box(mem, sc_), boxes(mem), slots(mem + 2 * G::VOL + t), F(pool), Fc(pool + boff),
        P(d.P) {
    static_assert(MODE == LINK, "the link constructor is for LINK sources");
    place(d, ox, oy, oz, t);
    const int o[3] = {ox, oy, oz};
#pragma unroll
    for (int k = 0; k < G::PER; ++k) {
      const int e = kCells<G>.c[t + k * G::NT];
      const int cc[3] = {e & 31, (e >> 5) & 31, (e >> 10) & 31};
      cel[k] = cc[0] * G::SX + cc[1] * G::SY + cc[2];
      int g[3];
      bool inner = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        g[a] = map_axis<CLAMP>(o[a] + cc[a] - G::H, d.S[a], d.ng);
        inner = inner && g[a] >= d.ng && g[a] < d.S[a] - d.ng;
      }
      const int q = (g[0] * d.S[1] + g[1]) * d.S[2] + g[2];
      off[k] = (unsigned)((int)boff + q);
      psrc[k] = (int)d.P;
      if (!inner) {
        const int2 m = reinterpret_cast<const int2*>(lmap)[q];
        if (link_entry_ok(m.x, m.y, pool_n)) {
          off[k] = (unsigned)m.x;
          psrc[k] = m.y;
        }
      }
    }
    fetch(ORDER::at(0));
  }

  __device__ __forceinline__ void place(const Dims& d, int ox, int oy, int oz, int t) {
    c = (G::lx(t) + G::H) * G::SX + (G::ly(t) + G::H) * G::SY + (G::lz(t) + G::H);
    gp = lane_point<G>(d, ox, oy, oz, t);
    gc = lane_centre<G, MODE>(d, ox, oy, oz, t);
    if constexpr (!WIDE) {
      gp <<= 3;
      gc <<= 3;
    }
  }

  __device__ __forceinline__ static int cells(int f) {
    return ORDER::edges(f) ? G::PER : G::PER_FACES;
  }

  __device__ __forceinline__ void fetch(int f) {
    const double* u = F + (long)f * P;
    const int n = cells(f);
#pragma unroll
    for (int k = 0; k < G::PER; ++k)
      if (k < n) {
        if constexpr (MODE == LINK)
          pf[k] = *at_byte(F, (off[k] + (unsigned)(f * psrc[k])) << 3);
        else if constexpr (WIDE)
          pf[k] = u[off[k]];
        else
          pf[k] = *at_byte(u, off[k]);
      }
    __builtin_amdgcn_sched_barrier(0);   // keep the loads here, ahead of the work they overlap
  }

  // field f, loaded before, into a box; next: the field to load while f is used (-1: none)
  __device__ __forceinline__ void stage_in(int f, int box, int next) {
    const int n = cells(f);
    lds = boxes + box * G::VOL;
#pragma unroll
    for (int k = 0; k < G::PER; ++k)
      if (k < n) lds[cel[k]] = pf[k];
    group_barrier();
    if (next >= 0) fetch(next);
  }
  __device__ __forceinline__ void stage(int f) {
    const int at = ORDER::pos(f);
    stage_in(f, at & 1, at + 1 < ORDER::N ? ORDER::at(at + 1) : -1);
  }

  __device__ __forceinline__ double center(int f) const {
    if constexpr (WIDE)
      return Fc[(long)f * P + gc];
    else
      return *at_byte(Fc + (long)f * P, gc);
  }
  __device__ __forceinline__ void park(int i, double x) { slots[i * G::NT] = x; }
  __device__ __forceinline__ double parked(int i) const { return slots[i * G::NT]; }
};

}  // namespace bssn
