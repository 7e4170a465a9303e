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
//   * 16 or 18 long-lived values per point are parked in LDS (bssn_rhs_point's keep/kept), which
//     the shared boxes leave room for (32 to 36 KB of slots, two workgroups per CU);
//   * fields are addressed by 32-bit byte offsets from their uniform base (fields below 4 GiB):
//     with 64-bit indices the address pairs of 9 fields lived, spilled, from the first loads to
//     the last stores, 1.1 GB of scratch written per stage (step 26.0, bare RHS 4.81 ms).
// Measured at 256^3, FD4 with KO 6, RK4 step / bare RHS: wave-private 37.37 / 5.96, shared 24.1 /
// 4.52 ms (FD order 4 does not spill). Other shapes, with 64-bit indices: 4x4x16 26.0 / 4.64,
// 4x8x8 27.8 / 4.65, 2x8x16 27.0 / 4.86, 8x8x8 29.0 / 5.06, 4x8x16 27.1 / 5.00, 8x4x16 27.3 /
// 5.12, 8x2x16 28.3 / 4.90, 4x4x8 (two waves) 31.5 / 4.84 ms.
//
// Order 4 stages fields into two boxes in turn, a barrier per field: the box written for field i
// was last read for field i - 2, which every wave has left.
//
// With the waits covered, LDS reads are the next bound. A mixed derivative d1_j(d1_i u) needs the
// first-derivative numerators of u along i at 2R points along j, each of 2R taps: formed per point
// that is 16 / 36 / 64 reads (orders 4 / 6 / 8) for each of three. Above order 4 the numerators are
// formed once per brick, along x on the brick extended by R in y and in z and along y on the brick
// extended by R in z (3.5 to 5 per lane, two of them the lane's own first derivatives), kept in LDS
// and read 2R at a time: 61 instead of 133 LDS accesses per point and field at order 6. They take
// the room of the second box and of some registers, so the box places of the staged cells are kept
// in LDS and the loads of the field after the metric wait for the end of the Ricci tensor (with
// those in registers 47 to 63 were spilled, and the step got slower, not faster).
// RK4 step / bare RHS, before and after: 128^3 FD6 3.93 / 0.848 -> 3.59 / 0.757 ms, 128^3 FD8 5.43 /
// 1.33 -> 4.01 / 0.906 ms. At order 4 (41 instead of 67 accesses) the whole equations lose: 256^3
// 24.5 / 4.53 -> 24.9 / 4.69 ms, the waits at the second barrier cost more than the reads; passes
// over single fields (one box) win at every order.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bssn_brick.h"
#include "bssn_dispatch.h"

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
  // first-derivative numerators for the mixed derivatives: along x on BX x (BY + 2R) x (BZ + 2R)
  // (both extensions at once are not used), along y on BX x BY x (BZ + 2R), z contiguous
  static constexpr int NZE = BZ + 2 * R, NYE = BY + 2 * R;
  static constexpr int PX = BX * NYE * NZE, PY = BX * BY * NZE;
  static constexpr int EXTRA = BX * 2 * R * BZ + 2 * (BX * BY * 2 * R);   // beside the lanes' own
  static constexpr int TASKS = (EXTRA + NT - 1) / NT;
  static constexpr int BOX_DOUBLES = VOL + PX + PY;       // one box and the numerators
  // The whole equations: two workgroups share a CU's 160 KB. At order 4 two boxes (one barrier per
  // field), no numerators and 18 parked values per point; above it the numerators, two boxes where
  // 16 parked values fit beside them, else one box and 18, and then the box places of the lanes'
  // cells, two in a word, as far as the LDS goes.
  static constexpr bool NUM = ORD > 4;
  static constexpr int HALF_CU = 80 * 1024 / 8;
  static constexpr int WHOLE_BOX = VOL + (NUM ? PX + PY : 0);
  static constexpr int BOXES = !NUM || VOL + WHOLE_BOX + 16 * NT <= HALF_CU ? 2 : 1;
  static constexpr int SLOTS = NUM && BOXES == 2 ? 16 : 18;
  static constexpr int SLOT0 = (BOXES - 1) * VOL + WHOLE_BOX, TABLE0 = SLOT0 + SLOTS * NT;
  static constexpr int PAIRS = (PER + 1) / 2;
  static constexpr int ROOM = (HALF_CU - TABLE0) * 2 / NT;
  static constexpr int TABLE = !NUM && KO ? 0 : (PAIRS < ROOM ? PAIRS : ROOM);
  static constexpr int LDS_DOUBLES = TABLE0 + (TABLE * NT + 1) / 2;
  static_assert(ROOM >= 0, "two workgroups share a CU's 160 KB of LDS");
};

// The numerators of a brick's extension, one task each: packed box index | place << 12 | axis << 24
// (axis 0: along x, places in the x array; 1: along y, places after it). Tasks past the last
// repeat the first one (the same value to the same place).
template <class G>
struct NumeratorTable {
  int c[G::TASKS * G::NT];
  constexpr NumeratorTable() : c() {
    constexpr int H = G::H, R = G::R;
    int n = 0;
    auto box = [](int x, int y, int z) { return (x + H) * G::SX + (y + H) * G::SY + (z + H); };
    auto along_x = [&](int x, int y, int z) {
      c[n++] = box(x, y, z) | ((x * G::NYE + y + R) * G::NZE + z + R) << 12;
    };
    for (int x = 0; x < G::BX; ++x)
      for (int d = 0; d < 2 * R; ++d)
        for (int z = 0; z < G::BZ; ++z) along_x(x, d < R ? d - R : G::BY + d - R, z);
    for (int x = 0; x < G::BX; ++x)
      for (int y = 0; y < G::BY; ++y)
        for (int d = 0; d < 2 * R; ++d) along_x(x, y, d < R ? d - R : G::BZ + d - R);
    for (int x = 0; x < G::BX; ++x)
      for (int y = 0; y < G::BY; ++y)
        for (int d = 0; d < 2 * R; ++d) {
          const int z = d < R ? d - R : G::BZ + d - R;
          c[n++] = box(x, y, z) | (G::PX + (x * G::BY + y) * G::NZE + z + R) << 12 | 1 << 24;
        }
    while (n < G::TASKS * G::NT) {
      c[n] = c[0];
      ++n;
    }
  }
  static_assert(G::VOL <= 4096 && G::PX + G::PY <= 4096, "packed tasks");
};

template <class G>
__constant__ NumeratorTable<G> kNumerators = NumeratorTable<G>();

// Barrier of the workgroup that orders its LDS accesses (global loads and stores stay in
// flight across it).
__device__ __forceinline__ void group_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Source of fields and derivatives for bssn_rhs_point over a shared box: as WaveSrc with one
// field in flight, with workgroup barriers where WaveSrc relies on a wave's LDS order. Every lane of
// the workgroup must run the whole stage sequence (lanes without a point of their own stage cells
// for the others). WIDE: 64-bit addresses, for fields of 4 GiB and more.
template <int ORD, bool KO, int MODE, class ORDER = RhsOrder, bool WIDE = false>
struct GroupSrc : BoxStencil<GroupGeo<ORD, KO>, Coef<ORD>> {
  using G = GroupGeo<ORD, KO>;
  using Box = BoxStencil<G, Coef<ORD>>;
  using Box::c;
  using Box::lds;
  using Box::sc;
  static constexpr bool kWhole = std::is_same<ORDER, RhsOrder>::value;   // the whole equations
  static constexpr int kBoxes = kWhole ? G::BOXES : 1;
  static constexpr bool kNum = G::NUM || !kWhole;
  double* base;         // the workgroup's LDS
  double* num;          // first-derivative numerators of the brick and its extension
  int t;                // the lane
  int task[G::TASKS];
  bool mixed;           // the current field has mixed derivatives:
  double m1[2];         // its x and y numerators at the point
  const double* F;      // stencil source state (LINK: the pool)
  const double* Fc;     // the block's state (centre values)
  long P;
  unsigned off[G::PER]; // byte offsets of this lane's staged cells in a field (LINK: pool
                        // offsets in doubles, WIDE: offsets in doubles)
  int psrc[MODE == LINK ? G::PER : 1];   // LINK: field stride of each staged cell's block
  // box places (bytes) of this lane's staged cells, two in a word; the whole equations keep the
  // first TABLE words in LDS
  static constexpr int kTable = kWhole ? G::TABLE : 0;
  int cel[G::PAIRS];
  double pf[G::PER];    // the next field's cells, in flight
  // the lane's point, clamped into the grid, and the place of its centre value (the point, or its
  // periodic image): byte offsets in a field (WIDE: indices)
  std::conditional_t<WIDE, long, unsigned> gp, gc;
  static constexpr int kParkSlots = G::SLOTS;

  __device__ __forceinline__ GroupSrc(double* mem, const double* F_, const Scales& sc_,
                                      const Dims& d, int ox, int oy, int oz, int t_,
                                      int first = ORDER::at(0))
      : Box(mem, sc_), base(mem), num(mem + kBoxes * G::VOL), t(t_), F(F_), Fc(F_), P(d.P) {
    static_assert(MODE != LINK, "LINK sources take the pool and the link map");
    place(d, ox, oy, oz);
    const int o[3] = {ox, oy, oz};
#pragma unroll
    for (int k = 0; k < G::PER; ++k) {
      const int e = kCells<G>.c[t + k * G::NT];
      const int cc[3] = {e & 31, (e >> 5) & 31, (e >> 10) & 31};
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
                                      const Dims& d, int ox, int oy, int oz, int t_)
      : Box(mem, sc_), base(mem), num(mem + kBoxes * G::VOL), t(t_), F(pool), Fc(pool + boff), P(d.P) {
    static_assert(MODE == LINK, "the link constructor is for LINK sources");
    place(d, ox, oy, oz);
    const int o[3] = {ox, oy, oz};
#pragma unroll
    for (int k = 0; k < G::PER; ++k) {
      const int e = kCells<G>.c[t + k * G::NT];
      const int cc[3] = {e & 31, (e >> 5) & 31, (e >> 10) & 31};
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

  __device__ __forceinline__ void place(const Dims& d, int ox, int oy, int oz) {
    c = (G::lx(t) + G::H) * G::SX + (G::ly(t) + G::H) * G::SY + (G::lz(t) + G::H);
#pragma unroll
    for (int k = 0; k < G::PAIRS; ++k) {
      int w = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (2 * k + h < G::PER) {
          const int e = kCells<G>.c[t + (2 * k + h) * G::NT];
          w |= ((e & 31) * G::SX + ((e >> 5) & 31) * G::SY + ((e >> 10) & 31)) << (3 + 16 * h);
        }
      if (k < kTable)
        table()[k * G::NT] = w;
      else
        cel[k] = w;
    }
#pragma unroll
    for (int k = 0; k < G::TASKS; ++k) task[k] = kNumerators<G>.c[t + k * G::NT];
    gp = lane_point<G>(d, ox, oy, oz, t);
    gc = lane_centre<G, MODE>(d, ox, oy, oz, t);
    if constexpr (!WIDE) {
      gp <<= 3;
      gc <<= 3;
    }
  }

  __device__ __forceinline__ int* table() const {
    return reinterpret_cast<int*>(base + G::TABLE0) + pin(t);
  }
  // the lane's point in the x and y numerators
  __device__ __forceinline__ int ix() const {
    const int l = pin(t);
    return (G::lx(l) * G::NYE + G::ly(l) + G::R) * G::NZE + G::lz(l) + G::R;
  }
  __device__ __forceinline__ int iy() const {
    const int l = pin(t);
    return G::PX + (l / G::BZ) * G::NZE + G::lz(l) + G::R;
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

  // field f, loaded before, into the box; next: the field to load while f is used (-1: none)
  __device__ __forceinline__ void stage_in(int f, int next) {
    const int n = cells(f);
    mixed = ORDER::edges(f);
    if constexpr (kBoxes == 2)   // the boxes alternate: this one's last field was left a barrier ago
      lds = base + (ORDER::pos(f) & 1) * G::VOL;
    else
      group_barrier();           // every wave is done with the previous field
#pragma unroll
    for (int k = 0; k < G::PAIRS; ++k)
      if (2 * k < n) {
        const unsigned w = (unsigned)pin(k < kTable ? table()[k * G::NT] : cel[k]);
        *at_byte(lds, w & 0xffff) = pf[2 * k];
        if (2 * k + 1 < n) *at_byte(lds, w >> 16) = pf[2 * k + 1];
      }
    group_barrier();
    if (next >= 0) fetch(next);
    if (kNum && mixed) {
#pragma unroll
      for (int k = 0; k < G::TASKS; ++k) {
        const int w = pin(task[k]);      // unpacked here, not once for all fields
        num[(w >> 12) & 4095] = Box::n1s(w & 4095, (w >> 24) ? G::SY : G::SX);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a) m1[a] = pin(Box::n1(c, a));
      num[ix()] = m1[0];
      num[iy()] = m1[1];
      group_barrier();
    }
  }
  // With numerators the field after the metric is not loaded until the Ricci tensor is done
  // (after_ricci): that is where the most values are live, and the loads in flight would be spilled.
  __device__ __forceinline__ void stage(int f) {
    const int at = ORDER::pos(f);
    stage_in(f, at + 1 < ORDER::N && !(kNum && f == GT5) ? ORDER::at(at + 1) : -1);
  }
  __device__ __forceinline__ void resume() {
    if constexpr (kNum) fetch(ORDER::at(ORDER::pos(GT5) + 1));
  }

  __device__ __forceinline__ double d1(int a) const {
    return kNum && mixed && a < 2 ? pin(m1[a & 1] * sc.s1[a]) : Box::d1(a);
  }
  // second derivatives: fields with mixed derivatives only
  __device__ __forceinline__ double d2(int i, int j) const {
    if (!kNum || i == j) return Box::d2(i, j);
    const int at = i == 0 ? ix() : iy(), s = j == 1 ? G::NZE : 1;
    double acc = 0.0;
#pragma unroll
    for (int k = 1; k <= G::R; ++k)
      acc += Coef<ORD>::d1(k) * (num[at + k * s] - num[at - k * s]);
    return pin(acc * sc.sm[i + j - 1]);
  }

  __device__ __forceinline__ double center(int f) const {
    if constexpr (WIDE)
      return Fc[(long)f * P + gc];
    else
      return *at_byte(Fc + (long)f * P, gc);
  }
  __device__ __forceinline__ void park(int i, double x) {
    base[(kWhole ? G::SLOT0 : G::BOX_DOUBLES) + i * G::NT + pin(t)] = x;
  }
  __device__ __forceinline__ double parked(int i) const {
    return base[(kWhole ? G::SLOT0 : G::BOX_DOUBLES) + i * G::NT + pin(t)];
  }
};

template <int ORD, bool KO, int MODE, class ORDER, bool WIDE>
__device__ __forceinline__ void after_ricci(GroupSrc<ORD, KO, MODE, ORDER, WIDE>& s) {
  s.resume();
}

}  // namespace bssn
