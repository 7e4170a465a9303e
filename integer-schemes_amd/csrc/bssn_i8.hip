// INT8-split derivative bundle (Ozaki scheme I on the INT8 matrix cores) for FD order 4.
//
// Precision form of the derivative bundle (3D/src/bssn3d/derivative_bundle.py:31-48): the
// 138 derivatives are taken from 2D slabs of one field, and on each slab the stencil is applied
// as a banded integer matrix by INT8 MFMA with INT32 accumulation, on int8 digits of the values.
// The reference's precision form (Ozaki scheme II with residues and CRT, for its Maxwell-Chern-
// Simons solver only: 2D/src/mcs2d/schemes/ozaki.py:257-562, 3D/src/mcs3d/schemes/ozaki.py:
// 162-282) contributes the per-block power-of-two scale (ozaki.py:316-323) and the banded
// stencil matrix (ozaki.py:286-306); the digits here are an Ozaki-I split instead of residues.
//
// One wave computes a 28 x 28 tile of outputs of one plane of one field from the 32 x 32 box
// around it (coordinates clamped to the grid, the reference's edge padding):
//   box values v -> c = 0.5 max + 0.5 min (stencils annihilate constants), sigma = 2^(6-E) with
//   max|v - c| = f 2^E, r0 = (v - c) sigma, q_s = rint(r_s), r_{s+1} = 128 (r_s - q_s):
//   |q_s| <= 64, every step exact; (v - c) sigma = sum_s q_s 2^(-7 s) + O(2^(-7 k)).
//   The k <= 7 digits are taken in groups of three (0..2, 3..5, and the last by itself where that
//   leaves one), each as one integer
//   N = rint(r 2^(7 (g - 1))) = sum_s q_s 2^(7 (g - 1 - s)) (g digits; the remainder is the same,
//   and a tie falls the same way), whose signed bytes are the int8 operands (32 x 32 planes):
//     B N   (rows: outputs along axis 1)   = sum of v_mfma_i32_32x32x32_i8(band, byte plane)
//     N B^T (columns: outputs along axis 2) = the same with N^T, transposed as words via LDS
//     B N B^T (mixed): the INT32 B N (25 bits and sign) in its four signed bytes, each times B^T
//   INT32 holds every exact result (the mixed one: 18 * 18 * 64 * 2^14.02 < 2^29).
//   Recombination in FP64: acc += P_g 2^(-7 s), s the group's last digit; D = (acc 2^-e) * scale.
//   The sums of digits 0..5 are exact in FP64 (at most 15 + 35 bits), so the only rounding is
//   that of digit 6, as if the digits had been added one by one.
// The integer stencils are those of common/src/mcs_common/derivatives.py:33-49 times 12
// (first and second derivatives) and 144 (mixed).
//
// Plane orientations: (y, z) planes at each x give d_y, d_yy, d_z, d_zz, d_yz; (x, z) planes at
// each y give d_x, d_xx, d_xz; (x, y) planes at each z give d_xy.
#include <hip/hip_runtime.h>

#include <math.h>

#include <type_traits>

#include "bssn_kernels.h"
#include "bssn_params.h"

namespace bssn {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int I8_TILE = 28, I8_BOX = 32;

// fields with second derivatives (alpha, chi, gt0..5, beta0..2) and the others
__constant__ int kTwoFields[11] = {ALPHA, CHI, GT0, GT1, GT2, GT3, GT4, GT5, BETA0, BETA1, BETA2};
__constant__ int kOneFields[13] = {KTR, AT0, AT1, AT2, AT3, AT4, AT5, GTI0, GTI0 + 1, GTI0 + 2,
                                   BB0, BB1, BB2};

// taps at offsets -2..2 (index t = 0..4)
__device__ __forceinline__ int tap1(int t) {
  return t == 0 ? 1 : (t == 1 ? -8 : (t == 3 ? 8 : (t == 4 ? -1 : 0)));
}
__device__ __forceinline__ int tap2(int t) {
  return (t == 0 || t == 4) ? -1 : ((t == 1 || t == 3) ? 16 : -30);
}

// The lane's 16 bytes of the banded matrix: row r = lane % 32 (an output), positions
// k = 16 (lane / 32) + j. The same bytes serve as the A operand B (rows r) and as the
// B operand B^T (columns r).
template <int W>
__device__ __forceinline__ v4i band_operand(int lane) {
  const int r = lane & 31, k0 = 16 * (lane >> 5);
  unsigned w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int t = k0 + j - r;
    int v = 0;
    if (r < I8_TILE && t >= 0 && t <= 4) v = W == 1 ? tap1(t) : tap2(t);
    w[j >> 2] |= ((unsigned)v & 0xffu) << (8 * (j & 3));
  }
  return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// Byte planes of 16 words: plane b holds byte b of each, in order.
template <int NP>
__device__ __forceinline__ void byte_planes(const int* w, v4i* plane) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int* a = w + 4 * g;
    const unsigned lo01 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u);
    const unsigned lo23 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u);
    plane[0][g] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    if constexpr (NP > 1) plane[1][g] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    if constexpr (NP > 2) {
      const unsigned hi01 = __builtin_amdgcn_perm(a[1], a[0], 0x07030602u);
      const unsigned hi23 = __builtin_amdgcn_perm(a[3], a[2], 0x07030602u);
      plane[2][g] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
      if constexpr (NP > 3) plane[3][g] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
    }
  }
}

// v as NP signed bytes: v = sum_b byte_b 256^b (|v| < 2^(8 NP - 1) - 2^(8 NP - 8))
template <int NP>
__device__ __forceinline__ int signed_bytes(int v) {
  constexpr int h = NP == 1 ? 0 : (NP == 2 ? 0x80 : (NP == 3 ? 0x8080 : 0x808080));
  return (v + h) ^ h;
}

// The contraction of a matrix of signed bytes (NP planes) with the band: rows (band times the
// matrix, planes in the B distribution) or columns (the matrix times band^T, A distribution).
template <int NP, bool ROWS>
__device__ __forceinline__ v16i contract(const v4i& band, const v4i* plane) {
  const v16i z16 = {};
  v16i sum = z16;
#pragma unroll
  for (int b = NP - 1; b >= 0; --b) {
    const v16i p = ROWS ? __builtin_amdgcn_mfma_i32_32x32x32_i8(band, plane[b], z16, 0, 0, 0)
                        : __builtin_amdgcn_mfma_i32_32x32x32_i8(plane[b], band, z16, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i)   // the partial sums may wrap, the result does not
      sum[i] = b == NP - 1 ? p[i] : (int)(((unsigned)sum[i] << 8) + (unsigned)p[i]);
  }
  return sum;
}

typedef v4i __attribute__((may_alias)) v4i_lds;
// 32 x 32 words; the rows' starts, 36 words apart, lie on 16 different groups of 4 banks
constexpr int I8_PITCH = 36;

// row r = lane % 32, positions 16 (lane / 32) + j of the words in t, as byte planes
template <int NP>
__device__ __forceinline__ void row_planes(const int* t, int lane, v4i* plane) {
  int w[16];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const v4i x = *(const v4i_lds*)&t[(lane & 31) * I8_PITCH + 16 * (lane >> 5) + 4 * g];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[4 * g + j] = x[j];
  }
  __builtin_amdgcn_wave_barrier();
  byte_planes<NP>(w, plane);
}

__device__ __forceinline__ double wave_max(double x) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) x = fmax(x, __shfl_xor(x, m, 64));
  return x;
}
__device__ __forceinline__ double wave_min(double x) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) x = fmin(x, __shfl_xor(x, m, 64));
  return x;
}

// C-layout of the 32 x 32 result: lane holds column lane % 32, rows row_of(i, lane)
__device__ __forceinline__ int row_of(int i, int lane) {
  return 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
}

struct I8Args {
  const double* F;
  double* D;
  int S[3];
  long P;
  double s1[3], s2[3], sm[3];
  int nslice;
};

// Launch geometry of one (ORIENT, TWO) pass over a grid of padded extents S: the number of
// wave tiles (fields x tiles along the plane's two axes x planes).
template <int ORIENT, bool TWO>
__host__ __device__ inline long i8_tiles(const int* S) {
  const int ax1 = ORIENT == 0 ? 1 : 0, ax2 = ORIENT == 2 ? 1 : 2;
  const int axp = ORIENT == 0 ? 0 : (ORIENT == 1 ? 1 : 2);
  const long nt1 = (S[ax1] + I8_TILE - 1) / I8_TILE, nt2 = (S[ax2] + I8_TILE - 1) / I8_TILE;
  return (TWO ? 11L : 13L) * nt1 * nt2 * S[axp];
}

// ORIENT 0: (y, z) planes at each x; 1: (x, z) planes at each y; 2: (x, y) planes at each z.
// TWO: the fields with second derivatives (else first derivatives only). ONE: a single digit,
// which as a group of three is multiplied as three byte planes (16^3 / 64^3: 40.5 / 176 -> 35.3 /
// 139 us, the same in one plane).
// One wave: tile w of the grid a, in the order below.
template <int ORIENT, bool TWO, bool ONE>
__device__ __forceinline__ void i8_tile(const I8Args& a, long w, int lane, int* t) {
  constexpr int AX1 = ORIENT == 0 ? 1 : 0;
  constexpr int AX2 = ORIENT == 2 ? 1 : 2;
  constexpr int AXP = ORIENT == 0 ? 0 : (ORIENT == 1 ? 1 : 2);
  constexpr bool D1A = ORIENT != 2;                 // first derivative along axis 1
  constexpr bool D2A = TWO && ORIENT != 2;          // second derivative along axis 1
  constexpr bool D1B = ORIENT == 0;                 // along axis 2 (z, from the (y, z) planes)
  constexpr bool D2B = TWO && ORIENT == 0;
  constexpr bool MIX = TWO;
  constexpr int NF = TWO ? 11 : 13;

  const int n1 = a.S[AX1], n2 = a.S[AX2], npl = a.S[AXP];
  const long st[3] = {(long)a.S[1] * a.S[2], (long)a.S[2], 1L};
  const int nt1 = (n1 + I8_TILE - 1) / I8_TILE, nt2 = (n2 + I8_TILE - 1) / I8_TILE;
  // (y, z) and (x, z) planes: tiles along z fastest, so the lines that two of them share are
  // complete before they leave L2; (x, y) planes: planes (along z) fastest
  int pl, t1, t2;
  if constexpr (ORIENT == 2) {
    pl = (int)(w % npl);
    w /= npl;
    t2 = (int)(w % nt2);
    w /= nt2;
    t1 = (int)(w % nt1);
    w /= nt1;
  } else {
    t2 = (int)(w % nt2);
    w /= nt2;
    t1 = (int)(w % nt1);
    w /= nt1;
    pl = (int)(w % npl);
    w /= npl;
  }
  const int fi = (int)w;
  if (fi >= NF) return;
  const int f = TWO ? kTwoFields[fi] : kOneFields[fi];
  const int o1 = t1 * I8_TILE, o2 = t2 * I8_TILE;
  const double* u = a.F + (long)f * a.P + (long)pl * st[AXP];

  // box values in the B-operand distribution: column c = lane % 32, rows 16 (lane / 32) + j
  const int c = lane & 31, hh = lane >> 5;
  int i2 = o2 - 2 + c;
  i2 = i2 < 0 ? 0 : (i2 > n2 - 1 ? n2 - 1 : i2);
  double r[16];
  double mx = -INFINITY, mn = INFINITY;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    int i1 = o1 - 2 + 16 * hh + j;
    i1 = i1 < 0 ? 0 : (i1 > n1 - 1 ? n1 - 1 : i1);
    r[j] = u[(long)i1 * st[AX1] + (long)i2 * st[AX2]];
    mx = fmax(mx, r[j]);
    mn = fmin(mn, r[j]);
  }
  mx = wave_max(mx);
  mn = wave_min(mn);
  const double off = 0.5 * mx + 0.5 * mn;
  double m = 0.0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    r[j] = r[j] - off;
    m = fmax(m, fabs(r[j]));
  }
  m = wave_max(m);
  int e = 0;
  if (m != 0.0) {
    int E;
    (void)frexp(m, &E);
    e = 6 - E;
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) r[j] = ldexp(r[j], e);

  if (m == INFINITY) {   // infinities have no digits: what the saturating conversion leaves
#pragma unroll
    for (int j = 0; j < 16; ++j) r[j] = r[j] == INFINITY ? -1.0 : 0.0;
  }

  // the groups of ns digits: 0..na-1 (ONE: none), 3..nb+2 (from five), and the last digit by
  // itself where threes leave one
  const int ns = a.nslice, na = ns < 3 ? ns : 3, nb = ns < 6 ? ns - na : 3;
  const bool more = !ONE && ns > 4, last = ONE || ns % 3 == 1;
  v4i qa[3], qb[3], qc[1], ta[3], tb[3], tc[1];   // byte planes of N and of N^T
  constexpr bool COLS = D1B || D2B;
  auto digits = [&](auto np, int g, v4i* q, v4i* tr) {
    constexpr int NP = decltype(np)::value;
    const double up = ldexp(1.0, 7 * (g - 1));
    int n[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const double x = r[j] * up, d = rint(x);
      r[j] = (x - d) * 128.0;
      n[j] = signed_bytes<NP>((int)d);
    }
    byte_planes<NP>(n, q);
    if constexpr (COLS) {
#pragma unroll
      for (int j = 0; j < 16; ++j) t[(16 * hh + j) * I8_PITCH + c] = n[j];
      __builtin_amdgcn_wave_barrier();
      row_planes<NP>(t, lane, tr);
    }
  };
  if constexpr (!ONE) digits(std::integral_constant<int, 3>(), na, qa, ta);
  if (more) digits(std::integral_constant<int, 3>(), nb, qb, tb);
  if (last) digits(std::integral_constant<int, 1>(), 1, qc, tc);
  const double wa = ldexp(1.0, -7 * (na - 1)), wb = ldexp(1.0, -7 * (na + nb - 1)),
               wc = ldexp(1.0, -7 * (ns - 1));
  double acc[16];
  auto add = [&](const v16i& p, double ws) {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = acc[i] + (double)p[i] * ws;
  };
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0;
  };
  const v4i band1 = band_operand<1>(lane);
  const v4i band2 = band_operand<2>(lane);

  // outputs: rows along axis 1, columns along axis 2 (lane's column c, rows row_of(i))
  double* Dp = a.D;
  const long plo = (long)pl * st[AXP];
  auto put = [&](int d, const double* acc, double scale, bool rows_out, bool cols_out) {
    double* dst = Dp + (long)d * a.P + plo;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int rr = row_of(i, lane);
      const int g1 = rows_out ? o1 + rr : o1 + rr - 2;
      const int g2 = cols_out ? o2 + c : o2 + c - 2;
      const bool ok1 = rows_out ? rr < I8_TILE : (rr >= 2 && rr < I8_TILE + 2);
      const bool ok2 = cols_out ? c < I8_TILE : (c >= 2 && c < I8_TILE + 2);
      if (ok1 && ok2 && g1 < n1 && g2 < n2)
        dst[(long)g1 * st[AX1] + (long)g2 * st[AX2]] = ldexp(acc[i], -e) * scale;
    }
  };
  const int slot = TWO ? fi : -1;
  auto columns = [&](const v4i& band) {
    clear();
    if constexpr (!ONE) add(contract<3, false>(band, ta), wa);
    if (more) add(contract<3, false>(band, tb), wb);
    if (last) add(contract<1, false>(band, tc), wc);
  };
  if constexpr (D1B) {
    columns(band1);
    put(3 * f + AX2, acc, a.s1[AX2], false, true);
  }
  if constexpr (D2B) {
    columns(band2);
    put(72 + 6 * slot + 5, acc, a.s2[AX2], false, true);
  }
  auto rows = [&](const v4i& band) {
    clear();
    if constexpr (!ONE) add(contract<3, true>(band, qa), wa);
    if (more) add(contract<3, true>(band, qb), wb);
    if (last) add(contract<1, true>(band, qc), wc);
  };
  if constexpr (D1A) {
    rows(band1);
    put(3 * f + AX1, acc, a.s1[AX1], true, false);
  }
  if constexpr (D2A) {
    rows(band2);
    put(72 + 6 * slot + (AX1 == 0 ? 0 : 3), acc, a.s2[AX1], true, false);
  }
  if constexpr (MIX) {
    // B N as signed bytes through LDS (forming it again costs less than keeping it)
    auto mixed = [&](auto np, const v16i& p, double ws) {
      constexpr int NP = decltype(np)::value;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        t[row_of(i, lane) * I8_PITCH + c] = signed_bytes<NP>(p[i]);
      __builtin_amdgcn_wave_barrier();
      v4i pl[NP];
      row_planes<NP>(t, lane, pl);
      add(contract<NP, false>(band1, pl), ws);
    };
    clear();
    if constexpr (!ONE) mixed(std::integral_constant<int, 4>(), contract<3, true>(band1, qa), wa);
    if (more) mixed(std::integral_constant<int, 4>(), contract<3, true>(band1, qb), wb);
    if (last) mixed(std::integral_constant<int, 2>(), contract<1, true>(band1, qc), wc);
    // pair index of (AX1, AX2): xy 1, xz 2, yz 4; scale index AX1 + AX2 - 1
    const int pair = AX1 == 0 ? (AX2 == 1 ? 1 : 2) : 4;
    put(72 + 6 * slot + pair, acc, a.sm[AX1 + AX2 - 1], true, true);
  }
}

#define BSSN_I8_LDS __shared__ __attribute__((aligned(16))) int t[I8_BOX * I8_PITCH]

// Workgroup -> tile, XCD-aware: the dispatcher deals workgroups round-robin over the 8 XCDs;
// remap so that each XCD takes a contiguous run of tiles (consecutive planes), whose loads and
// stores share cache lines along the plane axis (a line of 16 doubles along z holds the same
// point of 16 consecutive (x, y) planes). The grid is a multiple of 8; tiles past the last are
// empty (i8_tile returns on them).
__device__ __forceinline__ long xcd_tile() {
  const long G8 = (long)gridDim.x;
  const long w = (long)blockIdx.x;
  return (w & 7) * (G8 >> 3) + (w >> 3);
}

// What bounds the passes is the stores, rows of 28 doubles that start anywhere in a line, and the
// waits at two waves per SIMD. Taking the digits in groups of three (a third of the FP64
// conversions and sums, words instead of bytes through LDS, for 45 instead of 42 matrix products)
// and one output array at a time (16 sums live instead of 80: two waves per SIMD instead of one)
// took the five passes of a 166^3 state from 3.5 to 3.0 ms, the order of the tiles (i8_tile) from
// 3.0 to 2.6 ms: (y, z) planes 0.89 -> 0.70 and 0.51 -> 0.38, (x, z) planes 0.62 -> 0.57 and
// 0.34 -> 0.31, (x, y) planes 0.64 ms. Three or four waves per SIMD spill where second derivatives
// are taken (0.70 -> 0.85 and 1.11 ms); the first-derivative pass on (x, z) planes has the room
// for four (0.31 -> 0.26 ms).
template <int ORIENT, bool TWO, bool ONE>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(ORIENT == 1 && !TWO ? 4 : 1)))
void k_i8_plane(I8Args a) {
  BSSN_I8_LDS;
  i8_tile<ORIENT, TWO, ONE>(a, xcd_tile(), (int)threadIdx.x, t);
}

// The same pass over every block of a batch: block b owns wave tiles [pre[b], pre[b + 1]) of
// the launch; its bundle is the 138 arrays at D + blk[b].doff and its stencil scales are formed
// from its spacings with the host's rounding, so each block's bundle equals the single-grid
// bundle of that block bit for bit.
template <int ORIENT, bool TWO, bool ONE>
__global__ __launch_bounds__(64) void k_i8_plane_batch(const double* pool, double* D,
                                                       const BlockDesc* __restrict__ blks,
                                                       const long long* __restrict__ pre,
                                                       int nblk, int nslice) {
  BSSN_I8_LDS;
  const long long w = (long long)xcd_tile();
  int lo = 0, hi = nblk;                 // pre[lo] <= w < pre[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (pre[mid] <= w) lo = mid;
    else hi = mid;
  }
  const int b = __builtin_amdgcn_readfirstlane(lo);
  const BlockDesc blk = blks[b];
  I8Args a;
  a.F = pool + blk.off;
  a.D = D + blk.doff;
  for (int i = 0; i < 3; ++i) a.S[i] = blk.S[i];
  a.P = (long)blk.S[0] * blk.S[1] * blk.S[2];
  const Scales sc = make_scales(blk.h, 4, 0.0);
  for (int i = 0; i < 3; ++i) {
    a.s1[i] = uniform(sc.s1[i]);
    a.s2[i] = uniform(sc.s2[i]);
    a.sm[i] = uniform(sc.sm[i]);
  }
  a.nslice = nslice;
  i8_tile<ORIENT, TWO, ONE>(a, (long)(w - pre[b]), (int)threadIdx.x, t);
}

template <int ORIENT, bool TWO>
static hipError_t launch_i8_t(const I8Args& a, hipStream_t st) {
  const long n = (i8_tiles<ORIENT, TWO>(a.S) + 7) & ~7L;
  if (n > 0x7fffffffL) return hipErrorInvalidValue;
  if (a.nslice == 1)
    hipLaunchKernelGGL((k_i8_plane<ORIENT, TWO, true>), dim3((unsigned)n), dim3(64), 0, st, a);
  else
    hipLaunchKernelGGL((k_i8_plane<ORIENT, TWO, false>), dim3((unsigned)n), dim3(64), 0, st, a);
  return hipGetLastError();
}

// wave tiles of pass k (0: (y,z) planes, fields with second derivatives; 1: (y,z), the others;
// 2, 3: the same on (x,z) planes; 4: (x,y) planes, mixed d_xy) on a grid of padded extents S
long i8_pass_tiles(int k, const int* S) {
  switch (k) {
    case 0: return i8_tiles<0, true>(S);
    case 1: return i8_tiles<0, false>(S);
    case 2: return i8_tiles<1, true>(S);
    case 3: return i8_tiles<1, false>(S);
    default: return i8_tiles<2, true>(S);
  }
}

template <int ORIENT, bool TWO>
static hipError_t launch_i8_batch_t(const double* pool, double* D, const BlockDesc* blk,
                                    const long long* pre, long long n, int nblk, int nslice,
                                    hipStream_t st) {
  if (n == 0) return hipSuccess;
  n = (n + 7) & ~7LL;
  if (n > 0x7fffffffLL) return hipErrorInvalidValue;
  if (nslice == 1)
    hipLaunchKernelGGL((k_i8_plane_batch<ORIENT, TWO, true>), dim3((unsigned)n), dim3(64), 0, st,
                       pool, D, blk, pre, nblk, nslice);
  else
    hipLaunchKernelGGL((k_i8_plane_batch<ORIENT, TWO, false>), dim3((unsigned)n), dim3(64), 0, st,
                       pool, D, blk, pre, nblk, nslice);
  return hipGetLastError();
}

// the five passes over a batch; pre: 5 prefix arrays of nblk + 1 entries (device), total: the
// five tile counts (host)
hipError_t launch_batch_bundle_i8(const double* pool, double* D, const BlockDesc* blk,
                                  const long long* pre, const long long* total, int nblk,
                                  int nslice, hipStream_t st) {
  const long long* p = pre;
  const long long m = nblk + 1;
  hipError_t e;
  if ((e = launch_i8_batch_t<0, true>(pool, D, blk, p, total[0], nblk, nslice, st))) return e;
  if ((e = launch_i8_batch_t<0, false>(pool, D, blk, p + m, total[1], nblk, nslice, st))) return e;
  if ((e = launch_i8_batch_t<1, true>(pool, D, blk, p + 2 * m, total[2], nblk, nslice, st)))
    return e;
  if ((e = launch_i8_batch_t<1, false>(pool, D, blk, p + 3 * m, total[3], nblk, nslice, st)))
    return e;
  return launch_i8_batch_t<2, true>(pool, D, blk, p + 4 * m, total[4], nblk, nslice, st);
}

hipError_t launch_deriv_bundle_i8(const double* F, double* D, const Dims& d, const Scales& w,
                                  int nslice, hipStream_t st) {
  I8Args a;
  a.F = F;
  a.D = D;
  for (int i = 0; i < 3; ++i) {
    a.S[i] = d.S[i];
    a.s1[i] = w.s1[i];
    a.s2[i] = w.s2[i];
    a.sm[i] = w.sm[i];
  }
  a.P = d.P;
  a.nslice = nslice;
  hipError_t e;
  if ((e = launch_i8_t<0, true>(a, st)) != hipSuccess) return e;
  if ((e = launch_i8_t<0, false>(a, st)) != hipSuccess) return e;
  if ((e = launch_i8_t<1, true>(a, st)) != hipSuccess) return e;
  if ((e = launch_i8_t<1, false>(a, st)) != hipSuccess) return e;
  return launch_i8_t<2, true>(a, st);
}

}  // namespace bssn
