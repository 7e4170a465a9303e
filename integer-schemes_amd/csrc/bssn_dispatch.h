// Which of its two forms a kernel over bricks of grid points runs in: bricks of 64 points that a
// wave has to itself (WaveSrc, bssn_brick.h) or bricks of 256 points shared by four waves
// (GroupSrc, bssn_group.h). Host code only, without HIP, so that it can be tested as it stands.
#pragma once

namespace bssn {

// Points of a field from which its bytes no longer fit the shared form's 32-bit byte offsets
// (4 GiB). A bound of safety: those offsets wrap past it.
constexpr long long kGroupPoints = 1LL << 29;

// Bricks the chip runs at once: one wave-private brick per SIMD, two workgroups on a shared brick
// per compute unit, 256 compute units of four SIMDs. (On a device that shows fewer of them the
// rules below compare the forms at another number of rounds than they run; that costs time only.)
constexpr long kWaveSlots = 4 * 256;
constexpr long kGroupSlots = 2 * 256;

// Whether `groups` shared bricks take less time than `waves` wave-private bricks over the same
// points. Both run in rounds of as many as fit the chip; the last round of shared bricks counts
// 0.7 if it leaves one workgroup per compute unit (measured 0.6 to 0.75), and a launch of at most
// half a round of wave-private ones 0.75 (0.7 to 0.8). cost: what a full round
// of shared bricks (twice the lanes) takes, in rounds of wave-private ones. Counting rounds and
// not points covers both ways of wasting a shared brick: lanes without a point (its 16 points
// along z on a grid of 8) and a last round nearly empty (48 x 48 x 56 is two wave-private rounds
// full, and 64 shared bricks more than one).
constexpr bool shared_pays(double cost, long waves, long groups) {
  const long rest = groups % kGroupSlots;
  const double shared =
      (double)(groups / kGroupSlots) + (rest == 0 ? 0.0 : (rest <= kGroupSlots / 2 ? 0.7 : 1.0));
  return cost * shared <=
         (2 * waves <= kWaveSlots ? 0.75 : (double)((waves + kWaveSlots - 1) / kWaveSlots));
}

// The fused kernels (a single grid's or a batch's, over the points of one launch). At most one
// round of wave-private bricks is one brick's latency long either way, and theirs is the shorter
// (no barriers, more registers): FD4 RK4 step at 24^3 / 32^3 / 40^3 (1000 bricks) 115 / 127 / 155
// us against 135 / 141 / 192 us.
// The costs are fitted to both forms forced on 44 grids and 16 batches (wave-private / shared
// time, > 1: shared wins). Near the line, with the rounds (wave-private, shared):
//   FD4 RHS, 1.44:  39x82x75 (4, 2.7) 1.05, 256x256x12 (12, 8) 1.02, 60 padded blocks of 22^3 (13,
//     9) 1.03, 56^3 (3, 2) 0.99; 103x66x33 (4, 3) 0.91, 200x200x20 (13, 10) 0.88, 48x48x56 (2,
//     1.7) 0.83, 160x160x8 (4, 3.7) 0.73
//   FD4 step and FD6 step or RHS with Kreiss-Oliger terms, 1.19:  200x200x20 1.10, 1.04, 1.08;
//     160x160x20 (8, 6.7) 1.06, 1.05, 1.02; 103x66x33 1.01, 1.06, 1.11; 48x48x56 0.94, 0.95,
//     1.03; 100x100x8 (2, 1.7) 0.91, 0.94, 0.96; 160x160x8 0.88, 0.91, 0.90
//   FD6 without them, 1.11:  RHS and step, 200x200x20 1.14, 1.12; 48x48x56 1.07, 1.03; 100x100x8
//     1.01, 1.01; 160x160x8 0.95, 0.98; 256x256x8 (8, 8) 0.94, 0.98
//   FD8, 1:  160x160x8 1.07 (RHS) and 1.10 (step), 256x256x8 1.02 and 1.06, 48x48x56 1.19 and
//     1.13; 256x256x4 (4, 8) 0.52 and 0.62. RHS with Kreiss-Oliger terms 1.05: 0.99, 0.93, 1.11.
//     Batches 1.03: 500 blocks of 8^3 (4, 4) 0.99, 20 of 48x48x8 (6, 6) 0.98
constexpr bool fused_shared(int ord, bool rhs, bool ko, bool batch, long waves, long groups) {
  const double cost = ord == 4   ? (rhs ? 1.44 : 1.19)
                      : ord == 6 ? (ko ? 1.19 : 1.11)
                                 : (rhs && ko ? 1.05 : (batch ? 1.03 : 1.0));
  return waves > kWaveSlots && shared_pays(cost, waves, groups);
}

// The constraints, whose 24^3 and 32^3 samples of long runs are single rounds: FD4 24^3 / 32^3 /
// 40^3 11.5 / 12.0 / 13.7 us wave-private, 14.7 / 14.7 / 19.3 shared; FD6 15.8 / 16.6 / 19.7 and
// 17.3 / 17.4 / 23.5; FD8 20.7 / 21.8 / 26.6 and 21.0 / 21.1 / 29.4. Near the line
// (wave-private / shared time): FD4 39x82x75 1.08, 128x128x24 1.06, 64x64x16 0.95, 103x66x33
// 0.91, 48x48x56 0.82; FD6 64x64x12 1.07, 160x160x17 1.01, 45x45x52 0.97, 160x160x8 0.89; FD8
// 72x72x20 1.07, 100x100x8 1.05, 160x160x8 0.97, 256x256x8 0.90.
constexpr bool constraints_shared(int ord, long waves, long groups) {
  return shared_pays(ord == 4 ? 1.44 : (ord == 6 ? 1.19 : 1.1), waves, groups);
}

// The derivative bundle. The shared bricks write longer rows and few arrays at a time, so they win
// at every size (12^3 FD4 18.0 -> 5.8 us) unless half of their lanes or more have no point: arrays
// of up to 8 points along z, of more than one round of wave-private bricks at FD4, of two above.
// (wave-private / shared, FD4 fp64, BFP32 and FD6 fp64, BFP32): 256x256x8 1.09, 0.68, 0.90, 0.73;
// 160x160x8 1.16, 0.61, 0.92, 0.92; 100x100x8 0.90, 0.92, 1.10, 1.11; 256x256x4 0.53, 0.28, 0.51,
// 0.39; 160x160x17 1.48, 1.14, 1.41, 0.96. The maxima are faster shared at every size but of four
// points along z above FD4 (256x256x4 FD6 0.86, 160x160x8 1.58), narrower than their stencils.
constexpr bool bundle_shared(int ord, bool fp64, long waves, long groups) {
  if (ord == 4 && fp64) return groups < waves || waves <= kWaveSlots;
  return 2 * groups < waves || waves <= (ord == 4 ? 1 : 2) * kWaveSlots;
}

}  // namespace bssn
