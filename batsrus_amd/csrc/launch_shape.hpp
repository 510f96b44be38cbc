// launch_shape.hpp -- how many workgroups of the stage kernel a compute unit
// holds, and into how many parts a launch cuts the blocks' planes when the
// caller sets no shape.  Host arithmetic only.
#pragma once

namespace bats {

// LDS of a workgroup of the stage kernel (bytes): the haloed plane of its
// blocks and the fluxes of their x and y faces, with the 8-wave source in the
// body variant, or where it fits, the faces' normal field states
constexpr int kLdsPerCu = 160 * 1024;
constexpr int stage_lds(int NB, int elemSize, bool normalField) {
  const int blocks = 256 / (NB * NB);
  return blocks * (8 * (NB + 4) * (NB + 5) +
                   2 * (normalField ? 11 : 9) * (NB + 1) * NB) * elemSize +
         (256 / 64) * 8;
}
// workgroups that a compute unit is to hold (registers): two, three in FP32
constexpr int stage_want_per_cu(int elemSize) { return elemSize == 4 ? 3 : 2; }
constexpr bool stage_normal_field(int NB, int elemSize, bool wave8, bool body) {
  return wave8 && (body || stage_lds(NB, elemSize, true) *
                                   stage_want_per_cu(elemSize) <= kLdsPerCu);
}
// and those that the LDS lets it hold: one for the 8^3 body variant with the
// 8-wave source
constexpr int stage_per_cu(int NB, int elemSize, bool wave8, bool body) {
  const int lds =
      stage_lds(NB, elemSize, stage_normal_field(NB, elemSize, wave8, body));
  const int fit = kLdsPerCu / lds, want = stage_want_per_cu(elemSize);
  return fit < want ? fit : want;
}

// Time that nItem workgroups of one length take on 256 CUs of perCu places,
// in units of the time of a round that fills all places.  Measured: a CU with
// one workgroup of two is done with it sooner than with both, and each step
// of 256 costs a little more at its end than at its start; far beyond the
// places the workgroups no longer start together and only the last one's tail
// shows.
inline double launch_rounds(long nItem, int perCu) {
  const double x = (double)nItem / 256.0;
  const int n = (int)((nItem + 255) / 256);   // workgroups of the fullest CU
  const double r = x - (n - 1);               // how far into this step
  if (perCu == 1) return n <= 6 ? n - 0.17 * (1.0 - r) : x + 0.3;
  if (perCu == 2) {
    static const double step[6][2] = {{0.62, 0.74}, {0.87, 1.00}, {1.52, 1.70},
                                      {1.75, 1.90}, {2.40, 2.66}, {2.64, 2.89}};
    return n <= 6 ? step[n - 1][0] + (step[n - 1][1] - step[n - 1][0]) * r
                  : 0.425 * x + 0.48;
  }
  static const double third[3] = {0.68, 0.83, 1.00};
  return n <= 9 ? (n - 1) / 3 + third[(n - 1) % 3] : x / 3.0 + 0.35;
}

// Parts (2^shift) of the blocks of nGroup workgroups.  A workgroup marches
// through its planes one behind the other, whatever else runs: a grid of few
// blocks is done sooner in shorter parts, until all the places of the chip
// are taken, and a grid of a few times the places ends with a nearly empty
// last round that shorter parts fill.  Each part has the z face below its
// first plane to itself and starts anew: about 0.85 of a plane's time, 0.72
// with one place per CU, 0.55 in FP32 (0.75 with the 8-wave source).  The least
// of rounds times planes is taken, with two places only where it promises 5 %
// over whole blocks.  Over 1 to 2048 workgroups in steps of at most a quarter
// (FP64 Rusanov, HLLD, with the 8-wave source, B0 and the body) that is
// nowhere slower than whole blocks but for Rusanov on 1200 workgroups of 8^3
// blocks (1.04 of their time), at most 1.06 and in the mean 1.002 of the best
// shape's time; FP32 (HLLD, Rusanov with the 8-wave source) 1.02, 1.10 and
// 1.002.  Measured per launch, whole blocks against the rule's parts, HLLD:
// 8^3, 16 groups 76 -> 19 us, 128 groups 78 -> 40, 396 groups whole 106 (parts
// of two planes 119); 16^3, 64 groups 135 -> 35, 256 groups 136 -> 96, 512 and
// 1024 groups whole (182 and 382, in halves 192 and 394); 8^3 with body, B0
// and 8-wave source, 54 groups 127 -> 44 (one plane per part, right for two
// places per CU, 55).
inline int auto_split(int nGroup, int NB, int perCu, bool wave8) {
  const double start = perCu == 1 ? 0.72 : perCu == 2 ? 0.85
                       : wave8 ? 0.75 : 0.55;
  int best = 0;
  double least = 0.0;
  for (int s = 0; (NB >> s) >= 1; s++) {
    const double cost =
        launch_rounds((long)nGroup << s, perCu) * ((NB >> s) + start);
    if (s == 0) {
      least = perCu == 2 ? 0.95 * cost : cost;
    } else if (cost < least) {
      least = cost;
      best = s;
    }
  }
  return best;
}

}  // namespace bats
