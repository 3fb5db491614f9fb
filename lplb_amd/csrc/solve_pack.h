// Which batches of small LPs (G <= 16 and G * D <= 16) are solved four to a wave instead of one.  No other header here, so that
// the rule can be held against its figures on a CPU (tests/test_host.py).
//
// One LP per wave has the lowest latency; four to a wave take longer but need a quarter of the waves.  Alone on its SIMD a
// lone LP is the faster one throughout.  Up to 8 ranks its lanes are busy less than half the time, and it still is with three
// on a SIMD; four packed ones fill one wave of every SIMD and take no longer, then a second packed wave is behind until there
// are six or seven LPs per SIMD.  From 9 ranks on (16 pivots a step instead of 8) the second lone LP is already too many.
//
// How long a packed wave takes depends on the counts that one of its lanes reads: those of a whole rank, and a sixteenth
// of those that the wave fetches for its four LPs.  Measured, us a batch, one per wave / four per wave:
//    G, D   of a rank, in all      2048        3072        4096        5120        6144        7168        8192 LPs
//   (8, 2)    8    64     7.3 /  9.5   9.2 /  9.6  10.9 /  9.5  12.5 / 12.4  13.9 / 12.5  15.6 / 12.6  17.2 / 12.6
//   (8, 2)   32   256     7.8 / 10.7   9.7 / 10.7  11.2 / 11.0  12.7 / 14.4  14.3 / 14.8  16.0 / 15.2  17.5 / 15.4
//   (8, 2)    8   512     7.9 / 11.5   9.9 / 11.6  11.5 / 11.5  13.1 / 14.5  14.8 / 14.7  16.3 / 14.7  17.9 / 14.8
//   (8, 2)   32   512     8.1 / 11.9   9.9 / 11.9  11.5 / 12.2  13.0 / 15.6  14.9 / 16.1  16.3 / 16.5  17.9 / 16.7
//   (8, 2)    8  1024     8.6 / 14.0  10.8 / 14.1  12.3 / 14.1  13.8 / 16.8  15.5 / 17.0  20.3 / 17.3  21.8 / 17.4
//   (8, 2)   32  1024     9.0 / 14.4  10.7 / 14.4  12.3 / 14.6  13.9 / 18.0  15.8 / 18.4  21.1 / 18.9  23.6 / 19.3
//   (8, 2)   64   512     8.8 / 14.3  10.5 / 14.3  11.9 / 14.8  13.4 / 17.7  15.3 / 18.4  16.9 / 18.7  18.5 / 19.2
//   (8, 1)   32   256     7.7 /  9.9   9.3 / 10.1  10.8 / 10.2  12.3 / 13.2  13.8 / 13.8  15.6 / 14.1  16.8 / 14.3
//   (7, 2)   32   224     8.6 / 11.2  10.6 / 11.2  12.2 / 11.3  13.7 / 14.6  15.5 / 15.1  17.4 / 15.4  19.2 / 15.6   (padded)
//   (4, 2)   32   128     7.8 / 10.4   9.8 / 10.4  11.5 / 10.4  13.2 / 13.5  14.9 / 14.0  16.8 / 14.1  18.4 / 14.2   (padded)
//   (4, 2)   64   256     8.7 / 12.7  10.5 / 12.8  12.1 / 13.1  13.7 / 16.3  15.7 / 16.5  17.4 / 16.8  19.2 / 16.9   (padded)
//   (16, 1)  16   256    19.2 / 14.0  25.5 / 14.4  32.4 / 14.6  39.1 / 19.2  45.9 / 19.8  52.8 / 20.2  59.6 / 20.5
//   (16, 1)  16  1024    19.9 / 17.6  26.7 / 18.0  33.5 / 18.2  45.2 / 22.8  52.0 / 23.5  59.6 / 23.8  66.9 / 24.4
//   (10, 1)  25   250    20.3 / 17.6  27.1 / 17.7  34.1 / 18.2  40.7 / 22.7  48.1 / 23.1  55.1 / 23.7  62.1 / 24.2   (padded)
// (A number of LPs between two of these takes about as long as the larger one.)  Past 8192 packing stays ahead wherever it is
// ahead there, but for the first LPs beyond another four per SIMD at 48 experts of a rank and 8 ranks (9216: 20.2 / 20.5, 13312:
// 27.4 / 30.7) and from 10 to 12 per SIMD at 1024 experts (10240: 25.3 / 29.5); at 64 experts of a rank and 8 ranks the lone form is
// behind with 11 and 12 (12288: 25.4 / 23.4).
#pragma once

namespace lplb {

// n_experts: in all, of which per_rank are a rank's; per_simd: LPs for each SIMD, rounded up.
constexpr bool packing_pays(int G, int per_rank, int n_experts, int per_simd) {
  const int counts_of_a_lane = per_rank + n_experts / 16;
  return G > 8           ? per_simd > 1
         : per_simd == 4 ? counts_of_a_lane <= 48
         : per_simd == 6 ? counts_of_a_lane < 48
                         : per_simd > 6 && (per_rank <= 32 || counts_of_a_lane <= 84);
}

} // namespace lplb
