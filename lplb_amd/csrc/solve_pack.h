// Which batches of small LPs (G <= 16 and G * D <= 16) are solved four to a wave instead of one.  No other header here, so that
// the rule can be held against its figures on a CPU (tests/test_host.py).
//
// One LP per wave has the lowest latency; four to a wave take longer but need a quarter of the waves.  Alone on its SIMD a
// lone LP is the faster one throughout.  Up to 8 ranks its lanes are busy less than half the time, and it still is with three
// on a SIMD; four packed ones fill one wave of every SIMD and take no longer unless a rank has many experts, then a second packed wave
// is behind until there are six LPs per SIMD.  From 9 ranks on (16 pivots a step instead of 8) the second lone LP is already too many.
//
// How long a packed wave takes depends on the counts that one of its lanes reads: those of a whole rank, and a sixteenth
// of those that the wave fetches for its four LPs.  Measured, us a batch, one per wave / four per wave:
//    G, D   of a rank, in all      2048        3072        4096        5120        6144        7168        8192 LPs
//   (8, 2)    8    64     7.1 /  9.6   9.0 /  9.5  10.5 /  9.6  12.1 / 12.4  13.7 / 12.5  15.4 / 12.5  17.0 / 12.6
//   (8, 2)   32   256     7.3 /  9.7   9.0 /  9.9  10.7 / 10.3  12.2 / 13.3  13.8 / 13.8  15.5 / 14.2  17.0 / 14.4
//   (8, 2)    8   512     7.0 /  9.6   9.0 /  9.5  10.7 /  9.6  12.2 / 12.5  13.9 / 12.6  15.6 / 12.7  17.2 / 12.7
//   (8, 2)   32   512     7.4 /  9.8   9.2 / 10.1  10.8 / 10.5  12.3 / 13.6  13.9 / 14.0  15.7 / 14.4  17.4 / 14.8
//   (8, 2)    8  1024     7.3 / 10.0   9.3 / 10.1  11.1 / 10.1  12.5 / 13.0  14.2 / 13.1  18.7 / 13.2  20.4 / 13.4
//   (8, 2)   32  1024     7.6 / 10.2   9.4 / 10.5  11.1 / 10.9  12.7 / 14.2  14.3 / 14.4  19.0 / 15.0  20.7 / 15.4
//   (8, 2)   64   512     7.8 / 11.7   9.3 / 11.9  11.0 / 12.5  12.6 / 15.6  14.4 / 15.9  15.9 / 16.3  17.6 / 16.6
//   (8, 1)   24   192     6.9 /  9.4   8.5 /  9.3  10.0 /  9.6  11.6 / 12.3  13.1 / 12.6  14.9 / 12.9  16.5 / 13.7
//   (8, 1)   32   256     7.1 /  8.6   8.6 /  8.7   9.9 /  8.9  11.4 / 11.8  12.9 / 12.1  14.6 / 12.2  16.2 / 12.4
//   (8, 1)   40   320     7.0 /  9.8   8.7 / 10.0  10.2 / 10.3  11.8 / 12.9  13.4 / 13.3  15.1 / 13.9  16.8 / 14.2
//   (8, 1)   48   384     7.1 / 10.3   8.7 / 10.5  10.5 / 11.5  12.1 / 14.5  13.8 / 15.0  15.5 / 15.4  17.2 / 15.7
//   (7, 2)   32   224     8.1 / 10.6  10.1 / 10.9  11.7 / 11.2  13.3 / 14.4  15.3 / 14.8  17.0 / 15.0  18.4 / 15.4   (padded)
//   (4, 2)   32   128     7.7 / 10.1   9.6 / 10.1  11.3 / 10.2  13.0 / 13.1  14.8 / 13.4  16.5 / 13.7  18.0 / 13.8   (padded)
//   (4, 2)   64   256     8.0 / 11.3   9.9 / 11.3  11.5 / 11.6  13.2 / 14.5  15.2 / 14.8  16.7 / 14.9  18.4 / 14.9   (padded)
//   (16, 1)  16   256    18.7 / 12.6  25.3 / 12.8  32.2 / 13.1  38.9 / 17.9  45.8 / 18.5  52.6 / 18.9  59.5 / 19.4
//   (16, 1)  16  1024    18.7 / 13.4  25.7 / 13.6  32.6 / 13.9  43.8 / 18.8  50.8 / 19.5  57.7 / 20.0  64.7 / 20.5
//   (10, 1)  25   250    19.6 / 15.9  26.6 / 16.2  33.6 / 16.6  40.6 / 21.3  47.8 / 21.7  54.9 / 21.9  61.9 / 22.3   (padded)
// (A number of LPs between two of these takes about as long as the larger one.)  Past 8192 packing stays ahead wherever it is
// ahead there, but for 13 per SIMD at 48 and 64 experts of a rank and 8 ranks (13312: 25.7 / 26.1 and 25.5 / 26.6).
// With one slot a packed wave has half the edges to look after and pays up to 40 experts of a rank where it does up to 32 with more.
// Not in the rule: a rank whose experts are one or two short of a multiple of 16, whose packed wave ends its reads one by one ((8, 1), 31 of a rank,
// 4096 LPs 10.2 / 11.3, 6144 13.4 / 15.6; (8, 2), 30 of a rank, 10.5 / 12.1 and 14.2 / 18.1).
#pragma once

namespace lplb {

// D: slots; n_experts: in all, of which per_rank are a rank's; per_simd: LPs for each SIMD, rounded up.
constexpr bool packing_pays(int G, int D, int per_rank, int n_experts, int per_simd) {
  const int counts_of_a_lane = per_rank + n_experts / 16, few = D == 1 ? 40 : 32;
  return G > 8           ? per_simd > 1
         : per_simd == 4 ? per_rank <= few
         : per_simd == 6 ? per_rank < few || counts_of_a_lane < 48
         : per_simd == 7 ? per_rank <= 32 || counts_of_a_lane <= 84
                         : per_simd > 7 && (per_rank <= 32 || counts_of_a_lane <= 96);
}

} // namespace lplb
