// How many chunks of 64 indices a wave of the redirect takes per pass.  No other header here, so that the rule can be held against its
// figures on a CPU (tests/test_host.py).
//
// Two passes are in flight, so that one pass's ranking and stores overlap the next one's loads.  Four chunks, unless half of the CUs have
// nothing to do: then the passes, not the memory, take the time, and eight are half as many and gain 3 to 13 %.  Where the fours are odd in
// number half of the last such pass is idle, and costs as much as one with tokens in it; that is worth it from eleven fours on, as long as
// three quarters of the CUs have nothing to do, and with more than 64 sets, whose passes have another barrier, from seven.
//
// us a call (weighted_select_target), four / eight chunks, medians of nine runs at other places in memory:
//   sets of experts, slices; chunks of a wave in all: 16, 20, 24, 28, 32, 36, 40, 44, 48, 52, 64
//    16 of  32,  16   12.4 / 12.5  14.7 / 16.0  16.8 / 16.4  18.9 / 19.8  21.0 / 20.2  23.1 / 23.6  25.1 / 23.9  27.2 / 27.2  29.3 / 27.6  31.2 / 31.1  37.6 / 35.0
//    16 of  32,  64   12.8 / 12.9  14.9 / 16.2  17.3 / 16.8  19.0 / 19.9  21.0 / 20.3  23.1 / 23.6  25.5 / 24.7  27.2 / 27.4  29.4 / 27.9  31.4 / 31.5  38.1 / 35.9
//    16 of  32, 128   13.1 / 13.5  14.9 / 16.2  17.4 / 17.4  19.3 / 20.5  21.5 / 21.0  24.6 / 26.0  27.0 / 26.2  29.2 / 31.1  31.6 / 31.9  33.6 / 36.2  39.7 / 38.6
//    16 of 256,  16   10.5 / 10.2  12.3 / 12.9  14.0 / 13.3  15.8 / 16.1  17.5 / 16.3  19.2 / 19.2  20.8 / 19.2  22.6 / 22.2  24.1 / 22.2  25.7 / 25.3  30.8 / 27.8
//    16 of 256,  64   11.0 / 10.7  12.7 / 13.3  14.7 / 13.9  16.1 / 16.4  17.7 / 16.6  19.3 / 19.5  21.3 / 19.8  22.6 / 22.3  24.4 / 22.7  26.1 / 25.7  31.3 / 28.8
//    16 of 256, 128   11.7 / 11.8  12.6 / 13.3  14.8 / 14.3  16.6 / 17.0  18.1 / 17.4  22.3 / 22.4  24.5 / 23.6  26.7 / 27.6  30.2 / 29.8  31.7 / 32.8  36.2 / 35.1
//    32 of 256,  16   10.9 / 10.8  12.8 / 13.4  14.6 / 13.9  16.4 / 16.6  18.1 / 17.0  19.9 / 19.8  21.6 / 19.8  23.5 / 22.7  25.1 / 22.8  27.0 / 25.9  32.1 / 28.5
//    32 of 256,  64   11.5 / 11.1  13.1 / 13.7  14.9 / 14.4  16.7 / 16.8  18.4 / 17.2  20.0 / 19.9  22.1 / 20.4  23.5 / 22.9  25.4 / 23.2  27.2 / 26.4  32.6 / 29.5
//    32 of 256, 128   11.8 / 12.4  13.1 / 13.8  15.3 / 14.8  17.2 / 17.4  18.9 / 18.0  22.7 / 22.6  25.0 / 23.8  27.6 / 27.5  30.0 / 30.0  31.8 / 33.3  36.7 / 35.6
//    64 of 256,  16   12.2 / 12.2  14.3 / 15.4  16.4 / 15.9  18.5 / 18.9  20.5 / 19.4  22.6 / 22.6  24.6 / 23.0  26.5 / 26.1  28.6 / 26.5  30.6 / 29.7  36.7 / 33.7
//    64 of 256,  64   12.6 / 12.6  14.7 / 15.8  17.0 / 16.5  18.7 / 19.3  20.8 / 19.6  22.7 / 22.8  24.9 / 23.4  26.7 / 26.2  28.8 / 27.0  31.0 / 30.2  37.1 / 34.5
//    64 of 256, 128   13.5 / 13.3  14.7 / 15.8  17.1 / 17.0  19.1 / 19.9  21.0 / 20.4  24.4 / 25.3  26.8 / 25.5  29.0 / 30.0  31.3 / 31.3  33.3 / 35.1  39.2 / 37.9
//   128 of 256,  16   15.1 / 14.6  17.9 / 18.0  20.5 / 19.1  23.2 / 22.5  25.9 / 23.7  28.7 / 27.0  31.2 / 28.2  34.0 / 31.5  36.6 / 32.7  39.3 / 36.1  47.3 / 41.7
//   128 of 256,  64   15.5 / 15.0  18.1 / 18.5  20.9 / 19.5  23.5 / 22.8  26.1 / 24.0  28.8 / 27.2  31.7 / 28.6  34.2 / 31.7  36.9 / 33.1  39.8 / 36.4  47.9 / 42.6
//   128 of 256, 128   15.8 / 16.1  18.2 / 18.4  21.2 / 20.1  24.0 / 23.4  26.6 / 24.7  30.8 / 29.7  33.7 / 30.8  36.7 / 35.4  39.6 / 36.2  42.3 / 40.9  50.6 / 45.3
// (With more than half of the CUs at work: [1048576 x 8] in 256 slices, 16 sets, histogram, LP and redirect 41.6 / 42.2.)
#pragma once

namespace lplb {

// per_wave: chunks of a wave in all.
constexpr int redirect_chunks(long long per_wave, int n_sets, int n_slices, int n_cus) {
  const long long fours = (per_wave + 3) / 4;
  const bool many_sets = n_sets > 64, few_slices = 4ll * n_slices <= n_cus;
  if (per_wave >= 16 && 2ll * n_slices <= n_cus) {
    if (fours % 2 == 0 ? fours > 4 || few_slices || many_sets : many_sets ? fours >= 7 : fours >= 11 && few_slices)
      return 8;
  }
  return per_wave >= 8 ? 4 : per_wave >= 3 ? 2 : 1;
}

} // namespace lplb
