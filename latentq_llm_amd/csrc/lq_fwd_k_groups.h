// How many groups of waves share a tile of the weights-direct forward kernel (KS in lq_gemm_fwd.hip). Host arithmetic.
#pragma once

enum FwdTile { FWD_128x128, FWD_128x256, FWD_GATE_UP };  // 128 x 128 of one product, 128 x 256, 128 x 128 of two

// Two where no compute unit gets a second workgroup and K is long enough to pay for the second group's prologue and the way of
// the sums through LDS (64 or 128 KB of them). us with one group -> two, weights from HBM, by workgroups T on 256 units:
//   K                 512             768             1024            1280            1536            2048            3072            4096
//   128 x 128, T 160   8.4 ->  8.7   10.3 -> 10.4   12.0 -> 11.4   13.6 -> 13.1   15.4 -> 14.2   19.4 -> 17.5   27.2 -> 23.8   35.6 -> 30.3
//              T 256   8.7 ->  9.2   10.7 -> 11.2   12.9 -> 12.6   14.5 -> 14.7   16.8 -> 16.4   22.2 -> 21.0   31.3 -> 29.2   40.8 -> 36.9
//   128 x 256, T 128  12.2 -> 13.0   15.1 -> 15.8   17.5 -> 17.6   20.3 -> 20.7   22.9 -> 22.5   29.1 -> 28.1   40.6 -> 38.7   51.4 -> 48.9
//   gate / up, T 160  11.2 -> 13.4   14.0 -> 16.1   16.4 -> 18.1   19.5 -> 20.8   21.9 -> 22.9   27.4 -> 28.0   41.1 -> 40.2   51.6 -> 49.2
//              T 240  12.3 -> 14.5   15.4 -> 17.9   18.5 -> 20.8   22.3 -> 25.5   26.5 -> 28.7   34.0 -> 35.1   48.3 -> 48.1   62.8 -> 61.4
//              T 256  12.1 -> 14.7   15.8 -> 18.8   18.8 -> 21.2   22.4 -> 25.1   25.6 -> 27.8   33.0 -> 34.8   48.5 -> 49.0   62.6 -> 62.7
// With more than one workgroup to a unit a second group is always slower (T 264: 11.6 -> 15.7 to 50.0 -> 60.0).
constexpr int fwd_k_groups(FwdTile tile, long long workgroups, long long cus, int K) {
    if (workgroups > cus) return 1;
    const bool full = 16 * workgroups > 15 * cus;
    return K >= (tile == FWD_128x128 ? 1024 : tile == FWD_128x256 ? 1536 : full ? 4096 : 3072) ? 2 : 1;
}
