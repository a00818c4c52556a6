// tile workgroups units K, one set a line -> groups of waves
#include <cstdio>

#include "lq_fwd_k_groups.h"

int main() {
    int tile, K;
    long long wg, cus;
    while (scanf("%d %lld %lld %d", &tile, &wg, &cus, &K) == 4) printf("%d\n", fwd_k_groups((FwdTile)tile, wg, cus, K));
}
