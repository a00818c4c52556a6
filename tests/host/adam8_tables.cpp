// blocks units, one pair a line -> whether the step has tables
#include <cstdio>

#include "lq_adam8_tables.h"

int main() {
    long long blocks, cus;
    while (scanf("%lld %lld", &blocks, &cus) == 2) printf("%d\n", adam8_tables(blocks, cus));
}
