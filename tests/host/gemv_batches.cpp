// Runs gemv_batches_ahead with steps that keep count of the loads instead of issuing them: loads land in the order of their
// requests, codes are there when they are taken (the compiler sees to that), token rows only if what was waited for covers them.
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <vector>

#include "lq_gemv_batches.h"

struct Load {
    bool rows;
    int g0;
};

static void walk(int wave, int waves, int G, int M, int NT, bool qs) {
    std::deque<Load> flying;
    int rows = -1, codes = -1;  // the batch whose rows / codes were requested last
    bool reading = false;
    std::vector<int> seen, want;
    auto fail = [&](const char *what, int g0) {
        printf("%s: wave %d of %d, %d groups, %d rows, %d tiles, group %d\n", what, wave, waves, G, M, NT, g0);
        exit(1);
    };
    auto load_x = [&](int g0) {
        if (reading) fail("rows overwritten", g0);
        rows = g0;
        for (int m = 0; m < M; ++m) flying.push_back({true, g0});
    };
    auto load_codes = [&](int g0) {
        codes = g0;
        for (int n = NT * kUnroll + (!qs && g0 + kUnroll <= G ? 2 * NT : 0); n > 0; --n) flying.push_back({false, g0});
    };
    auto in_flight = [&](bool of_rows, int g0) {
        for (const Load &l : flying)
            if (l.rows == of_rows && l.g0 == g0) return true;
        return false;
    };
    auto multiply = [&](int g0, auto then) {
        if (codes != g0 || rows != g0) fail("another batch's operands", g0);
        while (in_flight(false, g0)) flying.pop_front();
        reading = true;
        then();
        if (in_flight(true, g0)) fail("rows not there", g0);
        reading = false;
        seen.push_back(g0);
    };
    gemv_batches_ahead(wave, waves, G, load_x, load_codes, multiply, [&]() { flying.clear(); });
    for (int g0 = wave * kUnroll; g0 < G; g0 += waves * kUnroll) want.push_back(g0);
    if (seen != want) fail("not the wave's batches", -1);
    if (!flying.empty()) fail("loads in flight at the end", -1);
}

int main() {
    for (int waves = 2; waves <= 8; ++waves)
        for (int wave = 0; wave < waves; ++wave)
            for (int G = 1; G < 90; ++G)
                for (int M : {1, 5, 8, 9, 12, 16})
                    for (int NT : {1, 2})
                        for (bool qs : {false, true}) walk(wave, waves, G, M, NT, qs);
    printf("ok\n");
}
