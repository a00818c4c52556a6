// Walks the stages of the staged forward kernel over slices of a row: what is requested and what is read between two barriers.
// argv: q_log pairs first end; prints a line and exits 1 for a piece of scales that is not there, or is overwritten, when it is read.
#include <cstdio>
#include <cstdlib>

#include "lq_staged_ring.h"

int main(int argc, char **argv) {
    int n = 0, q_log, pairs, first, end;
    while (scanf("%d %d %d %d", &q_log, &pairs, &first, &end) == 4) {
        const StagedSlice slice = {first, end, pairs != 0};
        const ScaleRing ring = {q_log, pairs != 0};
        int holds[8], since[8], next = ring.piece(first);  // per slot: the last piece requested, and during which stage
        for (int s = 0; s < 8; ++s) holds[s] = since[s] = -9;
        const int slots = ScaleRing::bytes(pairs != 0) / (q_log ? 4096 : 1024);
        auto fail = [&](const char *what, int u, int piece) {
            printf("%s: q_log %d pairs %d groups %d..%d stage %d piece %d\n", what, q_log, pairs, first, end - 1, u, piece);
            exit(1);
        };
        // during stage u: the pieces of stage u + 2 are requested (in front of the loop: of stages 0 and 1) ...
        auto request = [&](int u) {
            if (u + 2 >= slice.units()) return;
            for (; next <= ring.piece(slice.last_group(u + 2)); ++next) {
                const unsigned s = ring.slot(next);
                if ((int)s >= slots) fail("no such slot", u, next);
                // ... while waves that are behind read stage u's values, which they begin to after the barrier in front of stage u
                for (int kg = 0; kg < 2; ++kg) {
                    if (u < 0 || u >= slice.units_of(kg)) continue;
                    const int g = slice.group_of(u, kg), read = ring.piece(g < end ? g : end - 1);
                    if (ring.slot(read) == s && read != next) fail("overwritten while it is read", u, read);
                }
                holds[s] = next;
                since[s] = u;
            }
        };
        request(-2);
        request(-1);
        for (int u = 0; u < slice.units(); ++u) {
            for (int kg = 0; kg < 2; ++kg) {
                if (u >= slice.units_of(kg)) continue;
                const int g = slice.group_of(u, kg), piece = ring.piece(g < end ? g : end - 1);
                // the wait at the end of stage u - 1 leaves only what was requested during that stage in flight
                if (holds[ring.slot(piece)] != piece || since[ring.slot(piece)] > u - 2) fail("not there", u, piece);
            }
            request(u);
        }
        ++n;
    }
    printf("%d slices\n", n);
}
