// A wave's way through its batches of groups in gemv_kernel (lq_gemv.hip), the next batch's codes requested under the products of
// this one. The steps themselves are the caller's: the kernel's, or those of the host test, which keeps count of the loads.
#pragma once

#ifdef __HIPCC__
#define LQ_BATCHES __device__ __forceinline__
#else
#define LQ_BATCHES inline
#endif

constexpr int kUnroll = 4;  // groups per batch (scale/zero batches are 4 x bf16 = 8 bytes)

// Partial sum s < n_slots has the batches s, s + n_slots, ...; wave w takes the sums w, w + WAVES, ... (up to SPW of them).
//   load_x(g0), load_codes(g0)  request the token rows / the codes, scales and zeros of the batch that begins with group g0
//   multiply(g0, then)          takes a batch's codes, calls then(), multiplies the rows and has done with them
//   arrived()                   waits for all that has been requested
//   keep(i)                     the wave's i-th partial sum is complete (SPW > 1)
// The wait stands in front of the next batch's loads: behind them it would have to know their number to leave them in flight, and
// a short last batch has fewer than the others (no scales and zeros), so that token rows would be counted for them.
template <int WAVES, int SPW, class LoadX, class LoadCodes, class Multiply, class Arrived, class Keep>
LQ_BATCHES void gemv_batches_ahead(int wave, int n_slots, int G, LoadX &&load_x, LoadCodes &&load_codes, Multiply &&multiply,
                                   Arrived &&arrived, Keep &&keep) {
    int i = 0, g0 = wave * kUnroll;
    bool more = g0 < G && (SPW == 1 || wave < n_slots);
    if (more) {
        load_x(g0);
        load_codes(g0);
    }
    while (more) {
        const int i_now = i;
        multiply(g0, [&]() {
            g0 += n_slots * kUnroll;
            if (SPW > 1 && g0 >= G) {  // the wave's next partial sum
                ++i;
                const int s = wave + i * WAVES;
                g0 = i < SPW && s < n_slots ? s * kUnroll : G;
            }
            more = g0 < G;
            arrived();
            if (more) load_codes(g0);
        });
        if (more) load_x(g0);
        if (SPW > 1 && (!more || i != i_now)) keep(i_now);
    }
}
