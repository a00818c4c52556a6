// A wave's way through its batches of groups in gemv_kernel (lq_gemv.hip), the next batch's codes requested under the products of
// this one. The steps themselves are the caller's: the kernel's, or those of the host test, which keeps count of the loads.
#pragma once

#ifdef __HIPCC__
#define LQ_BATCHES __device__ __forceinline__
#else
#define LQ_BATCHES inline
#endif

constexpr int kUnroll = 4;  // groups per batch (scale/zero batches are 4 x bf16 = 8 bytes)

// Wave w of `step` takes the batches w, w + step, ... of the row's G groups.
//   load_x(g0), load_codes(g0)  request the token rows / the codes, scales and zeros of the batch that begins with group g0
//   multiply(g0, then)          takes a batch's codes, calls then(), multiplies the rows and has done with them
//   arrived()                   waits for all that has been requested
// The wait stands in front of the next batch's loads: behind them it would have to know their number to leave them in flight, and
// a short last batch has fewer than the others (no scales and zeros), so that token rows would be counted for them.
template <class LoadX, class LoadCodes, class Multiply, class Arrived>
LQ_BATCHES void gemv_batches_ahead(int wave, int step, int G, LoadX &&load_x, LoadCodes &&load_codes, Multiply &&multiply,
                                   Arrived &&arrived) {
    int g0 = wave * kUnroll;
    if (g0 >= G) return;
    load_x(g0);
    load_codes(g0);
    for (bool more = true; more;) {
        multiply(g0, [&]() {
            g0 += step * kUnroll;
            more = g0 < G;
            arrived();
            if (more) load_codes(g0);
        });
        if (more) load_x(g0);
    }
}
