// exchange.h -- values that travel between workgroups with their exchange's
// number: a 64-bit word is number | half of a double.  Plain device code over a
// load and a clock; also compiled for the host by the emulation in tests/emul.
#pragma once

namespace oq {

__device__ __forceinline__ unsigned long long x_word(unsigned ep, unsigned half)
{
    return (unsigned long long)ep << 32 | half;
}

// Polls the Q words load(0) .. load(Q - 1) until every one carries number ep.
// False if that takes longer than `wait` ticks of clock(), which is looked at
// every 64 polls: every wait ends.
template <int Q, class Load, class Clock>
__device__ __forceinline__ bool x_poll(unsigned long long (&w)[Q], unsigned ep, long long wait, Load load, Clock clock)
{
    long long t0 = 0;
    for (unsigned spin = 0;; ++spin) {
        bool ok = true;
#pragma unroll
        for (int q = 0; q < Q; ++q) w[q] = load(q);
#pragma unroll
        for (int q = 0; q < Q; ++q) ok = ok && (unsigned)(w[q] >> 32) == ep;
        if (ok) return true;
        if (spin % 64 == 63) {
            const long long now = clock();
            if (spin == 63) t0 = now;
            if (now - t0 > wait) return false;
        }
    }
}

}  // namespace oq
