// The bounded wait of the steppers' exchanges (oetqf.jl_amd/csrc/exchange.h)
// on the CPU: it returns the words once all of them carry the number, and ends
// by its clock when a word never does (left from the exchange before, never
// written, or from one ahead).
#include <cstdio>
#include <cstdlib>

#define __device__
#define __forceinline__ inline
#include "../../oetqf.jl_amd/csrc/exchange.h"

using namespace oq;

// Word q carries number `to` from poll at[q] on (-1: never), `from` before.
static int run(unsigned from, unsigned to, unsigned want, const long (&at)[4], long long wait, bool expect, long most)
{
    long polls = 0, ticks = 0;
    unsigned long long w[4];
    const bool ok = x_poll(
        w, want, wait,
        [&](int q) {
            if (q == 0 && ++polls > most) {
                printf("still waiting after %ld polls\n", most);
                exit(1);
            }
            return x_word(at[q] >= 0 && polls > at[q] ? to : from, 0x100u + (unsigned)q);
        },
        [&] { return (long long)(ticks += 10); });
    int bad = ok != expect;
    for (int q = 0; q < 4 && ok; ++q) bad += w[q] != x_word(want, 0x100u + (unsigned)q);
    if (!expect) bad += polls < 64 * (wait / 10);  // not before its time
    if (bad) printf("from %u to %u want %u: ok %d after %ld polls\n", from, to, want, (int)ok, polls);
    return bad;
}

int main()
{
    int bad = 0;
    bad += run(0, 1, 1, {0, 0, 0, 0}, 100, true, 1);
    bad += run(6, 7, 7, {3, 0, 200, 1}, 100, true, 201);
    bad += run(0xffffffffu, 0, 0, {5, 5, 6, 5}, 100, true, 7);        // the number wraps
    bad += run(6, 7, 7, {0, 0, -1, 0}, 100, false, 64 * 12);          // one word never comes
    bad += run(6, 6, 7, {0, 0, 0, 0}, 0, false, 64 * 2);              // a whole exchange never comes
    bad += run(0, 9, 7, {-1, 2, 2, 2}, 100, false, 64 * 12);          // out of step
    if (bad) return 1;
    printf("ok\n");
    return 0;
}
