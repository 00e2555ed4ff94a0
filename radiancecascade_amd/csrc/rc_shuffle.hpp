// The row order of a training epoch: the steps of a parallel Fisher-Yates
// shuffle, for the kernels of rc_mlp.hip and for a host build that runs them
// one after another.
//
// The shuffle of 0 .. n-1 swaps position i with j_i = r_i mod (i + 1) for i =
// n-1 .. 1, r the SplitMix64 stream after `state`, in parallel and with the
// sequential loop's result.  At step i position i gets its final value, the one
// position j_i holds, and the value of position i moves to j_i.  So the value
// position p holds at step i was put there by the latest earlier step that drew
// p, which is the smallest i' > i with j_i' = p, or is p itself if there is
// none; and step i' moved the value position i' held then, found the same way.
// With the steps that drew p listed in ascending order (linked with one
// exchange each, then each list sorted: ln(n / p) steps on average), step i's
// predecessor is the next in its own list, and the resolution follows the
// predecessors to a position nothing was moved into, a few hops.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define RC_HOST_DEVICE __host__ __device__
#else
#define RC_HOST_DEVICE
#endif

namespace rc {

constexpr int kShuffleList = 24;  // steps of a list sorted in a buffer; a longer one is sorted in place

RC_HOST_DEVICE inline uint64_t splitmix64_at(uint64_t state, uint64_t k)
{
    uint64_t z = state + (k + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// The position step i (1 .. n-1) draws: the stream's n-1-i th value.
RC_HOST_DEVICE inline int shuffle_target(uint64_t state, int n, int i)
{
    return (int)(splitmix64_at(state, (uint64_t)(n - 1 - i)) % (uint64_t)(i + 1));
}

// List p in ascending order; buf: LIST ints, `stride` apart.
template <int LIST>
RC_HOST_DEVICE inline void shuffle_sort_list(int p, int *head, int *next, int *buf, int stride)
{
    int len = 0, i = head[p];
    for (; i >= 0 && len < LIST; ++len) {
        const int after = next[i];
        int k = len;
        for (; k > 0 && buf[(k - 1) * stride] > i; --k) buf[k * stride] = buf[(k - 1) * stride];
        buf[k * stride] = i;
        i = after;
    }
    if (len < 2 && i < 0) return;
    head[p] = buf[0];
    for (int k = 0; k < len; ++k) next[buf[k * stride]] = k + 1 < len ? buf[(k + 1) * stride] : -1;
    while (i >= 0) {  // the rest, each put in its place in the list
        const int after = next[i];
        int before = -1, at = head[p];
        while (at >= 0 && at < i) {
            before = at;
            at = next[at];
        }
        next[i] = at;
        if (before < 0) head[p] = i;
        else next[before] = i;
        i = after;
    }
}

// Position i's final value: order[i] holds j_i (0 for i = 0), the lists are sorted.
RC_HOST_DEVICE inline void shuffle_resolve(int i, int *order, const int *head, const int *next)
{
    // the step whose swap put the value there (position 0 has no step of its own)
    int step = i == 0 ? head[0] : next[i];
    if (step < 0) return;  // order[i] = j_i already
    for (;;) {
        const int first = head[step];
        const int f = first != step ? first : next[step];  // a step may have drawn its own position
        if (f < 0) break;
        step = f;
    }
    order[i] = step;
}

}  // namespace rc
