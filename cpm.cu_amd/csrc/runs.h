// What the recurrences share: which of a step's sequences a launch takes, by the number of tokens each brings; values that
// are not finite; decays.
#pragma once
#include "common.h"

// The nth sequence (in the step's order, from 0) that brings at least `lo` and fewer than `hi` tokens, -1 if there are not
// so many; with hi = 0 every sequence counts.  All 64 lanes of the calling wavefronts must be live; the result is uniform.
__device__ inline int nth_run(const int* __restrict__ cu_q, int n_seqs, int nth, int lo, int hi) {
    if (hi == 0) return nth;
    const int lane = threadIdx.x & 63;
    for (int s0 = 0; s0 < n_seqs; s0 += 64) {
        const int s = s0 + lane;
        const int q = s < n_seqs ? cu_q[s + 1] - cu_q[s] : -1;
        unsigned long long found = __builtin_amdgcn_ballot_w64(q >= lo && q < hi);
        const int count = __builtin_popcountll(found);
        if (nth < count) {
            for (; nth > 0; --nth) found &= found - 1;
            return __builtin_amdgcn_readfirstlane(s0 + (int)__builtin_ctzll(found));
        }
        nth -= count;
    }
    return -1;
}

// Workgroup i of a sequence's heads -> head: neighbours take heads of different groups, so that a group's heads, which
// read the same rows, meet in one XCD (workgroups are dealt to the 8 XCDs in turn) wherever there are 8 groups or a multiple.
__device__ inline int grouped_head(int i, int heads, int groups) { return i % groups * (heads / groups) + i / groups; }

// Whether any of a wavefront's values, four a lane, is an infinity or no number.
__device__ inline bool wave_odd(float a, float b, float c, float d) {
    return __builtin_amdgcn_ballot_w64(a * 0.f + b * 0.f + c * 0.f + d * 0.f != 0.f) != 0;
}

// Log decays -A d for sums over a chunk.  Below -1000 one is as good as -1000 (the float factor is zero either way, beside
// whatever else it is summed with), and a sum through it then keeps the decays behind it: an infinite d, or A, forgets
// what came before and no more, as a factor of zero does token by token.  (No number stays none.)
__device__ inline float decay_rate(float A_log) {
    const float A = expf(A_log);
    return A > 3e38f ? 3e38f : A;
}
__device__ inline float decay_step(float d, float A) { return d > 1000.0f / A ? 1000.0f / A : d; }
