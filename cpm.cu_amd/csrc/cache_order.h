// Which token a workgroup of a kernel takes that writes rows of the cache, a token a workgroup.
#pragma once

// Workgroups are dealt to the 8 XCDs in turn, and 8 neighbouring tokens' values lie side by side, 2 bytes each (common.h:
// value_index): token t in workgroup t has every XCD write its 2 bytes of a line, which its L2 then holds and sends to memory
// alone.  Here an XCD takes 32 neighbouring tokens one behind the other (8 in what is left of 256), and lines meet in one L2.
// 2,048 tokens, us, before -> here: 32 heads on 8 of 128 features 30.2 -> 26.7, with norms of q and k 44.2 -> 41.9, 16 on 4 of 256
// 36.7 -> 32.3, latents of 512 10.3 -> 6.9; 300 tokens 7.3 -> 6.5, 9.9 -> 8.7, latents 4.6 -> 4.2; up to 24 the same within 0.1.
__device__ inline int cache_order(int wg, int tokens) {
    const int whole = tokens & ~255, more = tokens & ~63;
    if (wg < whole) return (wg & ~255) + (wg & 7) * 32 + (wg >> 3 & 31);
    if (wg < more) return (wg & ~63) + (wg & 7) * 8 + (wg >> 3 & 7);
    return wg;
}
