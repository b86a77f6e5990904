// chunk_map.h - which windows of the suffix stream each chunk (workgroup) takes.
// Plain C++, so that a host program can check the same code.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define CK_HD __host__ __device__ __forceinline__
#else
#define CK_HD inline
#endif

namespace ck {

// floor(x / d) for 0 <= x < 2^52, 1 <= d < 2^31 (here x <= W P with W < 2^31
// windows and P <= 2^20 chunks) from one IEEE double division: with
// n = floor(x / d), a quotient that is not the integer n is at most
// n + 1 - 1 / d, and rounding moves it up by at most (n + 1) 2^-53 < 1 / d
// (as (n + 1) d <= x + d < 2^53), so it truncates to n; an integer quotient is
// exact. A 64-bit integer division would expand to a few hundred scalar
// instructions per use, inline between the hot blocks of the kernels that map
// windows to chunks (the epilogue was 85% such code and missed the
// instruction cache on 6% of its fetches).
CK_HD int64_t div_nonneg(int64_t x, int64_t d) { return (int64_t)((double)x / (double)d); }

// Window ranges of the P chunks of one kv head group (W windows): chunk c covers
// [lo(c), lo(c + 1)). split == 0: P equal chunks, lo(c) = c W / P. split > 0 (P
// even): chunks 2j and 2j + 1 share the j-th of P / 2 equal ranges, the first
// taking split / 256 of it, in [1/2, 1) (the fused cascade kernel's two roles on
// one CU).
// With fewer windows than chunks each takes a chunk of its own, the first ones (split >
// 0: the last ones), in closed form without a division. So no chunk between two that hold
// windows is ever empty, and folding a cut sequence's partials tests nothing (ranges
// spread over all P chunks left empty ones inside a sequence there, and testing them, two
// chunk bounds per chunk of dependent double divisions, cost the cascade epilogue half
// of its 13.3 us at 8 sequences on a 2048-token prefix). The last chunks in the fused
// kernel, whose stage-1 units are on its first workgroups: a window there waits for a
// unit (1 sequence of 64 tokens, 32 / 8 heads, on a 1024-token prefix: 15.7 us on the
// first pairs, 12.1 here; 3 of 32 tokens 16.1 and 12.1).
struct ChunkMap {
    int64_t W;
    int P;
    int split;
    CK_HD int64_t lo(int c) const {
        if (W < P) {
            if (split == 0) return c < W ? c : W;
            return c > P - W ? c - (P - W) : 0;
        }
        if (split == 0) return div_nonneg((int64_t)c * W, P);
        const int h = P >> 1, j = c >> 1;
        const int64_t a = div_nonneg((int64_t)j * W, h);
        if ((c & 1) == 0) return a;
        return a + (((div_nonneg((int64_t)(j + 1) * W, h) - a) * split) >> 8);
    }
    // the chunk that owns window p < W
    CK_HD int owner(int64_t p) const {
        if (W < P) return (int)(split == 0 ? p : p + P - W);
        if (split == 0) return (int)div_nonneg((p + 1) * P - 1, W);
        const int j = (int)div_nonneg((p + 1) * (P >> 1) - 1, W);
        return 2 * j + (p >= lo(2 * j + 1) ? 1 : 0);
    }
};

// Chunks in use of a grid that has room for `most`: `few` once the sequences hold 12
// windows in the mean. The lengths decide, not the bound that the host knows (a table
// as wide as the longest context says nothing of them).
CK_HD int chunks_used(int64_t W, int batch, int most, int few) { return W >= (int64_t)12 * batch ? few : most; }

}  // namespace ck
