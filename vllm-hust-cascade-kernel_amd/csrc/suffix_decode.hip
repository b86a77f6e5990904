// suffix_decode.hip - per-sequence paged decode attention over each sequence's
// own suffix pages (cascade stage 2) on gfx950: the stand-alone op and the
// fused cascade's streaming waves compute their windows on the matrix cores.
//
// Role: replaces the closed CANN op npu_fused_infer_attention_score_v2 the
// reference calls for stage 2 (ascend-kernel/README.md:186-197): one query
// token per sequence, GQA, paged K/V, bf16 O plus a compact fp32 LSE that
// lse_merge folds into the stage-1 result. An empty suffix (kv length 0)
// yields O = 0, LSE = -inf, which the merge treats as weight 0.
//
// Arithmetic: S = q k^T * scale in fp32, online softmax in the log2 domain,
// P as two bf16 terms whose sum is P within 2^-16, or as three that hold fp32 P (the
// fused cascade above 4 heads per group, stage 1's decode form), fp32 accumulation, O = acc / l, LSE = ln(l) + max.
//
// MI355X design: HBM-bound streaming with a persistent, balanced grid and few
// instructions per byte (at 8 TB/s a CU receives about 15 bytes per cycle; a
// vector-ALU body of ~190 instructions per 32-token window was bound by its
// own issue, the matrix-core body takes ~90).
// * Suffix lengths vary widely (geometric in the benchmark), so the work is cut
//   into windows of 8 tokens per streaming wave (32 tokens on 4 waves) of one
//   sequence (the last window of a sequence may be short), and workgroup (kv
//   head group g, chunk c) takes the c-th 1/P of the list of all windows,
//   crossing sequence boundaries: every workgroup streams the same number of
//   windows and starts once.
// * Start-up: lengths -> window prefix sums (block scan in LDS), then a table
//   of the workgroup's windows (page id, valid tokens, sequence, segment
//   start/end) built in parallel in one round trip that also copies the first
//   q rows into LDS. The streaming loop reads the table from LDS; no load in
//   the loop depends on another load.
// * Two paged K/V layouts: NHD [blocks, 128, kv_heads, 128] (the stage-1 pool)
//   and BNSD [blocks, kv_heads, 128, 128] (the layout the reference's stage-2
//   op reads, ascend-kernel/README.md:182-183), so a BNSD pool needs no
//   transposing copy. A page, a token and a kv head are three strides.
// * K and V go straight from HBM into registers by buffer loads, no barrier in
//   the streaming loop. Each window gets a buffer descriptor (its first row as
//   base, its valid rows as range) built with scalar instructions, so a lane's
//   address is a fixed offset; rows past the sequence's end fall outside the
//   range (zeros, no bytes moved), and an invalid page id gets an empty range:
//   its rows read as zeros, the semantics of the pool's unmapped pages.
// * Scores S^T = K q^T and values O^T += V^T P^T on 16x16 bf16 MFMAs, V^T
//   through a per-wave LDS slot read back transposed (suffix_stream_body gives
//   the lane layouts). The running max moves only when a score exceeds it by more
//   than 2^kTau (a wave-uniform branch), so rescaling is rare; any reference point
//   gives the same O and LSE.
// * Closing a sequence never stops the stream: each wave writes its partial
//   (O, m, l) into the segment's slot of an LDS exchange ring and counts itself
//   in with an LDS atomic. Once all partials are in, each wave merges its share
//   into an LDS stash (one wave doing the whole merge fell behind the others by
//   it at every close), written out after the phase's loop. A wave waits only for
//   arrivals (with one exchange slot, also for shares) of a close that every wave
//   reaches without waiting for it, so every wait ends.
// * Cascade (stage 1 + suffix + merge): one fused kernel, one workgroup per CU.
//   Waves 0-3 run the stage-1 body (MFMA, LDS tiles: matrix cores and LDS),
//   waves 4-7 stream suffix windows; each role synchronises only its own four
//   waves through an LDS counter barrier, so the two run side by side instead
//   of one kernel after the other, and a small epilogue kernel merges the two
//   results.
// * The range is processed in phases of at most 512 windows and 8 segments (4 in
//   the fused kernel above 4 heads, where 8 do not fit beside the stage-1 tiles).
//   A phase starts with one round trip that fills the window table and copies
//   the q rows of its segments into LDS; the phase's loop has no barrier.
// * A segment that is a whole sequence writes bf16 O and the LSE directly; a
//   sequence cut by a chunk boundary leaves fp32 partials that a small fix-up
//   kernel folds (it also writes O = 0, LSE = -inf for empty suffixes).
#include <algorithm>
#include <cmath>

#include "ck_common.h"
#include "chunk_map.h"
#include "ck_internal.h"

// Bounded waits of this file's kernels that ran out (a broken invariant, never
// expected): counted here, read and reset by ck_wait_giveups.
static __device__ unsigned int g_wait_giveups;

namespace ck {
namespace {

constexpr int kD = 128;
constexpr int kPage = 128;
constexpr int kMaxGroup = 8;
constexpr int kMaxBatch = 1024;     // sequences per launch (prefix sums in LDS)
constexpr int kQSlots = 8;          // segments per phase (their q rows in LDS)
constexpr int kTable = 512;         // windows per table phase
constexpr float kTau = 8.0f;        // log2 headroom before the running max moves
constexpr uint32_t kOob = 0x80000000u;  // a buffer offset past every window's range
constexpr int kRsrcFlags = 0x00020000;  // buffer descriptor word 3 for gfx9 raw loads

// windows of loads in flight per streaming wave: 2 (24 registers per window and
// lane; 3 and 4 measured slower in the fused kernel), 1 in the stand-alone kernel
// above 4 heads (1 measured faster than 2 and 3).
constexpr int kTokDepth = 2;
// Share of each fused workgroup's suffix windows that its streaming waves take
// (in 1/256); the stage-1 waves take the rest after their stage-1 unit. What decides is
// a unit's tiles against the workgroup's windows, and no fixed share suits all: 208 /
// 224, us, 64 / 40 heads on 8192 tokens 54.6 / 52.1, 47 / 40 on 6037 39.0 / 36.8, 64 / 48
// on 8192 56.5 / 54.7, 100 / 64 on 8000 84.7 / 83.4; short prefixes the other way: 200 / 40
// on 1000 47.7 / 49.3, 256 / 64 on 2048 133.8 / 136.8. Above 4 heads per group 224 gains
// up to 5% and costs up to 3%; up to 4 heads 208 is ahead where it matters most (64 /
// 32 on 8192 46.4 / 48.2; 100 / 32 on 8000 58.5 / 56.8, most others within 1%).
constexpr int fused_split(int64_t group) { return group > 4 ? 224 : 208; }
static_assert(fused_split(8) >= 128 && fused_split(8) < 256 && fused_split(4) >= 128, "ChunkMap assumes a share in [1/2, 1)");

// LDS layout (bytes) of the stream body for G query heads per group and NW waves;
// SEGS segments per phase and RING exchange slots. The merged results of a phase's
// segments are held until its window loop is done; each wave's V transpose slot is
// 8 token rows of 256 bytes at a 288-byte pitch (the pitch puts the 4 rows of a
// transpose read in distinct bank groups).
constexpr int kVtPitch = 288;
template <int G, int NW, int SEGS = kQSlots, int RING = 2>
struct SfxLds {
    static constexpr int kSegs = SEGS;                                   // segments per phase
    static constexpr int kCw = 0;                                        // int cw[kMaxBatch + 1]
    static constexpr int kLen = ((kMaxBatch + 1) * 4 + 15) / 16 * 16;   // int len[kMaxBatch]
    static constexpr int kWtot = kLen + kMaxBatch * 4;                   // int wtot[NW]
    static constexpr int kTab = kWtot + 64;               // int pair tab[kTable + 8] (8 padding entries)
    static constexpr int kQs = kTab + (kTable + 8) * 8;                  // bf16 q[kSegs][G][kD]
    static constexpr int kX = RING;                                      // exchange ring slots
    static constexpr int kXo = kQs + kSegs * G * kD * 2;               // float xo[kX][NW][G][kD]
    static constexpr int kXml = kXo + kX * NW * G * kD * 4;              // float xml[kX][NW][G][2]
    static constexpr int kXsync = kXml + kX * NW * G * 2 * 4;            // int cnt[kX], gen[kX]
    static constexpr int kBar = kXsync + 2 * kX * 4;                     // int bar[2] (group barrier)
    static constexpr int kSo = (kBar + 8 + 15) / 16 * 16;                // float so[kSegs][G][kD]
    static constexpr int kSl = kSo + kSegs * G * kD * 4;                // float sl[kSegs][G]
    static constexpr int kSb = kSl + kSegs * G * 4;                     // int sb[kSegs]
    static constexpr int kVt = (kSb + kSegs * 4 + 15) / 16 * 16;        // char vt[NW][8][kVtPitch]
    static constexpr int kBytes = kVt + NW * 8 * kVtPitch;
    static_assert(kTab % 16 == 0 && kQs % 16 == 0 && kXo % 16 == 0 && kXml % 8 == 0 &&
                      kSo % 16 == 0,
                  "aligned LDS rows");
};

// window table entry: [0] = page id (-1: not a valid page), [1] = packed fields
__device__ __forceinline__ int tab_tv(int y) { return y & 127; }  // valid tokens 1 .. 64
__device__ __forceinline__ bool tab_first(int y) { return (y >> 7) & 1; }
__device__ __forceinline__ bool tab_last(int y) { return (y >> 8) & 1; }
__device__ __forceinline__ int tab_sub(int y) { return (y >> 9) & 3; }  // the window's quarter/half of its page
__device__ __forceinline__ int tab_b(int y) { return y >> 11; }


struct SuffixArgs {
    const uint16_t *q;
    const uint16_t *k;
    const uint16_t *v;
    const int32_t *bt;
    const int64_t *kv_seqlens;
    uint16_t *out;
    float *lse;
    float *part_o;    // [kv head groups][chunks][2][G][kD]
    float *part_lse;  // [kv head groups][chunks][2][G]
    int32_t *cw_out;  // [batch + 1] window prefix sums, written by workgroup 0
    int64_t bt_cols;
    int64_t num_blocks;
    int64_t page_stride;  // elements between pages (both layouts: 128 * kv_heads * 128)
    int64_t tok_stride;   // between tokens of a page: kv_heads * 128 (NHD) or 128 (BNSD)
    int64_t head_off;     // between kv heads:          128 (NHD) or 128 * 128 (BNSD)
    int batch;
    int num_heads;
    int kv_heads;  // kv head groups of the grid: physical kv heads x kv_sub
    int kv_sub;    // query-head groups per physical kv head (group = kv_sub x G)
    int kv_cap;
    int chunks;  // chunks of the window list per kv head group
    // PAIRS: ChunkMap's split; otherwise the chunks in use for long sequences (chunks_used).
    // One field for both: another word in the struct moved the fused kernel's argument
    // loads behind its stage-1 part (64 / 32 heads on 8192 tokens 50.3 -> 51.4 us).
    int split_few;
    float scale_log2;
};

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// x[l] op x[l ^ 16] and x[l] op x[l ^ 32] through v_permlane16_swap /
// v_permlane32_swap: swapping x with itself leaves x[l] in one result and the
// partner lane's x in the other (a VALU exchange, no LDS round trip).
__device__ __forceinline__ float max_xor16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// x in lanes 0-31, y of lane - 32 in lanes 32-63
__device__ __forceinline__ float swap_halves(float x, float y) {
    return __uint_as_float(
        __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false)[0]);
}
__device__ __forceinline__ float sum_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// bf16 terms of a probability (p >= 0): two values truncated to bf16 in one register;
// p - hi, at least min(p, 2^-100) (the median of three is max(p - hi, min(p, c)), as
// p - hi <= p); and r - mid plus 2^-23 r, positive with r and exact in the bits of r
// that truncation to bf16 keeps
__device__ __forceinline__ uint32_t term_hi(float p0, float p1) {
    return __builtin_amdgcn_perm(__float_as_uint(p1), __float_as_uint(p0), 0x07060302u);
}
__device__ __forceinline__ float trunc_bf16(float p) { return __uint_as_float(__float_as_uint(p) & 0xFFFF0000u); }
__device__ __forceinline__ float term_rest(float p) {
    return __builtin_amdgcn_fmed3f(p - trunc_bf16(p), p, 0x1p-100f);
}
__device__ __forceinline__ float term_rest2(float r) { return __builtin_fmaf(r, 1.0f + 0x1p-23f, -trunc_bf16(r)); }
// both bf16 values (>= 0) halved through their exponents; zero stays zero
__device__ __forceinline__ uint32_t halve_bf16x2(uint32_t x) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, x), u16x2{0x80, 0x80}));
}

__device__ __forceinline__ int64_t clamp_len(const SuffixArgs &a, int64_t kvl) {
    const int64_t lim = a.bt_cols * kPage;
    if (kvl > lim) kvl = lim;
    if (kvl > a.kv_cap) kvl = a.kv_cap;
    if (a.num_blocks <= 0) kvl = 0;
    return kvl < 0 ? 0 : kvl;
}

// The result row of stage-1's decode form: fp32 O and 8 copies of the LSE (a.out
// and a.lse then hold fp32 rows and padded LSEs).
__device__ __forceinline__ void write_f32_row(const SuffixArgs &a, int64_t row, int d4, f32x4 o, float lse_v) {
    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(a.out) + row * kD + 4 * d4) = o;
    if (d4 < 2) *reinterpret_cast<f32x4 *>(a.lse + row * 8 + 4 * d4) = f32x4{lse_v, lse_v, lse_v, lse_v};
}

// The stream body on NW waves (thread tid of the group's NW * 64) as workgroup lb
// of a grid of a.kv_heads * a.chunks, with the group's LDS at smem and its own
// barrier. Windows hold 8 NW tokens.
//
// A wave owns 8 tokens of every window, and lane (g, n) = (lane / 16, lane % 16):
// * S^T = K q^T on v_mfma_f32_16x16x32_bf16: A = K, row n = token n of the wave's
//   8 (rows 8-15 read nothing: zeros), dims 32 s + 8 g .. + 7 at step s, straight
//   from global memory; B = q of head n, the same dims. The result puts token
//   4 g + r, head n in register r of lane (g, n); lanes of rows 8-15 (g >= 2) and
//   of heads n >= G get score -inf through the scale's addend, hence p = 0.
// * O^T += V^T P^T on v_mfma_f32_16x16x16_bf16, 16-dim tiles of O: B = P^T is the
//   score layout itself (lane (g, n): tokens 4 g .. 4 g + 3 of head n), and A = V^T
//   comes from the V rows through the wave's LDS slot by ds_read_b64_tr_b16 (lane
//   (g, n): dim n of the tile, tokens 4 (g % 2) .. + 3). The operand's rows 8-15 are
//   the same 8 tokens again and carry another term of P. P enters as bf16 terms: hi
//   = p truncated and lo = p - hi rounded (|p - hi| < 2^-7 p, so p = hi + lo within
//   2^-16 p), one MFMA per tile; with EXACTP three truncated terms, which hold all
//   24 bits of p, two MFMAs per tile.
// * Every term is positive where p is (p - hi is taken as at least min(p, 2^-100), far
//   below the row sum, which is at least 1), so an infinite V element stays infinite:
//   a zero term, or a zero row beside it in the operand, would make NaN of it.
// * The softmax state of head n sits in lane (g, n), the same for every g: the
//   running max is reduced over the 4 groups when it moves, the row sum when the
//   segment closes, and O^T needs no reduction (the MFMA summed the tokens).
// * The merged result of a segment waits in an LDS stash, and the waves write a
//   phase's results out together after its window loop: a store in the loop
//   would count in the same vmcnt as the window loads, so every later wait of
//   the merging wave would also wait for its acknowledgement (or for loads
//   issued after it), a stall of about a round trip per merge.
//
// Two bodies on one CU may share one scan: the body given scan_src (the other
// body's LDS) skips its own, waits until scan_flag is set and reads the other's
// lengths and window prefix sums; the body given only scan_flag sets it once its
// scan is complete. PAIRS: chunk pairs (the fused kernel), every chunk of the grid.
template <int G, int NW, int D, bool F32, bool EXACTP, bool PAIRS, class L = SfxLds<G, NW>, class Bar>
__device__ __forceinline__ void suffix_stream_body(const SuffixArgs &a, CK_LDS char *smem, int lb, int tid,
                                                   const Bar &bar, CK_LDS int *scan_flag = nullptr,
                                                   const CK_LDS char *scan_src = nullptr) {
    static_assert(NW == 4, "the lane layouts below");
    static_assert(D + 1 <= 8, "table padding: D + 1 entries past a phase");
    constexpr int NB = D + 1;  // register ring slots: D windows in flight + the one in use
    constexpr int kThr = NW * 64;
    constexpr int kWin = 8 * NW;         // tokens per window
    constexpr int kWpp = kPage / kWin;   // windows per page
    CK_LDS int *cw = (CK_LDS int *)((scan_src ? scan_src : smem) + L::kCw);
    CK_LDS int *len = (CK_LDS int *)((scan_src ? scan_src : smem) + L::kLen);
    CK_LDS int *wtot = (CK_LDS int *)(smem + L::kWtot);
    CK_LDS i32x2 *tab = (CK_LDS i32x2 *)(smem + L::kTab);
    CK_LDS char *qs = smem + L::kQs;
    constexpr int R = L::kX;
    CK_LDS float *xo = (CK_LDS float *)(smem + L::kXo);
    CK_LDS float *xml = (CK_LDS float *)(smem + L::kXml);
    CK_LDS int *xcnt = (CK_LDS int *)(smem + L::kXsync);  // waves counted into each slot
    CK_LDS int *xgen = xcnt + R;                             // merges completed in each slot
    CK_LDS float *so = (CK_LDS float *)(smem + L::kSo);      // merged O of the phase's segments
    CK_LDS float *sl = (CK_LDS float *)(smem + L::kSl);      // their LSE
    CK_LDS int *sb = (CK_LDS int *)(smem + L::kSb);          // their sequence

    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int t = lane >> 3;  // V rows: token 8 wid + t of each window
    const int c = lane & 7;   // V rows: bytes 16 c and 128 + 16 c
    const int g = lb % a.kv_heads;  // kv head group: query heads g * G .. + G
    const int chunk = lb / a.kv_heads;
    const int gk = g / a.kv_sub;            // the physical kv head they read

    if (tid < R) {
        xcnt[tid] = 0;
        xgen[tid] = 0;
    }

    // ---- lengths and window prefix sums (kPer sequences per thread, block scan) ----
    if (scan_src == nullptr) {
        constexpr int kPer = kMaxBatch / kThr;
        // every load goes out before any is used (one round trip, not kPer): the
        // index is clamped into the batch, and entries past it are dropped below
        int64_t raw[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) raw[j] = a.kv_seqlens[min(kPer * tid + j, a.batch - 1)];
        int lv[kPer];
        int local = 0;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int i = kPer * tid + j;
            const int ln = i < a.batch ? (int)clamp_len(a, raw[j]) : 0;
            if (i < a.batch) len[i] = ln;
            lv[j] = (ln + kWin - 1) / kWin;
            local += lv[j];
        }
        int x = local;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        if (lane == 63) wtot[wid] = x;
        bar.sync();
        int wave_off = 0;
        for (int ww = 0; ww < wid; ++ww) wave_off += wtot[ww];
        int run = wave_off + x - local;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int i = kPer * tid + j;
            run += lv[j];
            if (i < a.batch) cw[i + 1] = run;
        }
        if (tid == 0) cw[0] = 0;
        bar.sync();
        if (lb == 0)
            for (int i = tid; i <= a.batch; i += kThr) a.cw_out[i] = cw[i];
        if (scan_flag != nullptr && tid == 0) *(volatile CK_LDS int *)scan_flag = 1;  // after the barrier above
    } else {
        // the other body's scan (bounded: it always completes, long before this
        // bound; a wait that runs out is counted)
        int spin = 0;
        for (; *(volatile CK_LDS int *)scan_flag == 0 && spin < (1 << 22); ++spin) __builtin_amdgcn_s_sleep(1);
        if (spin == (1 << 22)) count_giveup(&g_wait_giveups);
    }

    const int W = __builtin_amdgcn_readfirstlane(cw[a.batch]);  // scalar: ChunkMap branches on it
    const int P = PAIRS ? a.chunks : chunks_used(W, a.batch, a.chunks, a.split_few);
    if (!PAIRS && chunk >= P) return;  // uniform over the workgroup
    const ChunkMap cm{W, P, PAIRS ? a.split_few : 0};
    const int w0 = (int)cm.lo(chunk);
    const int w1 = (int)cm.lo(chunk + 1);
    if (w0 >= w1) return;  // uniform over the workgroup

    // ---- q rows: the s-th segment of a phase in slot s ------------------------------
    // The q rows of one sequence are G * 256 contiguous bytes: one or two wave DMAs.
    auto dma_q = [&](int bq, int slot) {
#pragma unroll
        for (int u0 = 0; u0 < G * 16; u0 += 64) {
            if (u0 + lane < G * 16)
                dma16(a.q + ((int64_t)bq * a.num_heads + g * G) * kD + (u0 + lane) * 8,
                      qs + slot * G * (kD * 2) + u0 * 16);
        }
    };
    // Largest b in [0, batch] with cw[b] <= x: two ballots over the wave's lanes
    // (a stride-S sample of cw, then the S entries after the last sample <= x)
    // instead of a binary search of ~10 dependent LDS reads.
    auto find_seq = [&](int x) {
        const int S = (a.batch + 64) / 64;  // 64 S > batch
        const uint64_t m1 = __builtin_amdgcn_ballot_w64(cw[min(lane * S, a.batch)] <= x);
        const int base = (__builtin_popcountll(m1) - 1) * S;  // cw is nondecreasing, cw[0] = 0 <= x
        const uint64_t m2 = __builtin_amdgcn_ballot_w64(lane < S && cw[min(base + lane, a.batch)] <= x);
        return base + __builtin_popcountll(m2) - 1;
    };

    // ---- per-lane constants ------------------------------------------------------------
    const int64_t tokb = a.tok_stride * 2;                      // bytes between token rows
    const uint32_t koff = (uint32_t)((8 * wid + t) * tokb + c * 16);   // V byte offset in a window
    const uint32_t win_bytes = (uint32_t)(kWin * tokb);          // a window's buffer range
    const char *kbase = reinterpret_cast<const char *>(a.k) + (int64_t)gk * a.head_off * 2;
    const char *vbase = reinterpret_cast<const char *>(a.v) + (int64_t)gk * a.head_off * 2;
    const int64_t pgb = a.page_stride * 2;
    const uint32_t pg32 = (uint32_t)pgb, win32 = win_bytes, tok32 = (uint32_t)tokb;
    // lane (mg, mn): its K rows (token 8 wid + mn, 16 bytes at
    // 64 s + 16 mg for step s; rows 8-15 read nothing), its V bytes (lane (t, c):
    // token t, bytes 16 c and 128 + 16 c, at koff) in the wave's LDS slot, read
    // back transposed (tile T at + 32 T), and the addend of its scores (-inf: a
    // padding row or head)
    const int mn = lane & 15, mg = lane >> 4;
    const uint32_t kfoff = mn < 8 ? (uint32_t)((8 * wid + mn) * tokb + 16 * mg) : kOob;
    CK_LDS char *vt = smem + L::kVt + wid * 8 * kVtPitch;
    const int vwo = t * kVtPitch + 16 * c;
    const int vro = (4 * (mg & 1) + (mn >> 2)) * kVtPitch + 8 * (mn & 3);
    const float sbias = (mg < 2 && mn < G) ? 0.f : -INFINITY;

    // the O^T tiles (dims 16 T + 4 mg + r of head mn), head mn's
    // softmax state (m; m + kTau, the rescale trigger; the exponent offset, m or
    // 0 while m = -inf; this lane's share of the row sum), q fragments, and the
    // P^T operands of the pending window (one per MFMA of a tile)
    f32x4 oacc[8];
    float m1, mt1, mz1, l1;
    u32x4 qf[4];
    constexpr int kPv = EXACTP ? 2 : 1;
    uint32_t pb[kPv][2];
    int nclose = 0;  // segments closed so far (exchange ring position)
    int qslot = 0;   // segment of the current phase
    u32x4 kbuf[NB][4];
    using VSlot = u32x4[2];
    VSlot vbuf[NB];
    int eyr[NB];               // packed table fields of the window in each ring slot
    // A window's loads: the buffer descriptor of its rows (K or V) starts at the
    // window and spans its valid tokens, so the range check returns 0 for the rows
    // of tokens past the sequence's end (or of an invalid page: range 0) and the
    // lane offsets are constants. The offset from 32-bit factors: a page is at most
    // 2^31 bytes (128 tokens x 2^16 heads x 256 B), a window's offset in its page
    // below that. A step spends few instructions on addresses: the stream wave's
    // instruction count per window is its critical path.
    struct TokWin {
        int64_t off;
        int range;
    };
    auto tok_win = [&](i32x2 e) __attribute__((always_inline)) {
        const int page = __builtin_amdgcn_readfirstlane(e[0]);
        const int ey = __builtin_amdgcn_readfirstlane(e[1]);
        const uint64_t off = (uint64_t)(uint32_t)max(page, 0) * pg32 + (uint32_t)tab_sub(ey) * win32;
        return TokWin{(int64_t)off, page < 0 ? 0 : (int)(tab_tv(ey) * tok32)};
    };

    // a window's K rows as the 4 A fragments of its score MFMAs
    auto issue_kfrag = [&](const TokWin &w, u32x4 *kf) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(kbase + w.off), (short)0, w.range, kRsrcFlags);
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
            kf[s4] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(kfoff + 64 * s4), 0, 0));
    };

    // a window's V rows (lane (t, c): token t, bytes 16 c and 128 + 16 c),
    // issued after the values of the window whose ring slot they reuse
    auto issue_v = [&](const TokWin &w, u32x4 &x0, u32x4 &x1) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t r =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(vbase + w.off), (short)0, w.range, kRsrcFlags);
        x0 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)koff, 0, 0));
        x1 = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(koff + 128), 0, 0));
    };

    // The merged result of sequence b's segment for query head h, dims 4 d4 .. 4 d4
    // + 3 (O normalised): bf16 O and the LSE when the segment is the whole
    // sequence, else an fp32 partial in the chunk's head or tail slot.
    auto write_result = [&](int b, int h, int d4, f32x4 on, float lse_v) __attribute__((always_inline)) {
        const bool head_part = cw[b] < w0;
        const bool tail_part = cw[b + 1] > w1;
        if (!head_part && !tail_part) {
            const int64_t row = (int64_t)b * a.num_heads + g * G + h;
            if constexpr (F32) {
                write_f32_row(a, row, d4, on, lse_v);
            } else {
                *reinterpret_cast<uint2 *>(a.out + row * kD + 4 * d4) =
                    make_uint2(pack_bf16x2(on[0], on[1]), pack_bf16x2(on[2], on[3]));
                if (d4 == 0) a.lse[row] = lse_v;
            }
        } else {
            const int64_t pidx = (((int64_t)g * (PAIRS ? a.chunks : P) + chunk) * 2 + (head_part ? 0 : 1)) * G + h;
            // non-temporal: read once, by the fix-up or cascade epilogue kernel
            __builtin_nontemporal_store(on, reinterpret_cast<f32x4 *>(a.part_o + pidx * kD + 4 * d4));
            if (d4 == 0) a.part_lse[pidx] = lse_v;
        }
    };

    // Merges query-head / dim pair u (h = u / 32, dims 4 (u % 32) .. + 3) of the NW
    // partials in exchange slot r into stash entry e.
    auto merge_pair = [&](int u, int r, int e) __attribute__((always_inline)) {
        const CK_LDS float *xo_r = xo + r * NW * G * kD;
        const CK_LDS float *xml_r = xml + r * NW * G * 2;
        const int h = u >> 5, d4 = u & 31;
        float mx = -INFINITY;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) mx = fmaxf(mx, xml_r[(ww * G + h) * 2]);
        const float mz = mx == -INFINITY ? 0.f : mx;
        float lt = 0.f;
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) {
            const float f = exp2_fast(xml_r[(ww * G + h) * 2] - mz);
            lt = fmaf(xml_r[(ww * G + h) * 2 + 1], f, lt);
            const f32x4 xa = *reinterpret_cast<const CK_LDS f32x4 *>(xo_r + (ww * G + h) * kD + 4 * d4);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = fmaf(xa[i], f, o[i]);
        }
        const float inv = lt > 0.f ? 1.0f / lt : 0.f;
        const float lse_v = lt > 0.f ? (mx + __log2f(lt)) * kLn2 : -INFINITY;
        const f32x4 on = f32x4{o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
        *reinterpret_cast<CK_LDS f32x4 *>(so + (e * G + h) * kD + 4 * d4) = on;
        if (d4 == 0) sl[e * G + h] = lse_v;
    };

    // This wave's share of the merge of close k (exchange slot k % R, sequence
    // b, stash entry e) once all NW partials are in (bounded wait: every wave
    // closes the same segments), so no single wave carries the whole merge. The
    // slot's arrival count only grows, NW per use, so use k / R is complete at
    // NW (k / R + 1) and nothing is reset or published: a wave at close k has
    // passed close k - 1's wait, for which every wave arrived after its reads of
    // close k - 2, the slot's previous use. Each step of a close costs an LDS round
    // trip, slow while the stage-1 waves keep the LDS busy, so the close has few.
    auto merge_share = [&](int k, int b, int e) __attribute__((always_inline)) {
        static_assert(R <= 2, "the slot reuse argument above");
        const int r = k % R;
        const int target = NW * (k / R + 1);
        {
            int spin = 0;
            for (; *(volatile CK_LDS int *)(xcnt + r) < target && spin < (1 << 22); ++spin)
                __builtin_amdgcn_s_sleep(1);
            if (spin == (1 << 22)) count_giveup(&g_wait_giveups);
        }
        asm volatile("" ::: "memory");
        constexpr int kPer = 32 * G / NW;  // pairs per wave
        static_assert(kPer * NW == 32 * G && kPer <= 64, "pairs split evenly over the waves");
        if (lane < kPer) merge_pair(wid * kPer + lane, r, e);
        if (wid == 0 && lane == 0) sb[e] = b;
        if constexpr (R == 1) {  // this wave's reads of the slot are done (LDS operations run in order)
            asm volatile("" ::: "memory");
            if (lane == 0) __hip_atomic_fetch_add(xgen, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };

    // The state of a new segment, set at the start and by every close
    // (a segment opens at the chunk's first window or right after the previous
    // segment's close).
    auto reset_seg = [&]() __attribute__((always_inline)) {
        m1 = -INFINITY;
        mt1 = -INFINITY;
        mz1 = 0.f;
        l1 = 0.f;
#pragma unroll
        for (int T = 0; T < 8; ++T) oacc[T] = f32x4{0.f, 0.f, 0.f, 0.f};
    };

    // Closes segment b (sequence b's windows in this range): hands the wave's (O, m, l)
    // to the exchange ring and merges its share of the NW partials into the phase's stash.
    auto close_seg = [&](int b) __attribute__((always_inline)) {
        // head mn's row sum over the 4 groups; O^T needs no reduction (the MFMAs
        // summed over the tokens)
        const float lt1 = sum_xor32(sum_xor16(l1));
        const int r = nclose % R;
        if constexpr (R == 1) {
            // one slot: every wave's share of the previous close's merge is done
            // (each has arrived there, so each finishes it; bounded)
            int spin = 0;
            for (; *(volatile CK_LDS int *)xgen < NW * nclose && spin < (1 << 22); ++spin) __builtin_amdgcn_s_sleep(1);
            if (spin == (1 << 22)) count_giveup(&g_wait_giveups);
            asm volatile("" ::: "memory");
        }
        CK_LDS float *xo_r = xo + r * NW * G * kD;
        CK_LDS float *xml_r = xml + r * NW * G * 2;
        if (mn < G) {
#pragma unroll
            for (int T = 0; T < 8; ++T)
                *reinterpret_cast<CK_LDS f32x4 *>(xo_r + (wid * G + mn) * kD + 16 * T + 4 * mg) = oacc[T];
            if (mg == 0) {
                xml_r[(wid * G + mn) * 2] = m1;
                xml_r[(wid * G + mn) * 2 + 1] = lt1;
            }
        }
        // a wave's LDS operations are performed in the order it issues them: its rows
        // are in before its arrival counts
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(xcnt + r, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        merge_share(nclose, b, qslot);
        ++nclose;
        ++qslot;
        reset_seg();
    };

    i32x2 enext = i32x2{-1, 0};  // the table entry of the next window to issue
    int eypend = 0;  // packed table fields of window n - 1
    // Values of the pending window: its V rows (lane (t, c) holds 32
    // bytes of token t) into the wave's LDS slot, back as the V^T fragments of the 8
    // dim tiles, then O^T += V^T P^T over the terms of P. The slot is written and read
    // by this wave only, whose LDS operations run in issue order.
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    auto pv_tok = [&](const VSlot &vv) __attribute__((always_inline)) {
        *reinterpret_cast<CK_LDS u32x4 *>(vt + vwo) = vv[0];
        *reinterpret_cast<CK_LDS u32x4 *>(vt + vwo + 128) = vv[1];
        uint2 vtf[8];
#pragma unroll
        for (int T = 0; T < 8; ++T) vtf[T] = lds_read_tr16(vt + vro + 32 * T);
#pragma unroll
        for (int T = 0; T < 8; ++T)
#pragma unroll
            for (int i = 0; i < kPv; ++i)
                oacc[T] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                    __builtin_bit_cast(s16x4, vtf[T]), __builtin_bit_cast(s16x4, uint2{pb[i][0], pb[i][1]}), oacc[T], 0,
                    0, 0);
    };
    // Window step, pipelined by one window: step n issues the K rows of
    // window n + D, computes the scores of window n and the values of window n - 1
    // (its P kept from the step before, its V rows still in their ring slot) -- two
    // independent chains in one basic block, so each fills the other's latencies --
    // then issues window n + D's V rows into the slot window n - 1's values just
    // left, closes window n - 1's segment if it ends there and finishes window n's
    // softmax. The table entry of the window to issue was read one step ahead and
    // the packed fields of each window travel in the ring with its data.
    auto step_tok = [&](auto jc, int n, int np) __attribute__((always_inline)) {
        constexpr int J = decltype(jc)::value;
        constexpr int JI = (J + D) % NB;  // window n + D, into the slot of window n - 1
        const i32x2 ei = enext;
        const TokWin wi = tok_win(ei);
        issue_kfrag(wi, kbuf[JI]);
        const int ey = eyr[J];
        const int eyp = eypend;
        eyr[JI] = __builtin_amdgcn_readfirstlane(ei[1]);
        if (tab_first(ey)) {
            // window n opens a segment: q of head mn (heads past G: any finite row,
            // their scores are -inf), in the slot after the segment window n - 1
            // may still close
            const CK_LDS char *qrow =
                qs + ((qslot + (tab_last(eyp) ? 1 : 0)) * G + (mn < G ? mn : 0)) * (kD * 2) + 16 * mg;
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) qf[s4] = *reinterpret_cast<const CK_LDS u32x4 *>(qrow + 64 * s4);
        }
        enext = tab[n + D + 1];  // at most np + D: a padding entry past the phase
        f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
            sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kbuf[J][s4]),
                                                         __builtin_bit_cast(bf16x8, qf[s4]), sc, 0, 0, 0);
        pv_tok(vbuf[JI]);
        issue_v(wi, vbuf[JI][0], vbuf[JI][1]);
        if (tab_last(eyp)) close_seg(tab_b(eyp));
        eypend = ey;
        float s[4];  // scores of tokens 4 mg + r, head mn; then p
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = fmaf(sc[r], a.scale_log2, sbias);
        {
            const int t1 = min(max(tab_tv(ey) - 8 * wid, 0), 8);
            if (t1 < 8) {
                asm volatile("");  // a branch (a sequence's last window)
#pragma unroll
                for (int r = 0; r < 4; ++r) s[r] = 4 * mg + r < t1 ? s[r] : -INFINITY;
            }
        }
        bool trig = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) trig |= s[r] > mt1;  // m = -inf: any real score
        if (__builtin_amdgcn_ballot_w64(trig)) {
            // head mn's max over its 8 tokens (the 4 groups), the same in its 4 lanes
            const float x = max_xor32(max_xor16(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
            if (x > m1) {
                const float f = exp2_fast(m1 - x);  // 0 from -inf
#pragma unroll
                for (int T = 0; T < 8; ++T) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) oacc[T][r] *= f;
                }
                l1 *= f;
                m1 = x;
                mt1 = x + kTau;
                mz1 = x;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = exp2_fast(s[r] - mz1);  // 0 for masked tokens and padding lanes
            l1 += s[r];
        }
        // P^T of window n for the next step: hi = p truncated to bf16 (exact in fp32), the
        // rest rounded to bf16; EXACTP truncates the rest too and takes what remains as
        // the third term. Only lanes 0-31 hold probabilities: lanes 32-63 take tokens
        // 2, 3 of lane - 32 for the arithmetic, and one swap of two terms then puts
        // the first in lanes 0-31 (rows 0-7) and the second in lanes 32-63 (rows 8-15)
        // of both operand registers. The third fills both, half of it in each.
        {
            const float p0 = swap_halves(s[0], s[2]), p1 = swap_halves(s[1], s[3]);
            const float r0 = term_rest(p0), r1 = term_rest(p1);
            const uint32_t hi = term_hi(p0, p1);
            const uint32_t mid = EXACTP ? term_hi(r0, r1) : pack_bf16x2(r0, r1);
            const auto b0 = __builtin_amdgcn_permlane32_swap(hi, mid, false, false);
            pb[0][0] = b0[0];
            pb[0][1] = b0[1];
            if constexpr (EXACTP) {
                const uint32_t lo = halve_bf16x2(term_hi(term_rest2(r0), term_rest2(r1)));
                const auto b1 = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
                pb[1][0] = b1[0];
                pb[1][1] = b1[1];
            }
        }
    };
    // after a phase's last window (np - 1, in slot (np - 1) % NB): its values and
    // its segment's close
    auto drain_tok = [&](int np) __attribute__((always_inline)) {
        const int js = (np - 1) % NB;  // wave-uniform
        static_for<NB>([&](auto jc) __attribute__((always_inline)) {
            if (js == decltype(jc)::value) pv_tok(vbuf[decltype(jc)::value]);
        });
        if (tab_last(eypend)) close_seg(tab_b(eypend));
    };

    // ---- phases of up to kTable windows and kQSlots segments: table and q rows,
    //      prologue loads, streaming loop --------------------------------------------
    const int nwin = w1 - w0;
    reset_seg();  // the chunk's first window opens a segment
    for (int p0 = 0; p0 < nwin;) {
        if (p0 > 0) {
            wait_vmcnt<0>();
            bar.sync();  // every wave is done with the previous phase's table and q rows
        }
        // The phase's segments: the first kQSlots non-empty sequences from the one
        // holding window w0 + p0 that start inside the chunk, read from one ballot
        // over 64 candidate sequences (every wave finds the same list on its own).
        const int bq0 = find_seq(w0 + p0);  // non-empty: cw[bq0 + 1] > w0 + p0
        const int bc = min(bq0 + lane, a.batch - 1);
        const int c_lo = cw[bc], c_hi = cw[bc + 1], c_len = len[bc];
        uint64_t segm = __builtin_amdgcn_ballot_w64(bq0 + lane < a.batch && c_hi > c_lo && c_lo < w1);
        int segb[L::kSegs], seg_lo[L::kSegs], seg_hi[L::kSegs], seg_len[L::kSegs];
#pragma unroll
        for (int sg = 0; sg < L::kSegs; ++sg) {
            seg_lo[sg] = 0x7FFFFFFF;  // never selected below
            segb[sg] = seg_hi[sg] = seg_len[sg] = 0;
            if (segm != 0) {
                const int l = __builtin_ctzll(segm);
                segm &= segm - 1;
                segb[sg] = bq0 + l;
                seg_lo[sg] = __builtin_amdgcn_readlane(c_lo, l);
                seg_hi[sg] = __builtin_amdgcn_readlane(c_hi, l);
                seg_len[sg] = __builtin_amdgcn_readlane(c_len, l);
                if (sg % NW == wid) dma_q(segb[sg], sg);
            }
        }
        int p1 = min(p0 + kTable, nwin);
        if (segm != 0) {
            p1 = min(p1, __builtin_amdgcn_readlane(c_lo, __builtin_ctzll(segm)) - w0);  // the next segment opens the next phase
        } else if (bq0 + 64 < a.batch) {
            p1 = min(p1, cw[bq0 + 64] - w0);  // candidates beyond the 64 examined: the next phase
        }
        const int np = p1 - p0;
        // D + 1 padding entries past the phase (no loads, no tokens) for the
        // one-step-ahead table reads of its last windows
        for (int i = tid; i < np + D + 1; i += kThr) {
            if (i >= np) {
                tab[i] = i32x2{-1, 0};
                continue;
            }
            const int wg = w0 + p0 + i;
            int b = segb[0], lo_b = seg_lo[0], hi_b = seg_hi[0], len_b = seg_len[0];
#pragma unroll
            for (int sg = 1; sg < L::kSegs; ++sg) {
                if (seg_lo[sg] <= wg) {  // the last segment starting at or before window wg
                    b = segb[sg];
                    lo_b = seg_lo[sg];
                    hi_b = seg_hi[sg];
                    len_b = seg_len[sg];
                }
            }
            const int k = wg - lo_b;
            const int tv = min(len_b - k * kWin, kWin);
            const int first = wg == max(lo_b, w0);
            const int last = wg == min(hi_b, w1) - 1;
            const int page = a.bt[(int64_t)b * a.bt_cols + k / kWpp];
            const bool ok = page >= 0 && (int64_t)page < a.num_blocks;
            const int ey = tv | (first << 7) | (last << 8) | ((k % kWpp) << 9) | (b << 11);
            tab[i] = i32x2{ok ? page : -1, ey};
        }
        wait_vmcnt<0>();  // q rows and page ids in
        bar.sync();
        qslot = 0;
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const i32x2 e = tab[j];  // j < D: a padding entry when j >= np
            const TokWin w = tok_win(e);
            issue_kfrag(w, kbuf[j]);
            issue_v(w, vbuf[j][0], vbuf[j][1]);
            eyr[j] = __builtin_amdgcn_readfirstlane(e[1]);
        }
        enext = tab[D];
        // "window -1" of the pipelined step (slot NB - 1): no values, no close;
        // its V slot is zeroed so that p = 0 times it stays 0
#pragma unroll
        for (int i = 0; i < kPv; ++i) pb[i][0] = pb[i][1] = 0u;
        vbuf[NB - 1][0] = u32x4{0u, 0u, 0u, 0u};
        vbuf[NB - 1][1] = u32x4{0u, 0u, 0u, 0u};
        eypend = 0;
        // full rounds of NB steps, then the rest: the ring slot of every step is a
        // compile-time constant and no step leaves the loop early, so the
        // compiler's vmcnt bookkeeping sees one path around the back edge
        int n = 0;
        for (int it = np / NB; it > 0; --it) {
            static_for<NB>([&](auto jc) __attribute__((always_inline)) {
                step_tok(jc, n + decltype(jc)::value, np);
            });
            n += NB;
        }
        const int rem = np - n;
        static_for<NB>([&](auto jc) __attribute__((always_inline)) {
            if (decltype(jc)::value < rem) {
                step_tok(jc, n + decltype(jc)::value, np);
            }
        });
        drain_tok(np);
        // the phase's merged results out, by every wave of the role: each merge
        // is done once every wave is past its last close
        bar.sync();
        const int nseg = qslot;  // segments closed in this phase (the same in every wave)
        for (int i = tid; i < nseg * G * 32; i += kThr) {
            const int e = i / (G * 32), u = i % (G * 32);
            const int h = u >> 5, d4 = u & 31;
            write_result(sb[e], h, d4, *reinterpret_cast<const CK_LDS f32x4 *>(so + (e * G + h) * kD + 4 * d4),
                         sl[e * G + h]);
        }
        p0 = p1;
    }
}

// The stand-alone stream kernel: the stream body (the
// fused kernel's streaming body) on 4 waves and at most 256 registers; two
// workgroups fit a CU up to 5 query heads per group (64 KB of LDS each at 4, 74 KB at
// 5), one above (103 KB at 8 heads).
template <int G, bool F32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void suffix_stream_kernel(SuffixArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    suffix_stream_body<G, 4, (G > 4 ? 1 : kTokDepth), F32, F32, false>(a, (CK_LDS char *)smem_raw, blockIdx.x, threadIdx.x,
                                                                WgBarrier{});
}
static_assert(SfxLds<5, 4>::kBytes <= 80 * 1024, "two stand-alone workgroups per CU up to 5 heads");
static_assert(SfxLds<kMaxGroup, 4>::kBytes <= 160 * 1024, "one above");

// Folds the partials of one query head of a sequence cut by chunk boundaries
// (chunks ca < cb): the tail slot (1) of chunk ca and the head slot (0) of every
// later chunk, weighted by exp(lse - max). Online over batches
// of kB chunks whose loads all go out before any is used: one memory round trip
// per batch, not one per chunk (a long sequence spans many chunks, and the
// slowest sequence sets the kernel's time).
template <int G>
__device__ __forceinline__ void fold_cut(const float *part_o, const float *part_lse, int g, const ChunkMap &cm,
                                         int hq, int d4, int ca, int cb, float4 &o_out, float &lse_out) {
    constexpr int kB = 8;
    auto pidx = [&](int ch, int sl) { return (((int64_t)g * cm.P + ch) * 2 + sl) * G + hq; };
    float m = -INFINITY, wsum = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c0 = ca; c0 <= cb; c0 += kB) {
        float pl[kB];
        float4 po[kB];
        // every chunk from ca to cb holds windows (ChunkMap); past cb, an in-bounds
        // index, dropped below
#pragma unroll
        for (int j = 0; j < kB; ++j) {
            const int64_t p = pidx(min(c0 + j, cb), c0 + j == ca ? 1 : 0);
            pl[j] = part_lse[p];
            po[j] = *reinterpret_cast<const float4 *>(part_o + p * kD + 4 * d4);
        }
        float mb = m;
#pragma unroll
        for (int j = 0; j < kB; ++j) {
            if (c0 + j > cb) {  // weight 0, and 0 * 0 (the clamped partial may be infinite)
                pl[j] = -INFINITY;
                po[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            mb = fmaxf(mb, pl[j]);
        }
        const float mu = mb == -INFINITY ? 0.f : mb;
        const float r = exp2_fast((m - mu) * kLog2e);  // 0 from m = -inf
        acc.x *= r;
        acc.y *= r;
        acc.z *= r;
        acc.w *= r;
        wsum *= r;
#pragma unroll
        for (int j = 0; j < kB; ++j) {
            const float wgt = exp2_fast((pl[j] - mu) * kLog2e);
            acc.x = fmaf(wgt, po[j].x, acc.x);
            acc.y = fmaf(wgt, po[j].y, acc.y);
            acc.z = fmaf(wgt, po[j].z, acc.z);
            acc.w = fmaf(wgt, po[j].w, acc.w);
            wsum += wgt;
        }
        m = mb;
    }
    const float inv = wsum > 0.f ? 1.0f / wsum : 0.f;
    o_out = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
    lse_out = wsum > 0.f ? m + __logf(wsum) : -INFINITY;
}

// One workgroup of 32 G threads per (sequence, kv head): empty suffixes get
// O = 0, LSE = -inf; a sequence cut by chunk boundaries gets its partials
// folded; others return. The window prefix sums and the grid arithmetic come as
// leading scalar parameters (preloaded into SGPRs at wave launch, as for the
// cascade epilogue), so the first load waits for no kernel-argument load.
template <int G, bool F32>
__global__ __launch_bounds__(kMaxGroup * 32) void suffix_fixup_kernel(const int32_t *cw, int kv_heads, int batch,
                                                                      SuffixArgs a) {
    const int b = blockIdx.x / kv_heads;
    const int g = blockIdx.x % kv_heads;
    const int hq = threadIdx.x >> 5;
    const int d4 = threadIdx.x & 31;
    const int64_t beg = cw[b], end = cw[b + 1], W = cw[batch];
    const int64_t row = (int64_t)b * a.num_heads + g * G + hq;
    if (end == beg) {
        if constexpr (F32) {
            write_f32_row(a, row, d4, f32x4{0.f, 0.f, 0.f, 0.f}, -INFINITY);
        } else {
            *reinterpret_cast<uint2 *>(a.out + row * kD + 4 * d4) = make_uint2(0, 0);
            if (d4 == 0) a.lse[row] = -INFINITY;
        }
        return;
    }
    const ChunkMap cm{W, chunks_used(W, batch, a.chunks, a.split_few), 0};
    const int ca = cm.owner(beg);
    const int cb = cm.owner(end - 1);
    if (ca == cb) return;  // written by the stream kernel
    float4 o;
    float l;
    fold_cut<G>(a.part_o, a.part_lse, g, cm, hq, d4, ca, cb, o, l);
    if constexpr (F32) {
        write_f32_row(a, row, d4, f32x4{o.x, o.y, o.z, o.w}, l);
    } else {
        *reinterpret_cast<uint2 *>(a.out + row * kD + 4 * d4) =
            make_uint2(pack_bf16x2(o.x, o.y), pack_bf16x2(o.z, o.w));
        if (d4 == 0) a.lse[row] = l;
    }
}

// Cascade epilogue (fused cascade decode): one workgroup of 32 G threads per
// (sequence, kv head), 32 threads x 4 dims per query head. Folds the stage-1
// split partials of the sequence's query token, the suffix result (whole, split
// partials or empty) and merges the two with the lse_merge arithmetic
//   m = max(l1, l2); w1 = exp(l1 - m); w2 = exp(l2 - m)
//   out = (o1 w1 + o2 w2) * (1 / (w1 + w2)),  lse = m + log(w1 + w2)
// (ascend-kernel/csrc/ops/lse_merge/op_kernel/kernel_lse_merge.cpp:237-289);
// a side at -inf has weight 0, both at -inf give out = 0, lse = -inf.
// Latency, not bytes, bounds it, so the loads go out in dependency order: the
// window prefix sums, then every stage-1 partial of the row (up to kPreS
// splits), then the suffix result those sums locate; the arithmetic waits once.
// What those first loads need (the prefix sums, the stage-1 result and the row
// arithmetic) comes as scalar kernel parameters ahead of the struct: the
// compiler preloads leading scalar parameters into SGPRs at wave launch, which
// takes the kernel-argument load off the first round trip.
// The host fills the whole struct; launch_epilogue passes s1, cw, b0, nb,
// num_heads and kv_heads again as the leading parameters the kernel reads.
struct EpilogueArgs {
    Stage1Result s1;
    const uint16_t *o2;     // bf16 [nb][H][kD] whole-sequence suffix results
    const float *lse2;      // [nb * H]
    const float *part_o;    // suffix partials [kv head groups][chunks][2][G][kD]
    const float *part_lse;  // [kv head groups][chunks][2][G]
    const int32_t *cw;      // [nb + 1] window prefix sums of the group
    uint16_t *out;          // bf16 [batch][H][kD]
    float *lse_out;         // [batch * H]
    int64_t b0;
    int nb;
    int num_heads;
    int kv_heads;  // kv head groups, as in SuffixArgs
    int chunks;
    int split_few;  // as in SuffixArgs
};

template <int G, bool PAIRS>
__global__ __launch_bounds__(kMaxGroup * 32) void cascade_epilogue_kernel(const int32_t *cw, const float *s1o, const float *s1lse,
                                                                         int64_t rows, int kv_heads, int nb, int num_heads,
                                                                         int b0, int splits, EpilogueArgs e) {
    constexpr int kBatch = 8;   // splits folded per rescale step
    constexpr int kPreS = 16;   // splits loaded up front
    const int bl = blockIdx.x / kv_heads;
    const int g = blockIdx.x % kv_heads;
    const int hq = threadIdx.x >> 5;
    const int d4 = threadIdx.x & 31;
    const int h = g * G + hq;
    const int64_t row = (int64_t)(b0 + bl) * num_heads + h;

    const int64_t beg = cw[bl], end = cw[bl + 1], W = cw[nb];

    // ---- stage-1 loads: the first kPreS splits of this query row ------------------
    float ls[kPreS];
    float4 os[kPreS];
    if (splits <= 1) {
        os[0] = *reinterpret_cast<const float4 *>(s1o + row * kD + 4 * d4);
        ls[0] = s1lse[row * 8];
    } else {
#pragma unroll
        for (int j = 0; j < kPreS; ++j) {
            const int s = j < splits ? j : splits - 1;
            ls[j] = s1lse[(int64_t)s * rows + row];
            os[j] = *reinterpret_cast<const float4 *>(s1o + ((int64_t)s * rows + row) * kD + 4 * d4);
        }
    }

    // ---- suffix: empty, whole (bf16 result) or cut by chunk boundaries ------------
    float l2 = -INFINITY;
    float4 o2 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (end > beg) {
        const ChunkMap cm = PAIRS ? ChunkMap{W, e.chunks, e.split_few}
                                  : ChunkMap{W, chunks_used(W, nb, e.chunks, e.split_few), 0};
        const int ca = cm.owner(beg);
        const int cb = cm.owner(end - 1);
        if (ca == cb) {
            const int64_t r2 = (int64_t)bl * num_heads + h;
            const uint2 w = *reinterpret_cast<const uint2 *>(e.o2 + r2 * kD + 4 * d4);
            o2 = make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
            l2 = e.lse2[r2];
        } else {
            fold_cut<G>(e.part_o, e.part_lse, g, cm, hq, d4, ca, cb, o2, l2);
        }
    }

    // ---- stage 1: fold the split partials (online, kBatch splits per step) --------
    float l1;
    float4 o1;
    if (splits <= 1) {
        o1 = os[0];
        l1 = ls[0];
    } else {
        float m = -INFINITY, wsum = 0.f;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        auto step = [&](const float *lb, const float4 *ob, int s0) {
            float mb = m;
#pragma unroll
            for (int j = 0; j < kBatch; ++j)
                if (s0 + j < splits) mb = fmaxf(mb, lb[j]);
            const float mu = mb == -INFINITY ? 0.f : mb;
            const float r = exp2_fast((m - mu) * kLog2e);
            acc.x *= r; acc.y *= r; acc.z *= r; acc.w *= r;
            wsum *= r;
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const float wgt = s0 + j < splits ? exp2_fast((lb[j] - mu) * kLog2e) : 0.f;
                acc.x = fmaf(wgt, ob[j].x, acc.x);
                acc.y = fmaf(wgt, ob[j].y, acc.y);
                acc.z = fmaf(wgt, ob[j].z, acc.z);
                acc.w = fmaf(wgt, ob[j].w, acc.w);
                wsum += wgt;
            }
            m = mb;
        };
#pragma unroll
        for (int s0 = 0; s0 < kPreS; s0 += kBatch)
            if (s0 < splits) step(ls + s0, os + s0, s0);
        for (int s0 = kPreS; s0 < splits; s0 += kBatch) {
            float lb[kBatch];
            float4 ob[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int s = s0 + j < splits ? s0 + j : splits - 1;
                lb[j] = s1lse[(int64_t)s * rows + row];
                ob[j] = *reinterpret_cast<const float4 *>(s1o + ((int64_t)s * rows + row) * kD + 4 * d4);
            }
            step(lb, ob, s0);
        }
        const float inv = wsum > 0.f ? 1.0f / wsum : 0.f;
        o1 = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
        l1 = wsum > 0.f ? m + __logf(wsum) : -INFINITY;
    }

    // ---- merge --------------------------------------------------------------------
    const float m = fmaxf(l1, l2);
    uint2 ow = make_uint2(0, 0);
    float lse_v = -INFINITY;
    if (m != -INFINITY) {
        const float w1 = expf(l1 - m), w2 = expf(l2 - m);
        const float s = w1 + w2;
        const float sinv = 1.0f / s;
        auto mix = [&](float x1, float x2) {
            const float t1 = (w1 == 0.f) ? 0.f : x1 * w1;
            const float t2 = (w2 == 0.f) ? 0.f : x2 * w2;
            return (t1 + t2) * sinv;
        };
        ow = make_uint2(pack_bf16x2(mix(o1.x, o2.x), mix(o1.y, o2.y)), pack_bf16x2(mix(o1.z, o2.z), mix(o1.w, o2.w)));
        lse_v = m + logf(s);
    }
    *reinterpret_cast<uint2 *>(e.out + row * kD + 4 * d4) = ow;
    if (d4 == 0) e.lse_out[row] = lse_v;
}

// Fused cascade kernel: workgroup i runs stage-1 unit i on waves 0-3 (the
// 128-row body with a 3-slot ring) and suffix chunk 2j on waves 4-7 (the stream
// body on 4 waves, 32-token windows) side by side on one CU: each SIMD holds one
// MFMA wave and one streaming wave, which fill each other's stalls, and the
// prefix pages and the suffix pages stream at the same time. When its stage-1
// unit is done, waves 0-3 stream suffix chunk 2j + 1, the last (256 - split) /
// 256 of the workgroup's windows, in the LDS the stage-1 tiles used: the two
// roles end together instead of the stage-1 waves idling while the suffix
// waves finish. Each role has its own LDS region and barrier; neither waits
// for the other.
constexpr int kFusedS1Lds = s1::wide_lds_bytes<3>();
template <int G>
using FusedSfx = SfxLds<G, 4, (G <= 4 ? kQSlots : 4), (G <= 4 ? 2 : 1)>;  // the stream body's layout on 4 waves
template <int G>
constexpr int fused_lds_bytes() { return kFusedS1Lds + FusedSfx<G>::kBytes + 32; }
static_assert(fused_lds_bytes<4>() <= 160 * 1024 && fused_lds_bytes<kMaxGroup>() <= 160 * 1024,
              "one fused workgroup per CU");
static_assert(FusedSfx<4>::kBytes <= kFusedS1Lds && FusedSfx<kMaxGroup>::kBytes <= kFusedS1Lds,
              "the stage-1 waves' stream body fits the tile ring");

template <int G>
__global__ __launch_bounds__(512) void cascade_fused_kernel(s1::Stage1Args s1a, int n1, SuffixArgs sa, int n2) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    CK_LDS char *smem = (CK_LDS char *)smem_raw;
    CK_LDS int *bars = (CK_LDS int *)(smem + kFusedS1Lds + FusedSfx<G>::kBytes);
    if (threadIdx.x < 5) bars[threadIdx.x] = 0;  // two role barriers, the scan flag
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = wave < 4 ? 1 : 0;  // 1: stage-1 waves (suffix chunk 2j + 1 afterwards)
    const GroupBarrier bar{bars + 2 * (1 - role), bars + 2 * (1 - role) + 1, 4, &g_wait_giveups};
    if (role == 1 && (int)blockIdx.x < n1) {
        s1::stage1_wide_body<4, 3>(s1a, smem, blockIdx.x, n1, threadIdx.x, bar);
        // The stream body's arguments stay in scalar registers across the stage-1
        // body (the compiler loads them with the kernel's other arguments at the
        // start): without a use here it reloads them from the kernel-argument
        // segment after the barrier below, a memory round trip on the stage-1
        // waves' way to their suffix windows (0.3-0.5 us per step).
        asm volatile("" ::"s"(sa.q), "s"(sa.head_off), "s"(sa.scale_log2), "s"(sa.cw_out));
        bar.sync();  // every stage-1 wave is done with the tile ring
    }
    if ((int)blockIdx.x < n2) {
        // The stream roles take kv head group blockIdx + 3 (mod kv_heads) while the
        // stage-1 unit order puts kv head x on XCD x (blockIdx % 8) at the usual
        // shapes: a workgroup's two roles then read different kv heads. Pages of
        // some kv heads are slower to fetch than others (by their address bits: up
        // to ~15% measured), and with both roles on one head their slowness stacked
        // on the same workgroups, which set the kernel's end (1.1-1.6 us per step).
        constexpr int kRoleRot = 3;
        const int g = ((int)blockIdx.x + kRoleRot) % sa.kv_heads, j = (int)blockIdx.x / sa.kv_heads;
        // the streaming waves scan the lengths; the stage-1 waves reuse that scan
        suffix_stream_body<G, 4, kTokDepth, false, (G > 4), true, FusedSfx<G>>(
            sa, smem + (role ? 0 : kFusedS1Lds), (2 * j + role) * sa.kv_heads + g, threadIdx.x & 255, bar, bars + 4,
            role ? smem + kFusedS1Lds : nullptr);
    }
}

int64_t ceil_div(int64_t x, int64_t y) { return (x + y - 1) / y; }

// partial (O, LSE) slots: 2 per (query head, chunk) -- the same count for any
// split of the heads into kv head groups
int64_t group_parts(int64_t num_heads, int64_t chunks) { return num_heads * chunks * 2; }

template <int G, bool PAIRS>
void launch_epilogue(const EpilogueArgs &e, unsigned grid, hipStream_t st) {
    hipLaunchKernelGGL((cascade_epilogue_kernel<G, PAIRS>), dim3(grid), dim3(32 * G), 0, st, e.cw, e.s1.o, e.s1.lse, e.s1.rows,
                       e.kv_heads, e.nb, e.num_heads, (int)e.b0, e.s1.splits, e);
}

template <int G>
int launch_fused(const s1::Stage1Args &s1a, int64_t n1, const SuffixArgs &a, const EpilogueArgs &epi,
                 hipStream_t st) {
    static std::atomic<uint64_t> lds_set{0};
    constexpr int kLds = fused_lds_bytes<G>();
    int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(&cascade_fused_kernel<G>), kLds, lds_set);
    if (rc != CK_OK) return rc;
    const int64_t n2 = (int64_t)a.kv_heads * (a.chunks / 2);  // chunk pairs (PAIRS)
    const int64_t grid = n1 > n2 ? n1 : n2;
    hipLaunchKernelGGL(cascade_fused_kernel<G>, dim3((unsigned)grid), dim3(512), kLds, st, s1a, (int)n1, a, (int)n2);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return static_cast<int>(e);
    launch_epilogue<G, true>(epi, (unsigned)(a.batch * a.kv_heads), st);
    CK_RETURN_LAUNCH();
}

template <int G, bool F32 = false>
int launch_suffix(const SuffixArgs &a, bool fixup, const EpilogueArgs *epi, hipStream_t st) {
    static std::atomic<uint64_t> lds_set{0};
    constexpr int kLds = SfxLds<G, 4>::kBytes;
    int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(&suffix_stream_kernel<G, F32>), kLds, lds_set);
    if (rc != CK_OK) return rc;
    hipLaunchKernelGGL((suffix_stream_kernel<G, F32>), dim3((unsigned)(a.kv_heads * a.chunks)), dim3(256), kLds, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return static_cast<int>(e);
    if (fixup)
        hipLaunchKernelGGL((suffix_fixup_kernel<G, F32>), dim3((unsigned)(a.batch * a.kv_heads)), dim3(32 * G), 0, st,
                           (const int32_t *)a.cw_out, a.kv_heads, a.batch, a);
    if (epi) launch_epilogue<G, false>(*epi, (unsigned)(a.batch * a.kv_heads), st);
    CK_RETURN_LAUNCH();
}

int check_suffix_dims(int64_t batch, int64_t num_heads, int64_t kv_heads, int64_t head_dim, int64_t kv_cap) {
    if (batch < 0 || batch > 0x7FFFFFFF || kv_cap < 0) return CK_E_INVALID_ARG;  // sequence indices are 32-bit
    if (head_dim != kD) return CK_E_UNSUPPORTED;
    if (kv_heads <= 0 || num_heads <= 0 || num_heads % kv_heads != 0) return CK_E_INVALID_ARG;
    if (num_heads > (1 << 16)) return CK_E_INVALID_ARG;
    if (kv_cap > (int64_t)1 << 30) return CK_E_INVALID_ARG;
    return CK_OK;
}

}  // namespace

// Query-head groups per kv head: a GQA group of more than kMaxGroup heads is
// split into the fewest equal groups of at most kMaxGroup heads. Each group is
// streamed as if it had its own kv head (the kernel reads the shared physical
// head), so the kernels keep their per-head registers bounded for any group.
int64_t suffix_sub_groups(int64_t num_heads, int64_t kv_heads) {
    const int64_t group = num_heads / kv_heads;
    for (int64_t n = (group + kMaxGroup - 1) / kMaxGroup; n < group; ++n)
        if (group % n == 0) return n;
    return group;
}

// Sequences per stream-kernel launch: the window/length prefix sums live in
// LDS (kMaxBatch entries) and must stay below 2^31 tokens.
int64_t suffix_group_batch(int64_t kv_cap) {
    int64_t n = kMaxBatch;
    const int64_t cap = kv_cap > 0 ? kv_cap : 1;
    if (n > 0x7FFFFFFF / cap) n = 0x7FFFFFFF / cap;
    return n < 1 ? 1 : n;
}

// Chunks of the window list (workgroups) per kv head group: a grid that is resident
// at once over all groups, one or two workgroups per CU, and no more chunks per
// sequence than folding their partials is worth.
// * One per CU above 5 query heads per group: two do not fit its LDS
//   (suffix_stream_kernel), and a second generation pays the start-up again
//   (64 / 8 heads, 64 suffixes of mean 512: 42.5 us with 512 workgroups, 36.3 with
//   256; 256 suffixes 115 / 109; 4 of mean 64 27.7 / 10.8).
// * Up to 5 heads the grid holds two per CU, and the kernels use half of them once
//   sequences hold 12 windows in the mean: half the partials and start-ups (512 / 256
//   chunks over the groups at 16 windows a sequence: 40 / 8 heads, 16 sequences 1.09, 64
//   1.03, 256 1.05 times the time; at 20 windows 1.05, 1.07, 1.03; 8 requests of 4096 on 8 /
//   2 heads 1.21). Below, the closes bound it and the second workgroup hides them (8
//   windows: 130 of 40 / 8 0.96; 4: 64 0.94, 256 0.90; 2: 256 0.83). A chunk of more than
//   one phase's 8 segments costs a phase more, and where the groups do not divide 256 to
//   15/16 CUs idle (71 of one head: 3 chunks on 213 CUs 59.1 us, 7 47.5): all, then.
// * A sequence of n windows spans chunks / batch chunks; its fold takes a memory
//   round trip per 8 (about 0.15 us a chunk) and a chunk's windows about 0.5 us
//   each: sqrt(cap / 8) chunks per sequence balance the two (8 / 1 heads, 7 requests
//   of 4096: 26.2 us over 512 chunks, 13.8 over 112, 15.6 over 56).
SuffixChunks suffix_default_chunks(int64_t batch, int64_t num_heads, int64_t kv_heads, int64_t kv_cap) {
    const int64_t groups = kv_heads * suffix_sub_groups(num_heads, kv_heads);
    const int64_t per_seq = std::max<int64_t>(8, (int64_t)std::sqrt((double)kv_cap / 8));
    auto upto = [&](int64_t grid) { return std::max<int64_t>(1, std::min(grid / groups, batch * per_seq)); };
    const int64_t most = upto(num_heads / groups > 5 ? 256 : 512), few = upto(256);
    return SuffixChunks{most, 256 / groups * groups >= 240 && batch <= kQSlots * few ? few : most};
}

// The chunk count the plan reports, whatever the batch: two workgroups per CU. A call
// that passes it (or none) gets suffix_default_chunks, which is never more.
int64_t suffix_plan_chunks(int64_t num_heads, int64_t kv_heads) {
    const int64_t p = 512 / (kv_heads * suffix_sub_groups(num_heads, kv_heads));
    return p > 0 ? p : 1;
}

int64_t suffix_fused_chunks(int64_t num_heads, int64_t kv_heads) {
    const int64_t groups = kv_heads * suffix_sub_groups(num_heads, kv_heads);
    const int64_t p = 256 / groups;
    return 2 * (p > 0 ? p : 1);  // a pair of chunks per fused workgroup
}

int64_t suffix_group_ws_bytes(int64_t nb, int64_t num_heads, int64_t kv_heads, int64_t chunks) {
    const int64_t parts = group_parts(num_heads, chunks);
    return parts * (kD + 1) * (int64_t)sizeof(float) + (nb + 1) * (int64_t)sizeof(int32_t) + 256;
}

int suffix_launch_group(const void *q, const void *k, const void *v, const int32_t *block_table, int64_t bt_cols,
                        const int64_t *kv_seqlens, int64_t b0, int64_t nb, int64_t num_heads, int64_t kv_heads,
                        int64_t num_blocks, int64_t kv_layout, float scale, int64_t kv_cap, SuffixChunks chunks,
                        void *out, float *lse, void *group_ws, const Stage1Result *cascade, void *final_out,
                        float *final_lse, hipStream_t stream, const s1::Stage1Args *fused, int64_t fused_units,
                        bool f32_out) {
    const int64_t sub = suffix_sub_groups(num_heads, kv_heads);
    const int64_t G = num_heads / kv_heads / sub;  // query heads per workgroup
    const int64_t parts = group_parts(num_heads, chunks.most);
    SuffixArgs a;
    a.q = static_cast<const uint16_t *>(q) + b0 * num_heads * kD;
    a.k = static_cast<const uint16_t *>(k);
    a.v = static_cast<const uint16_t *>(v);
    a.bt = block_table + b0 * bt_cols;
    a.kv_seqlens = kv_seqlens + b0;
    a.out = static_cast<uint16_t *>(out);
    a.lse = lse;
    a.part_o = static_cast<float *>(group_ws);
    a.part_lse = a.part_o + parts * kD;
    a.cw_out = reinterpret_cast<int32_t *>(a.part_lse + parts);
    a.bt_cols = bt_cols;
    a.num_blocks = num_blocks;
    a.page_stride = (int64_t)kPage * kv_heads * kD;
    a.tok_stride = kv_layout == CK_KV_BNSD ? kD : kv_heads * kD;
    a.head_off = kv_layout == CK_KV_BNSD ? (int64_t)kPage * kD : kD;
    a.batch = (int)nb;
    a.num_heads = (int)num_heads;
    a.kv_heads = (int)(kv_heads * sub);
    a.kv_sub = (int)sub;
    a.kv_cap = (int)kv_cap;
    a.chunks = (int)chunks.most;
    a.split_few = fused && cascade ? fused_split(G) : (int)chunks.few;
    a.scale_log2 = scale * kLog2e;
    EpilogueArgs e;
    if (cascade) {
        e.s1 = *cascade;
        e.o2 = a.out;
        e.lse2 = a.lse;
        e.part_o = a.part_o;
        e.part_lse = a.part_lse;
        e.cw = a.cw_out;
        e.out = static_cast<uint16_t *>(final_out);
        e.lse_out = final_lse;
        e.b0 = b0;
        e.nb = (int)nb;
        e.num_heads = (int)num_heads;
        e.kv_heads = a.kv_heads;
        e.chunks = a.chunks;
        e.split_few = a.split_few;
    }
    if (fused && cascade) {
        switch (G) {
            case 1: return launch_fused<1>(*fused, fused_units, a, e, stream);
            case 2: return launch_fused<2>(*fused, fused_units, a, e, stream);
            case 3: return launch_fused<3>(*fused, fused_units, a, e, stream);
            case 4: return launch_fused<4>(*fused, fused_units, a, e, stream);
            case 5: return launch_fused<5>(*fused, fused_units, a, e, stream);
            case 6: return launch_fused<6>(*fused, fused_units, a, e, stream);
            case 7: return launch_fused<7>(*fused, fused_units, a, e, stream);
            default: return launch_fused<8>(*fused, fused_units, a, e, stream);
        }
    }
    if (f32_out) {  // stage-1's decode form
        switch (G) {
            case 1: return launch_suffix<1, true>(a, true, nullptr, stream);
            case 2: return launch_suffix<2, true>(a, true, nullptr, stream);
            case 3: return launch_suffix<3, true>(a, true, nullptr, stream);
            case 4: return launch_suffix<4, true>(a, true, nullptr, stream);
            case 5: return launch_suffix<5, true>(a, true, nullptr, stream);
            case 6: return launch_suffix<6, true>(a, true, nullptr, stream);
            case 7: return launch_suffix<7, true>(a, true, nullptr, stream);
            default: return launch_suffix<8, true>(a, true, nullptr, stream);
        }
    }
    const bool fixup = cascade == nullptr;
    const EpilogueArgs *ep = cascade ? &e : nullptr;
    switch (G) {
        case 1: return launch_suffix<1>(a, fixup, ep, stream);
        case 2: return launch_suffix<2>(a, fixup, ep, stream);
        case 3: return launch_suffix<3>(a, fixup, ep, stream);
        case 4: return launch_suffix<4>(a, fixup, ep, stream);
        case 5: return launch_suffix<5>(a, fixup, ep, stream);
        case 6: return launch_suffix<6>(a, fixup, ep, stream);
        case 7: return launch_suffix<7>(a, fixup, ep, stream);
        default: return launch_suffix<8>(a, fixup, ep, stream);
    }
}

}  // namespace ck

using namespace ck;

extern "C" int ck_suffix_decode_plan(int64_t batch, int64_t num_heads, int64_t kv_heads, int64_t head_dim,
                                     int64_t kv_cap, int64_t *num_splits, int64_t *workspace_bytes) {
    int rc = check_suffix_dims(batch, num_heads, kv_heads, head_dim, kv_cap);
    if (rc != CK_OK) return rc;
    if (!num_splits || !workspace_bytes) return CK_E_NULL_PTR;
    const int64_t chunks = suffix_plan_chunks(num_heads, kv_heads);
    const int64_t nb = batch < suffix_group_batch(kv_cap) ? batch : suffix_group_batch(kv_cap);
    *num_splits = chunks;
    *workspace_bytes = batch > 0 ? suffix_group_ws_bytes(nb, num_heads, kv_heads, chunks) : 0;
    return CK_OK;
}

extern "C" int ck_suffix_decode(const void *q, const void *k, const void *v, const int32_t *block_table,
                                int64_t bt_cols, const int64_t *kv_seqlens, int64_t batch, int64_t num_heads,
                                int64_t kv_heads, int64_t head_dim, int64_t num_blocks, int64_t block_size,
                                int64_t kv_layout, float scale, int64_t kv_cap, int64_t num_splits, void *out,
                                float *lse, void *workspace, int64_t workspace_bytes, void *stream) {
    int rc = check_suffix_dims(batch, num_heads, kv_heads, head_dim, kv_cap);
    if (rc != CK_OK) return rc;
    if (block_size != kPage) return CK_E_UNSUPPORTED;
    if (kv_layout != CK_KV_NHD && kv_layout != CK_KV_BNSD) return CK_E_INVALID_ARG;
    if (bt_cols < 0 || num_blocks < 0 || kv_cap > bt_cols * kPage) return CK_E_INVALID_ARG;
    if (batch == 0) return CK_OK;
    if (!q || !k || !v || !block_table || !kv_seqlens || !out || !lse) return CK_E_NULL_PTR;
    // q/k/v rows and the workspace partials move up to 16 bytes per lane; the
    // fix-up kernel stores bf16 O four elements (8 bytes) at a time
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(v, 16) || !aligned_to(out, 8) ||
        !aligned_to(lse, 4) || !aligned_to(workspace, 16))
        return CK_E_INVALID_ARG;
    const SuffixChunks chunks = num_splits > 0 && num_splits != suffix_plan_chunks(num_heads, kv_heads)
                                    ? SuffixChunks{num_splits, num_splits}
                                    : suffix_default_chunks(batch, num_heads, kv_heads, kv_cap);
    if (kv_heads * suffix_sub_groups(num_heads, kv_heads) * chunks.most > 0x7FFFFFFF || chunks.most > (1 << 20))
        return CK_E_INVALID_ARG;
    const int64_t per_launch = suffix_group_batch(kv_cap);
    const int64_t nbmax = batch < per_launch ? batch : per_launch;
    if (workspace == nullptr || workspace_bytes < suffix_group_ws_bytes(nbmax, num_heads, kv_heads, chunks.most))
        return CK_E_WORKSPACE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    for (int64_t b0 = 0; b0 < batch; b0 += per_launch) {
        const int64_t nb = batch - b0 < per_launch ? batch - b0 : per_launch;
        rc = suffix_launch_group(q, k, v, block_table, bt_cols, kv_seqlens, b0, nb, num_heads, kv_heads,
                                 num_blocks, kv_layout, scale, kv_cap, chunks, static_cast<uint16_t *>(out) + b0 * num_heads * kD,
                                 lse + b0 * num_heads, workspace, nullptr, nullptr, nullptr, st, nullptr, 0);
        if (rc != CK_OK) return rc;
    }
    return CK_OK;
}

extern "C" int ck_wait_giveups(uint64_t *count, int reset) {
    if (!count) return CK_E_NULL_PTR;
    unsigned int v = 0;
    hipError_t e = hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_wait_giveups), sizeof(v), 0, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return static_cast<int>(e);
    *count = v;
    if (reset) {
        const unsigned int zero = 0;
        e = hipMemcpyToSymbol(HIP_SYMBOL(g_wait_giveups), &zero, sizeof(zero), 0, hipMemcpyHostToDevice);
        if (e != hipSuccess) return static_cast<int>(e);
    }
    return CK_OK;
}
