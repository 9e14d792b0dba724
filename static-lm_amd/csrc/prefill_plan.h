// Which prefill kernel runs for a batch.  No HIP dependencies, so host code
// and CPU tests can include it as well as the launcher.
#pragma once

namespace slm {

// The kernels of a prefill, numbered as SLM_PF_* in slm_attn.h.  The first ones
// are forms of the f32 kernel (prefill_mfma.hip), kSplit* those of the
// split-bf16 kernel (prefill_split.hip): eight waves per workgroup, each one
// (head, 16-row block, key split).
enum class PrefillKernel : int {
    kFourHeads = 0,
    kThreeHeads = 1,
    kTwoHeads = 2,
    kOneHead = 3,
    kKeySplit = 4,
    kPairedFourHeads = 5,
    kPairedOneHead = 9,
    kSplitKeys = 10,         // four (head, block), paired blocks, two key splits
    kSplitPaired = 11,       // eight (head, block), paired blocks
    kSplitConsecutive = 12,  // eight (head, block), consecutive blocks
};

inline bool on_split_kernel(PrefillKernel k) {
    return k == PrefillKernel::kSplitKeys || k == PrefillKernel::kSplitPaired ||
           k == PrefillKernel::kSplitConsecutive;
}

// Query heads per workgroup (hw, all of one KV head) and 16-row query blocks
// per workgroup (qs) of the head-group tiling.
struct PrefillTiling {
    int hw;
    int qs;
};

inline PrefillTiling prefill_tiling(int kv_mul) {
    if (kv_mul % 4 == 0) return {4, 1};
    if (kv_mul % 3 == 0) return {3, 1};
    if (kv_mul % 2 == 0) return {2, 2};
    return {1, 4};
}

// Whether the split kernel takes a prefill of hd 64 with `cols` (head, 16-row
// block) columns.  Its arithmetic per key tile is half that of hd 128 behind the
// same set-up and barriers, so it takes more columns to win, and the f32
// kernel's four key splits serve what does not fill the CUs: from three columns
// per CU (32 heads in 8 KV heads: 256 rows, two per CU, 13.8 against 12.5 us in
// f32, 384 rows 17.6 against 20.8, 512 rows 20.8 against 26.7).  Key splits up
// to eight columns per CU (16 heads, 2048 rows: 79.7 us, paired 81.4, f32 109.9;
// 3000 rows: 152, 139, 201), paired blocks up to sixteen (32 heads, 2048 rows:
// 106 us, consecutive 112, f32 150; 3000 rows: 214, 200, 312).
//
// With one workgroup (four columns) per CU its time follows the heaviest
// block's keys (10.5 us + 23 ns a key), that of the f32 kernel, whose small
// workgroups fill in behind each other, the keys that all columns see together.
// So long histories of few columns need more of them, counted by the keys that
// the average row sees: split against f32, start 0, at 3.0 / 3.5 / 3.9 columns
// per CU 4 heads 81.8 / 95.1 / 105.6 against 62.4 / 83.5 / 103.3 us (3072 to 3994
// rows), 6 heads 57.8 / 67.3 / 74.3 against 48.8 / 64.5 / 75.6, 9 heads 42.2 /
// 48.4 / - against 39.5 / 48.5 / -, 12 heads (1024 rows) 32.9 against 33.0; 8
// heads, 1536 rows at start 600 63.0 against 65.2.  With a second workgroup on
// some of the CUs, at 4.1 / 4.5 / 5.0: 8 heads 67.6 / 73.8 / 81.9 against 63.2 /
// 71.5 / 84.1, 12 heads 49.4 / 54.0 against 49.0 / 54.7, 14 heads (1200 rows) 41.8
// against 42.8.
inline bool hd64_splits(long cols, int cus, int start, int n) {
    if (cols < 3L * cus) return false;
    const double keys = (double)start + n;
    const double seen = (double)cols / cus * (start + 0.5 * n) / keys;
    if (cols <= 4L * cus) return seen >= 2.2 - 768.0 / keys;
    const double least = 3.0 - 1280.0 / keys;
    return seen >= (least < 2.5 ? least : 2.5);
}

// Which kernel a prefill of n rows from row `start` runs, for head_dim,
// num_heads query heads (kv_mul per KV head) on a device of `cus` CUs: a pure
// function of the batch, the shape and the CU count.  The launcher and the
// kernel query of the C ABI both call it.
inline PrefillKernel prefill_plan(int head_dim, int num_heads, int kv_mul, int cus, int start,
                                  int n) {
    const PrefillTiling t = prefill_tiling(kv_mul);
    const long cols = ((long)n + 15) / 16 * num_heads;  // (head, 16-row block)
    if (head_dim == 128) {
        // Short prefills whose head-group tiling gives at most one workgroup
        // per CU run one wave per SIMD, and the heaviest causal block sets
        // the time (its tiles in series: 16 at 512 rows, against 8.5 on
        // average).  Pairs of blocks i and n_qb-1-i, one head and four key
        // splits per workgroup (no GQA sharing of the tiles, 200 VGPRs) give
        // every SIMD the same share, from 256 rows and while that grid fits
        // the CUs once: below 256 rows 13% slower than four heads.  Four split
        // tiles do not fit the LDS, and the split kernel's two key splits stay
        // behind: 256 rows 20.7 against 22.1 us, 512 rows of 16 heads 28.4
        // against 32.9, 256 rows at start 8000 348 against 385.
        const long wgs = (long)((n + 16 * t.qs - 1) / (16 * t.qs)) * (num_heads / t.hw);
        const long pairs = ((n + 15) / 16 + 1) / 2;
        if (n >= 256 && wgs <= cus && pairs * num_heads <= cus)
            return PrefillKernel::kPairedOneHead;
        // Under four key tiles there is little to gain and the splitting's
        // set-up shows (Llama-3-8B shape, per call, split against f32: 64 rows
        // 13.6 against 12.1 us, 128 rows 16.5 against 17.4).  Then all eight
        // waves on as few columns as fill the CUs: with two key splits while
        // that grid fits the CUs once (512 rows 34.3 against 39.5 us paired
        // and 37.0 in f32; 512 rows at start 2000 131 against 181 and 180),
        // then paired blocks while that does (1024 rows 71 against 91 and 87
        // us consecutive; 777 rows at start 1000 131 against 141), then
        // consecutive ones (2048 rows 187 against 214 paired; 4096 rows 690
        // against 780).
        if ((long)start + n >= 128)
            return cols <= 4L * cus   ? PrefillKernel::kSplitKeys
                   : cols <= 8L * cus ? PrefillKernel::kSplitPaired
                                      : PrefillKernel::kSplitConsecutive;
    }
    if (head_dim == 64 && hd64_splits(cols, cus, start, n))
        return cols <= 8L * cus    ? PrefillKernel::kSplitKeys
               : cols <= 16L * cus ? PrefillKernel::kSplitPaired
                                   : PrefillKernel::kSplitConsecutive;
    // Short prefills, head_dim <= 64: when the head-group tiling gives fewer
    // than two workgroups per CU, one head and one 16-row query block per
    // workgroup with its key tiles split over four waves, as long as the
    // heaviest block keeps two tiles per split: more workgroups, and the
    // heaviest block's tiles walked by four SIMDs instead of one.  (Each
    // thread then prefetches four tiles' share: 169 VGPRs at hd 64, 312 at
    // hd 128.)
    if (head_dim <= 64) {
        constexpr int KSP = 4;
        const int qs = t.hw == 1 ? 4 : t.hw == 2 ? 2 : 1;
        const long wgs = (long)((n + 16 * qs - 1) / (16 * qs)) * (num_heads / t.hw);
        const long tiles = ((long)start + n + 31) / 32;  // the heaviest block's
        if (wgs < 2L * cus && tiles >= 2L * KSP) return PrefillKernel::kKeySplit;
    }
    if (head_dim <= 96 && t.hw == 4) {
        // Paired blocks (i and n_qb-1-i) in the four-head kernel: where the
        // four-head grid has more workgroups than CUs and the paired grid
        // (8-wave workgroups, one per CU) is at most one or two per CU.
        // Interleaved per call against the four-head kernel, GQA 4 (32 heads):
        // at 1024 rows hd 16 / 32 / 48 / 96 23.8 / 35.5 / 48.2 / 77.8 against
        // 26.8 / 38.7 / 54.8 / 91.9 us, at 2048 rows 55.7 / 87.4 / 123.3 /
        // 222.2 against 60.8 / 97.2 / 137.9 / 248.9, hd 96 at 768 rows 59.3
        // against 66.0; it lost with 1.5 per CU (1536 rows: +2.4% at hd 96)
        // and from three per CU (4096 rows: +1.8%, against the four-head
        // kernel's three 4-wave workgroups per CU); with three heads per
        // workgroup and for MHA it gained nothing or lost (hd 64: SmolLM2
        // shape; MHA at 2048 rows +19%).
        const long wgs = (long)((n + 15) / 16) * (num_heads / 4);
        const long pwgs = (((long)n + 15) / 16 + 1) / 2 * (num_heads / 4);
        if (wgs > cus && (pwgs <= cus || pwgs == 2L * cus))
            return PrefillKernel::kPairedFourHeads;
    }
    if (t.hw == 4) return PrefillKernel::kFourHeads;
    if (t.hw == 3) return PrefillKernel::kThreeHeads;
    if (t.hw == 2) return PrefillKernel::kTwoHeads;
    return PrefillKernel::kOneHead;
}

// Whether the attention kernel of a prefill also appends the batch's K and V
// rows.  Every workgroup must then hold a whole KV head's queries (one block
// group, all heads of the KV head), so that each row has one writer and every
// reader of a new row is in its workgroup: batches of at most 16 rows (four or
// three heads per KV head), 32 (two) or 64 (one).  It saves the append launch,
// which takes as long as such a batch's attention (16 rows of 6 heads of 48, per
// call: 7.1 us appended apart, 4.6 inside), but few workgroups then wait for all
// the rows: up to 2560 values of K and V each per KV head.  Apart against
// inside, 6 heads without GQA: hd 48, 48 / 56 rows 7.2 / 7.3 against 7.1 / 7.5 us;
// hd 64, 40 / 64 rows 7.7 / 8.1 against 7.2 / 8.5; hd 96, 24 / 33 rows 7.3 / 9.2
// against 7.0 / 9.7; hd 128, 17 / 24 / 64 rows 8.0 / 8.2 / 11.6 against 7.5 / 8.1 /
// 14.7; hd 256, 8 / 16 / 64 rows 11.2 / 11.7 / 19.1 against 10.6 / 12.2 / 26.5.
inline bool prefill_appends(int head_dim, int num_heads, int kv_mul, int cus, int start, int n) {
    if (n < 2 || (long)n * head_dim > 2560) return false;
    const PrefillTiling t = prefill_tiling(kv_mul);
    const PrefillKernel k = prefill_plan(head_dim, num_heads, kv_mul, cus, start, n);
    return t.hw == kv_mul && n <= 16 * t.qs &&
           (k == PrefillKernel::kFourHeads || k == PrefillKernel::kThreeHeads ||
            k == PrefillKernel::kTwoHeads || k == PrefillKernel::kOneHead);
}

}  // namespace slm
