// Causal prefill attention on bf16 matrix cores with f32 operands split in
// three (v_mfma_f32_16x16x32_bf16) for gfx950.
//
// Replaces the per-row loop of forward_batch_with_kv (transformer.rs:563-593),
// where row b at position p = start + b attends to cache rows 0..p.
//
// Precision.  An f32 value is the sum of three bf16 values x1 + x2 + x3 (each
// the rounded remainder of the ones before), so a product is nine bf16
// products, exact in f32; x2*y3, x3*y2 and x3*y3 (below 2^-25 of the product)
// are left out.  The other six are added to the accumulator one after another,
// small ones first: six roundings for 32 products, where
// v_mfma_f32_16x16x4_f32 has eight (error against 64 bits at 4096 rows 7.1e-7,
// in f32 8.6e-7).
//
// What bounds it: six bf16 products at 16 times the f32 MFMA rate.  A 16 x 32
// x 128 product takes 48 MFMAs of 16 cycles against 64 of 32 for f32; the VALU
// work (softmax, splitting K, V and P) overlaps MFMAs of another wave of the
// SIMD only in part, and at 4096 rows the matrix pipes are busy half the time.
//
// Tiling.  A workgroup holds HW query heads of one KV head, QS blocks of 16
// query rows and KSP key splits, a wave for each; with PAIR the blocks are i
// and n_blocks-1-i (every workgroup then has the same causal work), and the
// waves are numbered key split first, then head, then block, so a SIMD holds
// the same head and key split of the heavy and the light block.  Keys stream
// through LDS in tiles of 32 rows (split k attends tiles k, k + KSP, ...),
// split once per workgroup into three bf16 planes:
//   S^T = K . Q^T    A = K rows, B = Q^T (registers): lane (lr = l%16, g =
//                    l/16) ends with the scores of query lr against keys 16kk
//                    + 4g + r in register r of subtile kk;
//   O^T = V^T . P^T  A = V^T; B = P^T: lane group g supplies its own eight
//                    probabilities, keys 4g + (0..3) and 16 + 4g + (0..3), so
//                    they never move between lanes and V is stored with its
//                    keys in that order.
// Each wave's share of the next tiles goes from memory into its own LDS bytes
// by DMA, so no registers are held for it.  At hd 128 the planes and raw bytes
// take 128 KiB of LDS (160 with key splits), one workgroup and two waves per SIMD
// for a CU; at hd 64 half of that, two workgroups.
//
// Values that cannot be split.  inf, and finite values that round to a bf16 inf,
// make NaN when split, and the remainders of values below 2^-109 run out of
// bf16's exponents.  The splitting therefore keeps the largest magnitudes of q,
// K and V, and a wave computes its rows again in f32 from the cache
// (attend_f32, attend_plain) if a result is not finite, q or K reach 2^64, or
// the terms of an output sum are so small beside V's values that bits lost in P
// or V could show (least_sum).  Looking costs 1-2% (Llama-3-8B shape, per call:
// 4096 rows 677 -> 682 us, 777 rows at start 1000 96.1 -> 97.7), computing again
// several times the call.
#include <math.h>

#include "attn_common.h"
#include "prefill_plan.h"
#include "slm_internal.h"
#include "tile_range.h"

namespace slm {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct SplitParams {
    const float* q;
    const float* k_cache;
    const float* v_cache;
    const float* cos_t;
    const float* sin_t;
    float* out;
    int start;
    int n;
    int dim;
    int num_heads;
    int kv_dim;
    int kv_mul;
    int half;
    float scale_log2;
};

// The larger one, or NaN if either is (v_maximum3_f32 for two in turn).
__device__ __forceinline__ float maximum(float a, float b) {
    return __builtin_elementwise_maximum(a, b);
}

// ... over the wave.
__device__ __forceinline__ float wave_maximum(float x) {
    x = maximum(x, dpp<0x128>(x));
    x = maximum(x, dpp<0x124>(x));
    x = maximum(x, dpp<0x122>(x));
    x = maximum(x, dpp<0x121>(x));
    const uint32_t u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t w = __float_as_uint(maximum(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    return maximum(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ v4f mfma(bf8 a, bf8 b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Two values as bf16 pairs: x = p1 + p2 + p3 (24 bits).
__device__ __forceinline__ void split2(float x0, float x1, uint32_t* p1, uint32_t* p2,
                                       uint32_t* p3) {
    const auto pack = [](float a, float b) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf2));
    };
    *p1 = pack(x0, x1);
    x0 -= __uint_as_float(*p1 << 16);
    x1 -= __uint_as_float(*p1 & 0xFFFF0000u);
    *p2 = pack(x0, x1);
    x0 -= __uint_as_float(*p2 << 16);
    x1 -= __uint_as_float(*p2 & 0xFFFF0000u);
    *p3 = pack(x0, x1);
}

__device__ __forceinline__ void split8(const float (&x)[8], uint4 (&p)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) split2(x[2 * i], x[2 * i + 1], &w[0][i], &w[1][i], &w[2][i]);
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
}

template <int HD, int HW, int QS, int KSP, bool PAIR>
__global__ __launch_bounds__(64 * QS * HW * KSP, HD == 64 ? 4 : 2) void prefill_split_kernel(
    SplitParams p) {
    constexpr int NB = KSP == 1 ? 2 : 1;  // plane buffers
    constexpr int NWS = QS * HW;       // waves of one key split
    constexpr int NW = NWS * KSP;
    constexpr int NT = 64 * NW;
    constexpr int KT = 32;             // keys per tile
    constexpr int PL = KT * HD / 8;    // 16-byte chunks per plane of a K or V tile
    constexpr int KC = HD / 8;         // chunks per K row
    constexpr int NS = 2 * PL * KSP / NT;  // chunks a thread splits per step
    constexpr int NKS = HD / 32;       // k-steps of K . Q^T
    constexpr int NDT = HD / 16;       // 16-dim tiles of O^T
    static_assert(2 * PL * KSP % NT == 0 && PL % 64 == 0, "whole chunks, a wave's in one tile");
    static_assert(HD == 128 || HD == 64, "k_slot; a wave's V dims in one lane group");
    // K planes: row r's chunk c (dims 8c..8c+7) in slot c ^ 2(r & 7) (rows of
    // 256 bytes) or c ^ (r & 6) (of 128).  V
    // planes: dim d's chunk g (the keys lane group g supplies) in slot g ^
    // v_swz(d).  A 64-lane ds_read_b128 is served in four cycles of 16 lanes of
    // a half-wave that agree in the parity of lane bits 2-4 (bit 0 may also
    // count); with these slots the 16 lanes of the planes' reads and stores cover
    // the 64 banks once, either way.  What conflicts are left (11% of the LDS
    // cycles at 4096 rows) come with the raw K bytes, read 32 bytes apart.
    __shared__ __align__(16) struct {
        uint4 k[NB * KSP][3][PL];
        uint4 v[NB * KSP][3][PL];
        float raw[2 * KSP * PL * 8];  // f32 K and V of the next step's tiles
    } sm;
    auto k_slot = [](int r, int c) { return r * KC + (c ^ (HD == 128 ? (r & 7) << 1 : r & 6)); };
    auto v_swz = [](int d) { return ((d >> 4) & 1) | (((d >> 2) & 1) << 1); };

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15;
    const int lg = lane >> 4;
    const int kspl = wave % KSP;
    const int hw = wave / KSP % HW;
    const int qs = wave / (KSP * HW);

    // blockIdx.x = block pair * head groups + head group: consecutive
    // workgroups go round-robin to the 8 XCDs, so with 8 head groups each XCD's
    // L2 serves one KV head's K/V; longest causal ranges first.  With an odd
    // block count the middle pair's second block is its first, and its waves
    // hold no rows.
    const int n_qb = (p.n + 15) / 16;
    const int n_hg = p.num_heads / HW;
    const int hg = (int)blockIdx.x % n_hg;
    const int pi = (int)blockIdx.x / n_hg;
    const int g = (hg * HW) / p.kv_mul;
    const int head = hg * HW + hw;
    int q0, last;  // first query row of this wave; the workgroup's rows end at last
    if constexpr (PAIR) {
        const int pj = pi * (QS / 2) + qs % (QS / 2);  // this wave's pair
        const int heavy = n_qb - 1 - pj;
        q0 = qs < QS / 2 ? (heavy >= pj ? heavy * 16 : p.n) : (pj < heavy ? pj * 16 : p.n);
        last = min(p.n, (n_qb - pi * (QS / 2)) * 16);
    } else {
        const int qb = (n_qb + QS - 1) / QS - 1 - pi;
        q0 = (qb * QS + qs) * 16;
        last = min(p.n, (qb + 1) * QS * 16);
    }
    const int kv_len = p.start + last;
    const int n_tiles = (kv_len + KT - 1) / KT;
    const int wave_rows = max(0, min(16, p.n - q0));
    const int wave_last_pos = p.start + q0 + wave_rows - 1;
    const int row = q0 + lr;
    const bool row_ok = row < p.n;

    // dims 32 ks + 8 lg .. +7 of this lane's query, rotated and scaled
    auto load_q8 = [&](int ks, float (&x)[8]) __attribute__((always_inline)) {
        const long r = row_ok ? row : 0;
        const float* src = p.q + r * p.dim + head * HD + 32 * ks + 8 * lg;
        float4 a = ld4(src), b = ld4(src + 4);
        if (p.cos_t) {
            const long tr = (p.start + r) * (long)p.half + 16 * ks + 4 * lg;
            const float4 c = ld4(p.cos_t + tr), s = ld4(p.sin_t + tr);
            a = rope4_exact(a, make_float2(c.x, c.y), make_float2(s.x, s.y));
            b = rope4_exact(b, make_float2(c.z, c.w), make_float2(s.z, s.w));
        }
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = row_ok ? v[i] * p.scale_log2 : 0.0f;
    };

    const float* kg = p.k_cache + g * HD;
    const float* vg = p.v_cache + g * HD;
    static_assert(tile_range_fits(KT, kMaxKvDim), "tile ranges must fit 32 bits");

    // Shares.  A step's chunks are those of the KSP K tiles, then those of the
    // V tiles; chunk i*NT + tid is this thread's, so a wave's 64 chunks lie in
    // one tile.  Within it chunk f holds K row f / KC, dims 8 (f % KC) .., or
    // V dim f % HD, lane group f / HD.  The wave's chunks arrive as two pieces
    // of 64 16-byte loads (V piece h: keys 16h + 4g + (0..3) of the wave's 64
    // dims), in raw bytes that only this wave reads back.
    // (a step's tiles are whole multiples of the threads, or one tile is half)
    auto share_v = [&](int i) {
        return NT <= PL ? i * NT >= PL * KSP : i * NT + wave * 64 >= PL * KSP;
    };
    auto share_slot = [&](int i) {
        return NT <= PL ? i * NT / PL % KSP : (i * NT + wave * 64) / PL % KSP;
    };
    auto share_first = [&](int i) { return (i * NT + wave * 64) % PL; };  // within the tile
    int off[NS][2];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        const int fw = share_first(i);
        const bool is_v = share_v(i);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = fw * 2 + h * 64 + lane;  // float4 of the tile
            const int key = 16 * h + 4 * (fw / HD) + (lane >> 4);
            off[i][h] = is_v ? (key * p.kv_dim + fw % HD + 4 * (lane & 15)) * 4
                             : ((e / (HD / 4)) * p.kv_dim + (e % (HD / 4)) * 4) * 4;
        }
    }
    // tiles kt0 .. kt0 + KSP - 1; those past the last read as zeros
    auto dma = [&](int kt0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int u = i * NT + wave * 64;  // uniform
            const int kb = min(kt0 + share_slot(i), n_tiles) * KT;
            const int bytes = kb < kv_len ? (int)tile_range_bytes(kv_len, kb, KT, p.kv_dim) : 0;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>((share_v(i) ? vg : kg) + (long)kb * p.kv_dim), 0, bytes,
                0x00020000);
            // inline assembly: the compiler must not make LDS reads of the
            // planes wait for it; the wave waits (vmcnt) before it reads its
            // share back.  M0 holds the wave's LDS destination; lane l's 16
            // bytes land at M0 + 16*l.  The load must not issue in the cycle
            // after the scalar write of M0 (one wait state, which the compiler
            // does not put in ahead of inline assembly).
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const unsigned dst = (unsigned)(unsigned long)(
                    __attribute__((address_space(3))) float*)&sm.raw[u * 8 + h * 256];
                asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off[i][h]),
                             "s"(r), "{m0}"(dst) : "memory");
            }
        }
    };
    // Largest magnitudes of the K values and of the V values that this thread
    // splits; the V values are all of dim tid % HD.
    float top_k = 0.0f, top_v = 0.0f;
    static_assert(NT % HD == 0 && PL % HD == 0, "a thread's V chunks share their dim");
    auto top8 = [](float t, const float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) t = maximum(maximum(t, fabsf(x[j])), fabsf(x[j + 1]));
        asm volatile("" : "+v"(t));  // here, not after the loop's other shares: registers
        return t;
    };
    // Splits this wave's share into the planes of buffer buf.
    auto stage = [&](int buf) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int u = i * NT + wave * 64;
            const int slot = buf * KSP + share_slot(i), f = share_first(i) + lane;
            float x[8];
            uint4 pl[3];
            if (!share_v(i)) {  // uniform
                const float4 a = ld4(&sm.raw[(u + lane) * 8]), b = ld4(&sm.raw[(u + lane) * 8 + 4]);
                x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w;
                x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
                top_k = top8(top_k, x);
                split8(x, pl);
#pragma unroll
                for (int k = 0; k < 3; ++k) sm.k[slot][k][k_slot(f / KC, f % KC)] = pl[k];
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = sm.raw[u * 8 + j * 64 + lane];
                top_v = top8(top_v, x);
                split8(x, pl);
                const int d = f % HD;
#pragma unroll
                for (int k = 0; k < 3; ++k) sm.v[slot][k][d * 4 + (f / HD ^ v_swz(d))] = pl[k];
            }
        }
        // the raw bytes are read (and the planes written) before the next DMA
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };

    dma(0);
    bf8 qf[3][NKS];  // Q^T fragments, three planes
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        float x[8];
        uint4 pl[3];
        load_q8(ks, x);
        top_k = top8(top_k, x);
        split8(x, pl);
#pragma unroll
        for (int k = 0; k < 3; ++k) qf[k][ks] = __builtin_bit_cast(bf8, pl[k]);
    }

    // Softmax state (log2 domain): m, the running max (-inf before the first
    // key); om, the offset the score accumulators start from (negm holds -om:
    // the K . Q^T MFMAs then return s - om, and exp2 takes them as they are);
    // lim, how far a tile's max may exceed om before the state is rescaled
    // (-inf before the first tile, which therefore always rescales).
    v4f o[NDT], negm;
    float m, l, om, lim;
    auto reset = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NDT; ++i) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
        negm = v4f{0.f, 0.f, 0.f, 0.f};
        m = -INFINITY;
        l = 0.0f;
        om = 0.0f;
        lim = -INFINITY;
    };
    reset();

    // Causal mask and online softmax of one tile: scores (less om) in,
    // probabilities out.
    auto softmax = [&](int kb, v4f (&s)[2]) __attribute__((always_inline)) {
        if (kb + KT - 1 > p.start + q0) {  // uniform: some key may be masked
            const int last_key = p.start + q0 + lr - kb - 4 * lg;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * kk + r > last_key) s[kk][r] = -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int j = 1; j < 8; ++j) mx = fmaxf(mx, s[j >> 2][j & 3]);
        mx = rows_max(mx);
        if (__any(mx > lim)) {  // wave-uniform
            // without key splits the first tile holds key 0 <= qpos; with them
            // it may mask every key of a query, whose state then stays empty
            const float mn = fmaxf(m, mx + om);
            const bool none = KSP > 1 && mn == -INFINITY;
            const float alpha = none ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            l *= alpha;
#pragma unroll
            for (int i = 0; i < NDT; ++i) o[i] *= alpha;
            const float d = none ? 0.0f : mn - om;
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j >> 2][j & 3] -= d;
            m = mn;
            if (!none) {
                om = mn;
                lim = kLazyRescale;
                negm = v4f{-mn, -mn, -mn, -mn};
            }
        }
        float ps = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float e = __builtin_amdgcn_exp2f(s[j >> 2][j & 3]);
            s[j >> 2][j & 3] = e;
            ps = j == 0 ? e : ps + e;
        }
        l += ps;
    };

    // A tile from its planes.  The fragments come in groups of six, 12 MFMAs
    // each; a group is read while the one before it is in use (two waves per
    // SIMD do not cover the LDS latency by themselves).
    auto attend = [&](int kb, int slot) __attribute__((always_inline)) {
        constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
        bf8 f[2][2][3];
        auto load_k = [&](int ks, bf8 (&d)[2][3]) __attribute__((always_inline)) {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    d[kk][k] = __builtin_bit_cast(
                        bf8, sm.k[slot][k][k_slot(16 * kk + lr, 4 * ks + lg)]);
        };
        auto load_v = [&](int dt, bf8 (&d)[2][3]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int dim = 16 * (dt + i) + lr;
                    d[i][k] =
                        __builtin_bit_cast(bf8, sm.v[slot][k][dim * 4 + (lg ^ v_swz(dim))]);
                }
        };
        auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 6; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // two MFMAs
            }
        };
        v4f s[2] = {negm, negm};
        load_k(0, f[0]);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const bf8(&c)[2][3] = f[ks & 1];
            if (ks + 1 < NKS)
                load_k(ks + 1, f[(ks + 1) & 1]);
            else
                load_v(0, f[(ks + 1) & 1]);
#pragma unroll
            for (int e = 0; e < 6; ++e)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) s[kk] = mfma(c[kk][A[e]], qf[B[e]][ks], s[kk]);
            interleave();
        }
        softmax(kb, s);
        bf8 pf[3];
        {
            const float x[8] = {s[0][0], s[0][1], s[0][2], s[0][3],
                                s[1][0], s[1][1], s[1][2], s[1][3]};
            uint4 pl[3];
            split8(x, pl);
#pragma unroll
            for (int k = 0; k < 3; ++k) pf[k] = __builtin_bit_cast(bf8, pl[k]);
        }
#pragma unroll
        for (int dt = 0; dt < NDT; dt += 2) {
            const bf8(&c)[2][3] = f[(NKS + dt / 2) & 1];
            if (dt + 2 < NDT) load_v(dt + 2, f[(NKS + dt / 2 + 1) & 1]);
#pragma unroll
            for (int e = 0; e < 6; ++e)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    o[dt + i] = mfma(c[i][A[e]], pf[B[e]], o[dt + i]);
            interleave();
        }
    };

    const int n_steps = (n_tiles + KSP - 1) / KSP;
    if constexpr (NB == 1) {
        for (int st = 0; st < n_steps; ++st) {
            stage(0);
            if (st + 1 < n_steps) dma((st + 1) * KSP);
            __syncthreads();  // the planes are whole
            const int kb = (st * KSP + kspl) * KT;
            if (wave_rows > 0 && kb <= wave_last_pos) attend(kb, kspl);  // wave-uniform
            __syncthreads();  // every wave is done with them
        }
    } else {
        // Half of the waves split the next tile before they attend this one,
        // the others afterwards, so that splitting runs beside MFMAs: waves w and
        // w + 4 share a SIMD, one of each with four heads per workgroup (with
        // two or one both are alike).
        auto next = [&](int st, int buf) __attribute__((always_inline)) {
            if (st + 1 >= n_steps) return;
            stage(buf ^ 1);
            if (st + 2 < n_steps) dma(st + 2);
        };
        stage(0);
        if (n_steps > 1) dma(1);
        for (int st = 0; st < n_steps; ++st) {
            // the planes of tile st are whole, and every wave is done with the
            // other buffer
            __syncthreads();
            const int buf = st & 1;
            if (qs & 1) next(st, buf);
            const int kb = st * KT;
            if (wave_rows > 0 && kb <= wave_last_pos) attend(kb, buf);  // wave-uniform
            if (!(qs & 1)) next(st, buf);
        }
    }

    // For the check of the results below: every thread's top_v and each wave's
    // largest of both, in raw bytes of the wave's own (it has read them back).
    constexpr int kWaveRaw = 512;  // floats of a wave's chunks of share 0
    {
        float* t = &sm.raw[wave * kWaveRaw];
        t[lane] = top_v;
        t[64] = wave_maximum(top_k);  // the same in every lane
        t[65] = wave_maximum(top_v);
    }
    if constexpr (KSP == 1) __syncthreads();

    if constexpr (KSP > 1) {
        // Merge of the key splits: splits 1..KSP-1 hand each lane's O
        // registers, max and sum partial to split 0 through LDS (lane
        // contiguous), which folds them in split order.
        constexpr int NR = NDT * 4 + 2;  // floats per lane
        static_assert((KSP - 1) * NWS * 64 * NR * 4 <= (int)sizeof(sm.k), "clear of raw");
        float* s_merge = reinterpret_cast<float*>(&sm);
        const int ws = qs * HW + hw;
        if (kspl > 0) {
            float* dst = s_merge + ((kspl - 1) * NWS + ws) * NR * 64 + lane;
#pragma unroll
            for (int i = 0; i < NDT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[64 * (4 * i + r)] = o[i][r];
            dst[64 * (NR - 2)] = m;
            dst[64 * (NR - 1)] = l;
        }
        __syncthreads();
        if (kspl > 0) return;  // no barrier follows
        float mk[KSP];
        float mx = m;
#pragma unroll
        for (int k = 1; k < KSP; ++k) {
            mk[k] = s_merge[((k - 1) * NWS + ws) * NR * 64 + lane + 64 * (NR - 2)];
            mx = fmaxf(mx, mk[k]);
        }
        om = mx;  // the sums' common offset
        const float s0 = __builtin_amdgcn_exp2f(m - mx);
        l *= s0;
#pragma unroll
        for (int i = 0; i < NDT; ++i) o[i] *= s0;
#pragma unroll
        for (int k = 1; k < KSP; ++k) {
            const float* src = s_merge + ((k - 1) * NWS + ws) * NR * 64 + lane;
            const float sk = __builtin_amdgcn_exp2f(mk[k] - mx);
            l += src[64 * (NR - 1)] * sk;
#pragma unroll
            for (int i = 0; i < NDT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[i][r] += src[64 * (4 * i + r)] * sk;
        }
    }

    if (wave_rows == 0) return;
    // normalise and store: lane holds out[row][16 dt + 4 lg + (0..3)]
    auto store = [&]() __attribute__((always_inline)) {
        const float inv = 1.0f / rows_sum(l);
        if (!row_ok) return;
        float* dst = p.out + (long)row * p.dim + head * HD + 4 * lg;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
            *reinterpret_cast<float4*>(dst + 16 * dt) =
                make_float4(o[dt][0] * inv, o[dt][1] * inv, o[dt][2] * inv, o[dt][3] * inv);
    };
    store();

    // Whether the planes held enough of the operands (bf16's exponents end at
    // 2^-126, and planes below that may count as zero): with kv_len keys,
    // probabilities up to 2^kLazyRescale and values up to top, an output sum is
    // off by less than kv_len * (top + 2^kLazyRescale) * 2^-122, which is below
    // the roundings of a sum whose terms' magnitudes add up to least_sum(top);
    // a score of operands below 2^64 by less than 2^-50.
    auto least_sum = [&](float top) {
        return (float)kv_len * fmaf(top, 0x1p-96f, 0x1p-96f * (1 << (int)kLazyRescale));
    };
    float z = l * 0.0f;  // NaN once any of the row's values is not finite
    float least = INFINITY;
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            z = fmaf(o[i][r], 0.0f, z);
            least = fminf(least, fabsf(o[i][r]));
        }
    top_k = top_v = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        top_k = maximum(top_k, sm.raw[w * kWaveRaw + 64]);
        top_v = maximum(top_v, sm.raw[w * kWaveRaw + 65]);
    }
    bool again = row_ok && (z != z || !(top_k < 0x1p64f));
    const bool low = row_ok && !(least >= least_sum(top_v));
    if (!__any(again || low)) return;

    int g8 = lg;
    asm volatile("" : "+v"(g8));  // made here, not held through the loop above: registers
    g8 *= 8;
    // A tile in f32 from the cache rows, on f32 matrix instructions where every
    // query of the wave sees all its keys (step j of a product takes one dim or
    // key from each lane group) ...
    auto attend_f32 = [&](int kb, const float (&x)[NKS][8], bool abs_v)
                          __attribute__((always_inline)) {
        v4f s[2] = {negm, negm};
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                const long r = min(kb + 16 * kk + lr, kv_len - 1);
                const float* src = kg + r * p.kv_dim + 32 * ks + g8;
                const float4 a = ld4(src), b = ld4(src + 4);
                const float y[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    s[kk] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i], x[ks][i], s[kk], 0, 0, 0);
            }
        softmax(kb, s);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const long r = min(kb + 4 * lg + 16 * (j >> 2) + (j & 3), kv_len - 1);
            const float* src = vg + r * p.kv_dim + lr;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const float v = src[16 * dt];
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(abs_v ? fabsf(v) : v,
                                                            s[j >> 2][j & 3], o[dt], 0, 0, 0);
            }
        }
    };
    // ... and a key at a time on the diagonal: masked keys take no part in the sums.
    auto attend_plain = [&](int kb, const float (&x)[NKS][8]) __attribute__((always_inline)) {
        v4f s[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) s[kk] = v4f{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll 1
        for (int k = 0; k < KT && kb + k < kv_len; ++k) {
            const float* kr = kg + (long)(kb + k) * p.kv_dim + g8;
            float d = 0.0f;
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const float4 a = ld4(kr + 32 * ks), b = ld4(kr + 32 * ks + 4);
                const float y[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) d = fmaf(x[ks][i], y[i], d);
            }
            d += __shfl_xor(d, 16);
            d += __shfl_xor(d, 32);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (16 * (j >> 2) + 4 * lg + (j & 3) == k) s[j >> 2][j & 3] = d - om;
        }
        softmax(kb, s);
#pragma unroll 1
        for (int k = 0; k < KT && kb + k < kv_len; ++k) {
            float pk = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (16 * (j >> 2) + 4 * lg + (j & 3) == k) pk = s[j >> 2][j & 3];
            pk = __shfl(pk, lr + 16 * ((k >> 2) & 3));
            const bool on = kb + k <= p.start + row;
            const float* vr = vg + (long)(kb + k) * p.kv_dim + 4 * lg;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const float4 v = ld4(vr + 16 * dt);
                const float w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (on) o[dt][r] = fmaf(w[r], pk, o[dt][r]);
            }
        }
    };
    float x[NKS][8];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) load_q8(ks, x[ks]);
    if (!__any(again)) {
        // Small sums are mostly zeros of dims without values, or sums that
        // cancelled out (one in 10^7 does, to exactly zero).  The first tile's
        // terms usually reach least_sum.
        uint32_t small = 0;  // which of this lane's sums
        auto by_dim = [&](auto at_each) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NDT; ++i) {
                float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // largest value of dims 16 i + 4 lg + ..
#pragma unroll 1
                for (int j = 0; j < NT / HD; ++j) {
                    const int at = j * HD + 16 * i + 4 * lg;
                    const float4 y = ld4(&sm.raw[(at >> 6) * kWaveRaw + (at & 63)]);
                    t[0] = maximum(t[0], y.x), t[1] = maximum(t[1], y.y);
                    t[2] = maximum(t[2], y.z), t[3] = maximum(t[3], y.w);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) at_each(i, r, t[r]);
            }
        };
        by_dim([&](int i, int r, float top) {
            if (low && top != 0.0f && !(fabsf(o[i][r]) >= least_sum(top))) small |= 1u << (4 * i + r);
        });
        if (!__any(small)) return;
        const float offset = om;
        reset();
        om = offset;
        negm = v4f{-om, -om, -om, -om};
        lim = INFINITY;  // om stays
        attend_f32(0, x, true);
        by_dim([&](int i, int r, float top) {
            if (small >> (4 * i + r) & 1) again |= !(o[i][r] >= least_sum(top));
        });
        if (!__any(again)) return;
    }

    reset();
    int kb = 0;
#pragma unroll 1
    for (; kb + KT - 1 <= p.start + q0; kb += KT) attend_f32(kb, x, false);
#pragma unroll 1
    for (; kb <= wave_last_pos; kb += KT) attend_plain(kb, x);
    store();
}

template <int HD, int HW, int QS, int KSP, bool PAIR>
hipError_t launch_t(const Shape& s, const SplitParams& pp, hipStream_t st) {
    const int groups = ((pp.n + 15) / 16 + QS - 1) / QS;
    hipLaunchKernelGGL((prefill_split_kernel<HD, HW, QS, KSP, PAIR>),
                       dim3(groups * (s.num_heads / HW)), dim3(64 * QS * HW * KSP), 0, st, pp);
    return hipGetLastError();
}

template <int HD, int HW>
hipError_t launch_hw(const Shape& s, const SplitParams& pp, PrefillKernel form, hipStream_t st) {
    switch (form) {
        case PrefillKernel::kSplitKeys: return launch_t<HD, HW, 4 / HW, 2, true>(s, pp, st);
        case PrefillKernel::kSplitPaired: return launch_t<HD, HW, 8 / HW, 1, true>(s, pp, st);
        case PrefillKernel::kSplitConsecutive: return launch_t<HD, HW, 8 / HW, 1, false>(s, pp, st);
        default: return hipErrorInvalidValue;
    }
}

template <int HD>
hipError_t launch_hd(const Shape& s, const SplitParams& pp, PrefillKernel form, hipStream_t st) {
    // four heads on the tiles where there are so many: 4096 rows of the
    // Llama-3-8B shape 672 against 690 us with two
    if (form == PrefillKernel::kSplitConsecutive && s.kv_mul % 4 == 0)
        return launch_t<HD, 4, 2, 1, false>(s, pp, st);
    return s.kv_mul % 2 == 0 ? launch_hw<HD, 2>(s, pp, form, st)
                             : launch_hw<HD, 1>(s, pp, form, st);
}

}  // namespace

hipError_t launch_prefill_split(const Shape& s, const PrefillArgs& a, PrefillKernel form,
                                hipStream_t st) {
    SplitParams pp{a.q,   a.k_cache, a.v_cache,   a.cos_t,  a.sin_t,  a.out, a.start,
                   a.n,   s.dim,     s.num_heads, s.kv_dim, s.kv_mul, s.half,
                   1.4426950408889634f / sqrtf((float)s.head_dim)};
    switch (s.head_dim) {
        case 64: return launch_hd<64>(s, pp, form, st);
        case 128: return launch_hd<128>(s, pp, form, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace slm
