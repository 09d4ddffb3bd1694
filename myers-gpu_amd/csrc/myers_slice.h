// Candidate-sliced verification of reads of up to 1024 bases.
//
// The bit-vector kernels (myers_device.h) hold 32 rows of one candidate in a
// word; their update needs an add with carry and two funnel shifts per word,
// and gfx950 issues those at half the rate of plain bit operations.  Here a
// word holds one row of 32 candidates.  The rows of a column are then updated
// one after the other with the deltas of the single cell (the block recurrence
// of src/myers-4bits.c:115-134 at a width of one bit), which is seven bit
// operations per 32 cells, all of them double rate: the match bit against the
// text (two v_bitop3: x = (r0 ^ t0) | tN, ne = x | (r1 ^ t1), reads and text as
// bit planes of their 2-bit codes, tN marking text N), D0 = ~ne | Mv | hm, and
// the four output deltas.  The word update of the bit-vector form costs 10
// operations, 6.5 slots of the single rate against 3.5 here.
//
//   * SL lanes of the wave share a group of 32 candidates; lane b of a group
//     holds R = W * 32 / SL consecutive rows (W = ceil(m / 32), the same for
//     the whole chunk) as four words per row, Pv, Mv and the two planes of the
//     read, in registers.  Lanes run diagonally (lane b computes column t - b at
//     step t) and pass their top row's horizontal delta on by one DPP shift.
//   * A group's candidates may differ in length: the p = 32 W - m rows missing
//     to R * SL are taken out one or a few per lane (row 0 .. K-1 of a lane
//     passes the deltas through for the candidates of its mask), so the last
//     row of the last lane is row m of every candidate.
//   * Text comes from bit planes of the reference (three words per 32 bases,
//     built once when it is loaded).  Every 32 steps each candidate's next 32
//     columns are transposed (32 x 32 bits, five ds_swizzle stages) into one
//     word per column and plane, which the lanes read from LDS.
//   * The last row's deltas go to LDS step by step and come back transposed,
//     32 columns per candidate, for the running score and its first minimum.
//   * A chunk with an N in a read takes the read's N plane from LDS as well
//     (eight operations).  A chunk with a Peq that is not one code per base,
//     or with reads of different W (a bin table forced by the caller), runs
//     the bit-vector kernel.
#ifndef MYERS_SLICE_H
#define MYERS_SLICE_H

#include "myers_device.h"

namespace {

// Truth tables of the match: a | (b ^ c), and ~a | b | c.
constexpr uint32_t kOrXor = 0xF0u | (0xCCu ^ 0xAAu);
constexpr uint32_t kNotOrOr = (~0xF0u & 0xFFu) | 0xCCu | 0xAAu;
constexpr uint32_t kSelect = 0xCAu;                    // a ? b : c

template <int SL>
struct SliceShape {
    static constexpr int kGroups = 64 / SL;             // groups of 32 candidates per wave
    static constexpr int kCands = 32 * kGroups;         // candidates per chunk
    static constexpr int kBatches = kCands / 64;        // candidates per lane where a lane takes a candidate
    static constexpr int kCols = SL + 32;               // text columns held per group: this block's 32, SL before it
    // LDS of a chunk, in 16-byte units: each group's first read, the
    // candidates (kCandWords words each), the text columns (first the table of
    // the chunk's reads), the score row's deltas and the reads' N plane (first
    // the reads' Peq, staged).
    static constexpr int kFirstU4 = (kGroups + 4) / 4;
    // block, window, length (~0: skipped), then index and, where the rows leave
    // no registers for it, the running state
    static constexpr bool cold(int r) { return 4 * r + 4 * kBatches > 108; }
    static constexpr int kCandWords = SL >= 32 ? 7 : 4;
    static constexpr int kCandU4 = kCands * kCandWords / 4;
    static constexpr int kTextU4 = kFirstU4 + kCandU4;  // the text columns start here
    static constexpr int kOutU4 = kTextU4 + kGroups * kCols;           // deltas: uint2 per column and group, then spare ones
    static constexpr int kPlaneU4 = kOutU4 + kGroups * 16 + 4;
    // a fifth word per row, the reads' N, fits the registers up to 26 rows
    static constexpr bool rows_n(int r) { return 5 * r + 4 * kBatches <= 134; }
    // (the least part is for staging: eight reads of R SL bases)
    static constexpr int ws_u4(int r) { return kPlaneU4 + (rows_n(r) ? r * SL / 4 : ((r + 1) / 2) * 32); }
    // rows that a lane can lack: R SL - m < 32 - SL where R is odd (the reads of
    // fewer rows are those of R - 1), else < 32
    static constexpr int skip_rows(int r) { return SL >= 32 || (r & 1) ? 1 : 2; }
    static_assert(kCands <= kGroups * kCols, "the table of reads fits the text columns");
};

// Longest reads (in words) of each form: at most 32 rows per lane, or 24 where
// a lane also keeps the state of two candidates.
constexpr int slice_max_words(int sl) { return sl >= 32 ? 32 : 12; }

// LDS hand-over between the lanes of one wave: its accesses execute in order,
// so only the compiler has to keep them so.
__device__ __forceinline__ void slice_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Transpose the 32 x 32 bits held by each half of the wave (lane j's bit c
// goes to lane c's bit j): stage d swaps the off-diagonal d x d blocks with
// lane j ^ d.
template <int D>
__device__ __forceinline__ uint32_t transpose_stage(uint32_t x, uint32_t lane) {
    constexpr uint32_t kLow = D == 16 ? 0x0000FFFFu : D == 8 ? 0x00FF00FFu : D == 4 ? 0x0F0F0F0Fu
                              : D == 2 ? 0x33333333u : 0x55555555u;
    const uint32_t y = (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (D << 10) | 0x1F);
    const bool up = (lane & (uint32_t)D) != 0u;
    const uint32_t rot = __builtin_amdgcn_alignbit(y, y, up ? (uint32_t)D : 32u - (uint32_t)D);
    return __builtin_amdgcn_bitop3_b32(up ? kLow : ~kLow, rot, x, kSelect);
}
__device__ __forceinline__ uint32_t transpose32(uint32_t x, uint32_t lane) {
    x = transpose_stage<16>(x, lane);
    x = transpose_stage<8>(x, lane);
    x = transpose_stage<4>(x, lane);
    x = transpose_stage<2>(x, lane);
    return transpose_stage<1>(x, lane);
}

// One step of one lane: its R rows of one column.  t = text planes of the
// column (x, y the code's bits, z N); hp / hm the horizontal delta entering
// row 0 and, on return, leaving row R-1.  Each operation is fixed in place:
// the next row's match bits between the dependent operations of this row keep
// the double-rate issue going (245 TCUPS against 236 with a row's operations
// in their natural order, 204-190 with two or more rows interleaved; 32 rows,
// three waves per SIMD, the loop alone).
// N: how reads with N take part: not at all (kPlain: none in the chunk), or
// with their rows' N plane in rn (kRowsN) or, where registers do not hold it,
// in LDS at np (kPlaneN).
enum SliceN { kPlain = 0, kRowsN = 1, kPlaneN = 2 };
#define SLICE_FIX __builtin_amdgcn_sched_barrier(0)
template <int R, int K, int kN>
__device__ __forceinline__ void slice_step(uint32_t (&Pv)[R], uint32_t (&Mv)[R], const uint32_t (&r0)[R],
                                           const uint32_t (&r1)[R], const uint32_t (&rn)[kN == kRowsN ? R : 1],
                                           const uint32_t (&skip)[K], const uint4 &t, const uint2 *np, uint32_t &hp,
                                           uint32_t &hm) {
    uint2 n0 = make_uint2(0u, 0u), n1 = n0, n2 = n0;    // N plane of this pair of rows and the next two pairs
    if constexpr (kN == kPlaneN) {
        n0 = np[0];
        if constexpr (R > 2) n1 = np[64];
    }
    uint32_t x = kN != kPlain ? r0[0] ^ t.x : __builtin_amdgcn_bitop3_b32(r0[0], t.x, t.z, kXorOr);
    uint32_t ne = __builtin_amdgcn_bitop3_b32(x, r1[0], t.y, kOrXor);
    if constexpr (kN != kPlain) ne = __builtin_amdgcn_bitop3_b32(ne, kN == kRowsN ? rn[0] : n0.x, t.z, kOrXor);
    SLICE_FIX;
#pragma unroll
    for (int i = 0; i < R; i++) {
        uint32_t ne_next = 0;
        if constexpr (kN == kPlaneN) {
            if (i % 2 == 0 && i + 4 < R) n2 = np[(i / 2 + 2) * 64];
        }
        const uint32_t n_next = kN == kRowsN ? rn[kN == kRowsN && i + 1 < R ? i + 1 : 0] : i % 2 == 0 ? n0.y : n1.x;   // row i + 1's
        const uint32_t d0 = __builtin_amdgcn_bitop3_b32(ne, Mv[i], hm, kNotOrOr);
        SLICE_FIX;
        if (i + 1 < R) {
            const uint32_t r = r0[i + 1 < R ? i + 1 : i];
            x = kN != kPlain ? r ^ t.x : __builtin_amdgcn_bitop3_b32(r, t.x, t.z, kXorOr);
        }
        SLICE_FIX;
        uint32_t hm_out = Pv[i] & d0;
        SLICE_FIX;
        uint32_t hp_out = __builtin_amdgcn_bitop3_b32(Mv[i], d0, Pv[i], kOrNor);
        SLICE_FIX;
        if (i + 1 < R) ne_next = __builtin_amdgcn_bitop3_b32(x, r1[i + 1 < R ? i + 1 : i], t.y, kOrXor);
        SLICE_FIX;
        Pv[i] = __builtin_amdgcn_bitop3_b32(hm, d0, hp, kOrNor);
        SLICE_FIX;
        Mv[i] = hp & d0;
        SLICE_FIX;
        if constexpr (kN != kPlain) {
            if (i + 1 < R) ne_next = __builtin_amdgcn_bitop3_b32(ne_next, n_next, t.z, kOrXor);
            SLICE_FIX;
        }
        if (i < K) {
            hp_out = __builtin_amdgcn_bitop3_b32(skip[i < K ? i : 0], hp, hp_out, kSelect);
            hm_out = __builtin_amdgcn_bitop3_b32(skip[i < K ? i : 0], hm, hm_out, kSelect);
        }
        hp = hp_out;
        hm = hm_out;
        ne = ne_next;
        if (i % 2 == 1) {
            n0 = n1;
            n1 = n2;
        }
    }
}

// The horizontal delta of the lane below, 0 for the first lane of a group.
template <int SL>
__device__ __forceinline__ uint32_t slice_from_below(uint32_t v, uint32_t not_first) {
    if constexpr (SL > 16) {
        v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);   // wave_shr:1
    } else {
        v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);   // row_shr:1
    }
    if constexpr (SL != 16 && SL != 64) v &= not_first;
    return v;
}

// What a chunk needs of the batch, the same in every lane (as arguments of a
// function they come in vector registers: uniform() brings them back).
struct SliceBatch {
    const uint32_t *peq, *planes;
    uint2 *results;
    uint32_t last_block;
    float threshold;
    uint32_t nreads, max_cols;
    // first rows only: where the candidates kept go, and the counts (list == nullptr: all rows)
    uint32_t *list, *kept, *tally;
};
template <typename T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<T *>(((uint64_t)hi << 32) | lo);
}
using SliceLds = __attribute__((address_space(3))) uint4;

constexpr uint32_t kSliceMaxCols = 1u << 27;            // columns of a window (longer ones run the bit-vector kernel)

// The first minimum of 32 columns from col0 (src-api/coreMyersGPU-CC35.cu:
// 205-207,227-228).  hp / hm: bit j is the delta of column col0 + j, masked to
// the window; end: the score after them.  Eight columns at a time, the last
// ones first: on falling scores the least score is found early, and bytes
// that cannot reach it in any lane are passed over.
__device__ __forceinline__ void slice_first_min(uint32_t hp, uint32_t hm, int32_t end, uint32_t col0,
                                                int32_t &min_score, uint32_t &min_col) {
    int32_t low = min_score;
    uint32_t at = ~0u;                                  // the first of the columns seen that has `low`
#pragma unroll
    for (int q = 3; q >= 0; q--) {
        const uint32_t p8 = (hp >> (8 * q)) & 0xFFu, m8 = (hm >> (8 * q)) & 0xFFu;
        const int32_t falls = __builtin_popcount(m8), begin = end - (int32_t)__builtin_popcount(p8) + falls;
        // an equal score in an earlier column of the block replaces a later one
        const int32_t reach = low + (at != ~0u ? 1 : 0);
        if (__ballot(begin - falls < reach) != 0ull) {
            // key = 64 score + column: the least is the first minimum
            int32_t key = begin * 64 + 8 * q, least = 0x7FFFFFFF;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                key += (int32_t)(((p8 >> j) & 1u) << 6) - (int32_t)(((m8 >> j) & 1u) << 6);
                least = min(least, key + j);
            }
            const bool better = (least >> 6) < reach;
            low = better ? least >> 6 : low;
            at = better ? (uint32_t)least & 63u : at;
        }
        end = begin;
    }
    if (at != ~0u) min_col = col0 + at;
    min_score = low;
}

// Take in the deltas of 32 columns from col0.  The columns before them are
// searched for a new minimum only now, and only if some lane's may hold one:
// they cannot once a later score is below all of theirs, so the falling part
// of the score row is not searched at all.
__device__ __forceinline__ void slice_score(uint32_t hp, uint32_t hm, uint32_t col0, uint32_t &best,
                                            uint32_t &min_col, uint32_t &php, uint32_t &phm) {
    const int32_t score = (int32_t)(best & 0xFFFFu), end = score + (int32_t)__builtin_popcount(hp) - (int32_t)__builtin_popcount(hm);
    int32_t min_score = (int32_t)(best >> 16);
    const int32_t least = score - (int32_t)__builtin_popcount(php);      // no earlier score is less
    if (__ballot(least < min_score && least <= end) != 0ull)
        slice_first_min(php, phm, score, col0 - 32u, min_score, min_col);
    php = hp;
    phm = hm;
    best = (uint32_t)end | ((uint32_t)min_score << 16);
}

// The same where only a bound from below of the least score is asked for: of
// eight columns each, the score before them less their falls (which can be
// below zero where rises lie between them, a score cannot).
__device__ __forceinline__ void slice_bound(uint32_t hp, uint32_t hm, uint32_t &best) {
    int32_t score = (int32_t)(best & 0xFFFFu), low = (int32_t)(best >> 16);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int32_t falls = (int32_t)__builtin_popcount((hm >> (8 * q)) & 0xFFu);
        low = min(low, score - falls);
        score += (int32_t)__builtin_popcount((hp >> (8 * q)) & 0xFFu) - falls;
    }
    best = (uint32_t)score | ((uint32_t)max(low, 0) << 16);
}

// Planes of 32 bases of the reference.
__device__ __forceinline__ uint3 slice_planes(const uint32_t *__restrict__ planes, uint32_t block,
                                              uint32_t last_block) {
    return *reinterpret_cast<const uint3 *>(planes + (size_t)min(block, last_block) * 3u);
}

// The columns of a chunk whose read planes are in place (kN: SliceN).  A lane's
// candidates: number 64 k + lane of the chunk, i.e. candidate lane % 32 of group
// 2 k + lane / 32.
template <int SL, int R, int kN>
__device__ __forceinline__ void slice_columns(const SliceBatch &a, uint4 *lds, uint32_t lane, const uint32_t (&r0)[R],
                                              const uint32_t (&r1)[R], const uint32_t (&rn)[kN == kRowsN ? R : 1],
                                              const uint32_t (&skip)[SliceShape<SL>::skip_rows(R)]) {
    using S = SliceShape<SL>;
    constexpr int K = S::skip_rows(R), kB = S::kBatches;
    constexpr uint32_t kUnroll = R >= 16 ? 2u : 4u, kC = (uint32_t)S::kCands;
    constexpr bool kCold = S::cold(R);
    uint32_t *cand = reinterpret_cast<uint32_t *>(lds + S::kFirstU4);
    uint4 *text = lds + S::kTextU4;
    uint2 *out = reinterpret_cast<uint2 *>(lds + S::kOutU4);
    const uint2 *np = reinterpret_cast<const uint2 *>(lds + S::kPlaneU4) + lane;
    const uint32_t b = lane % (uint32_t)SL, group = lane / (uint32_t)SL;
    const uint32_t not_first = b != 0u ? ~0u : 0u;

    // before a lane's first column it reads text that matches no row: with no
    // match and no delta from below, Pv = ~0 and Mv = 0 stay as they are
    for (uint32_t i = lane; i < (uint32_t)(S::kGroups * SL); i += 64u)
        *reinterpret_cast<uint3 *>(text + (i / (uint32_t)SL) * (uint32_t)S::kCols + i % (uint32_t)SL) =
            make_uint3(~0u, 0u, ~0u);
    // score | first minimum << 16, its column, and the deltas of the 32 columns
    // not searched yet
    uint32_t best[kB], min_col[kB], php[kB], phm[kB];
#pragma unroll
    for (int k = 0; k < kB; k++) {
        uint32_t *cd = cand + 64u * (uint32_t)k + lane;
        uint32_t m = cd[2 * kC];
        if (a.list != nullptr && m != ~0u) m = (uint32_t)(R * SL);      // (the word is the threshold)
        best[k] = m == ~0u ? 0u : (m | (m << 16));
        min_col[k] = php[k] = phm[k] = 0u;
        if constexpr (kCold) {
            // the index moves to the unused word beside the candidate's text column
            text[((uint32_t)(2 * k) + (lane >> 5)) * (uint32_t)S::kCols + (uint32_t)SL + (lane & 31u)].w = cd[3 * kC];
            cd[3 * kC] = 0u;
            cd[4 * kC] = best[k];
            cd[5 * kC] = cd[6 * kC] = 0u;
        }
    }
    uint32_t Pv[R], Mv[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        Pv[i] = ~0u;
        Mv[i] = 0u;
    }
    // the text of the next block, requested a block ahead where registers allow
    constexpr bool kAhead = 4 * R + 10 * kB <= 84;
    uint3 cur[kB], nxt[kB];
    auto request = [&](int k, uint32_t blk) {
        cur[k] = slice_planes(a.planes, blk, a.last_block);
        nxt[k] = slice_planes(a.planes, blk + 1u, a.last_block);
    };
    if constexpr (kAhead) {
#pragma unroll
        for (int k = 0; k < kB; k++) request(k, cand[64 * k + (int)lane]);
    }
    uint32_t hp = 0, hm = 0;
    const uint4 *t_lane = text + group * (uint32_t)S::kCols + (uint32_t)SL - b;
    const uint32_t out_inc = b == (uint32_t)(SL - 1) ? 1u : 0u;
    const uint32_t nsteps = a.max_cols + (uint32_t)(SL - 1);

    uint32_t last0 = 0;                                 // first column of the last block
    for (uint32_t s0 = 0; s0 < nsteps; s0 += 32u) {
        // what follows from the lane's number is computed anew in every block:
        // held over the steps, it would take registers from the rows
        uint32_t l = lane;
        if constexpr (kCold) asm volatile("" : "+v"(l));
        // this block's text: columns s0 .. s0 + 31 of every candidate
        slice_sync();
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const uint32_t *cd = cand + 64u * (uint32_t)k + l;
            const uint32_t blk = cd[0] + (s0 >> 5), shift = cd[kC];         // (the low five bits)
            if constexpr (!kAhead) request(k, blk);
            uint3 w;
            w.x = transpose32(__builtin_amdgcn_alignbit(nxt[k].x, cur[k].x, shift), l);
            w.y = transpose32(__builtin_amdgcn_alignbit(nxt[k].y, cur[k].y, shift), l);
            w.z = transpose32(__builtin_amdgcn_alignbit(nxt[k].z, cur[k].z, shift), l);
            if constexpr (kAhead) request(k, blk + 1u);
            uint4 *tg = text + ((uint32_t)(2 * k) + (l >> 5)) * (uint32_t)S::kCols;
            const uint32_t col = l & 31u;
            if (s0 != 0u && col >= (uint32_t)(32 - SL))
                *reinterpret_cast<uint3 *>(tg + col - (uint32_t)(32 - SL)) = *reinterpret_cast<uint3 *>(tg + (uint32_t)SL + col);
            slice_sync();
            *reinterpret_cast<uint3 *>(tg + (uint32_t)SL + col) = w;
        }
        slice_sync();
        const uint32_t nj = min(32u, nsteps - s0);
        // the top lane writes the score row's deltas, the others to the spare slots
        uint32_t oi = out_inc ? (l / (uint32_t)SL) * 32u : (uint32_t)S::kGroups * 32u + (l & 7u);
        uint4 t = t_lane[0];
        for (uint32_t j = 0; j < nj; j += kUnroll) {
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) {
                // (the last step of a block reads one past its columns: not used)
                const uint4 t_next = t_lane[j + u + 1u];
                hp = slice_from_below<SL>(hp, not_first);
                hm = slice_from_below<SL>(hm, not_first);
                slice_step<R, K, kN>(Pv, Mv, r0, r1, rn, skip, t, np, hp, hm);
                out[oi] = make_uint2(hp, hm);
                oi += out_inc;
                t = t_next;
                SLICE_FIX;
            }
        }
        slice_sync();
        if constexpr (kCold) asm volatile("" : "+v"(l));
        // step s0 + j gave the score row's deltas of column s0 + j - (SL-1)
        const uint32_t col0 = s0 - (uint32_t)(SL - 1);              // wraps in the first block
        const uint32_t before = s0 < (uint32_t)(SL - 1) ? (uint32_t)(SL - 1) - s0 : 0u;   // steps without a column
        // a candidate's result may still change (not asked of the first rows only)
        bool open = a.threshold < 0.0f || a.list != nullptr;
#pragma unroll
        for (int k = 0; k < kB; k++) {
            const uint2 v = out[((uint32_t)(2 * k) + (l >> 5)) * 32u + (l & 31u)];
            uint32_t *cd = cand + 64u * (uint32_t)k + l;
            if constexpr (kCold) {
                min_col[k] = cd[3 * kC];
                best[k] = cd[4 * kC];
                php[k] = cd[5 * kC];
                phm[k] = cd[6 * kC];
            }
            const uint32_t seen = col0 + before, ncols = cd[kC] >> 5;
            const uint32_t left = ncols > seen ? ncols - seen : 0u;
            const uint32_t mask = (left >= 32u ? ~0u : (1u << left) - 1u) << before;
            const uint32_t vp = transpose32(v.x, l) & mask, vm = transpose32(v.y, l) & mask;
            if (a.list != nullptr) slice_bound(vp, vm, best[k]);
            else slice_score(vp, vm, col0, best[k], min_col[k], php[k], phm[k]);
            if (a.threshold >= 0.0f && a.list == nullptr) {
                // the score falls by one per column at most: it cannot get
                // under the threshold or the minimum so far any more where it
                // less the columns left is not below both
                const uint32_t m = cd[2 * kC], after = left > 32u - before ? left - (32u - before) : 0u;
                const uint32_t bound = min(threshold_of(m, a.threshold) + 1u, best[k] >> 16);
                open |= m != ~0u && (best[k] & 0xFFFFu) < bound + after;
            }
            if constexpr (kCold) {
                cd[3 * kC] = min_col[k];
                cd[4 * kC] = best[k];
                cd[5 * kC] = php[k];
                cd[6 * kC] = phm[k];
            }
        }
        last0 = col0;
        if (__ballot(open) == 0ull) break;
    }
    // the last columns, and the results
    uint32_t tried = 0, kept = 0;
#pragma unroll
    for (int k = 0; k < kB; k++) {
        const uint32_t *cd = cand + 64u * (uint32_t)k + lane;
        if constexpr (kCold) {
            min_col[k] = cd[3 * kC];
            best[k] = cd[4 * kC];
            php[k] = cd[5 * kC];
            phm[k] = cd[6 * kC];
        }
        const int32_t score = (int32_t)(best[k] & 0xFFFFu);
        int32_t min_score = (int32_t)(best[k] >> 16);
        if (__ballot(score - (int32_t)__builtin_popcount(php[k]) < min_score) != 0ull)
            slice_first_min(php[k], phm[k], score, last0, min_score, min_col[k]);
        const uint32_t m = cd[2 * kC];
        const uint32_t index =
            kCold ? text[((uint32_t)(2 * k) + (lane >> 5)) * (uint32_t)S::kCols + (uint32_t)SL + (lane & 31u)].w : cd[3 * kC];
        if (a.list != nullptr) {
            // the first rows' least score bounds the read's from below
            const bool keep = index != ~0u && m != ~0u && (uint32_t)min_score <= m;
            const uint64_t keeps = __ballot(keep);
            const uint32_t n = (uint32_t)__builtin_popcountll(keeps);
            uint32_t at = 0;
            if (lane == 0u && n != 0u) at = atomicAdd(a.kept, n);
            at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
            if (keep) a.list[at + (uint32_t)__builtin_popcountll(keeps & ((1ull << lane) - 1ull))] = index;
            else if (index != ~0u) a.results[index] = m == ~0u ? make_uint2(0u, kSkipScore) : make_uint2(kNoMatch, kNoMatch);
            tried += (uint32_t)__builtin_popcountll(__ballot(index != ~0u && m != ~0u));
            kept += n;
            continue;
        }
        if (index == ~0u) continue;                     // past the bin's last candidate
        uint2 r = make_uint2(0u, kSkipScore);
        if (m != ~0u) {
            r = make_uint2(min_col[k], (uint32_t)min_score);
            // threshold mode: score <= (uint32)((float)m * e) (src/checksum-2.c:88,104-105)
            if (a.threshold >= 0.0f && r.y > threshold_of(m, a.threshold)) r = make_uint2(kNoMatch, kNoMatch);
        }
        a.results[index] = r;
    }
    if (a.list != nullptr && lane == 0u) {
        atomicAdd(a.tally, tried);
        atomicAdd(a.tally + 1, kept);
    }
}

// A chunk whose live candidates' reads all have W words and at most R SL
// bases; tab: its `nreads` distinct reads in chunk order, {entry, m, live
// candidates of the group, 0}.
// False (nothing written) if a read's Peq is not one code per base.
//
// Not inlined: as a part of one large kernel, the register allocator spills
// the rows of one form for the sake of another.
template <int SL, int R>
__device__ __noinline__ bool slice_run(SliceBatch a, SliceLds *lds_at) {
    using S = SliceShape<SL>;
    constexpr int K = S::skip_rows(R), W = (R * SL + 31) / 32;
    static_assert(R >= K && R <= 32, "rows per lane");
    static_assert(!S::cold(R) || S::kCandWords == 7, "room for the running state");
    a.peq = uniform_ptr(a.peq);
    a.planes = uniform_ptr(a.planes);
    a.results = uniform_ptr(a.results);
    a.list = uniform_ptr(a.list);
    a.kept = uniform_ptr(a.kept);
    a.tally = uniform_ptr(a.tally);
    a.last_block = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.last_block);
    a.threshold = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(a.threshold)));
    a.max_cols = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.max_cols);
    const uint32_t nreads = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.nreads);
    const uint32_t lane = __lane_id();
    uint4 *lds = (uint4 *)lds_at;
    const uint32_t *first_read = reinterpret_cast<const uint32_t *>(lds);
    const uint4 *tab = lds + S::kTextU4;
    uint4 *stage = lds + S::kOutU4;
    constexpr uint32_t kPass = (uint32_t)(S::ws_u4(R) - S::kOutU4) / (uint32_t)W;      // reads staged at a time
    const uint32_t b = lane % (uint32_t)SL, group = lane / (uint32_t)SL;
    const uint32_t my_first = first_read[group], my_end = first_read[group + 1u];
    uint32_t bad = 0, any_n = 0;
    // Stage the Peq of up to kPass reads at a time and hand each read of this
    // lane's group to `body` with the three planes of the lane's rows.
    auto each_read = [&](auto body) {
        for (uint32_t f0 = 0; f0 < nreads; f0 += kPass) {
            // word j of read f0 + r: planes 0 and 1 of its codes, N; rows that
            // do not hold exactly one code are bad
            const uint32_t here = min(kPass, nreads - f0);
            slice_sync();
            for (uint32_t it = lane; it < here * (uint32_t)W; it += 64u) {
                const uint4 rd = tab[f0 + it / (uint32_t)W];
                const uint32_t j = it % (uint32_t)W;
                uint4 w = make_uint4(0u, 0u, 0u, 0u);
                if (rd.z != 0u && 32u * j < rd.y) {
                    const uint32_t *p = a.peq + (size_t)(rd.x + (j >> 2)) * 20u + (j & 3u);
                    const uint32_t pa = p[0], pc = p[4], pg = p[8], pt = p[12], pn = p[16];
                    const uint32_t rows = rd.y - 32u * j >= 32u ? ~0u : (1u << (rd.y & 31u)) - 1u;
                    const uint32_t seen = pa | pc | pg | pt | pn;
                    const uint32_t twice = (pa & pc) | ((pa | pc) & pg) | ((pa | pc | pg) & pt) |
                                           ((pa | pc | pg | pt) & pn);
                    w = make_uint4(pc | pt, pg | pt, pn, 0u);
                    bad |= (twice | ~seen) & rows;
                    any_n |= pn & rows;
                }
                stage[it] = w;
            }
            slice_sync();
            const uint32_t lo = max(my_first, f0), hi = min(my_end, f0 + here);
            for (uint32_t f = lo; f < hi; f++) {
                const uint4 rd = tab[f];
                if (rd.z == 0u) continue;
                // the p rows missing to R SL, one or a few per lane: `lack` of
                // them here, its row 0 at read position q0
                const uint32_t p = (uint32_t)(R * SL) - rd.y, each = p / (uint32_t)SL, more = p % (uint32_t)SL;
                const uint32_t lack = each + (b < more ? 1u : 0u);
                const int32_t q0 = (int32_t)(b * (uint32_t)R) - (int32_t)(b * each + min(b, more)) - (int32_t)lack;
                const int32_t wlo = q0 >> 5;            // floor; -1 for the first lane's missing rows
                const uint32_t sh = (uint32_t)q0 & 31u;
                const uint4 *sw = stage + (f - f0) * (uint32_t)W;
                uint4 x = make_uint4(0u, 0u, 0u, 0u), y = x;
                if (wlo >= 0) x = sw[wlo];
                if (wlo + 1 < W) y = sw[wlo + 1];
                body(rd.z, lack, __builtin_amdgcn_alignbit(y.x, x.x, sh), __builtin_amdgcn_alignbit(y.y, x.y, sh),
                     __builtin_amdgcn_alignbit(y.z, x.z, sh));
            }
        }
    };
    uint32_t r0[R], r1[R], skip[K];
#pragma unroll
    for (int i = 0; i < R; i++) r0[i] = r1[i] = 0u;
#pragma unroll
    for (int i = 0; i < K; i++) skip[i] = 0u;
    each_read([&](uint32_t who, uint32_t lack, uint32_t p0, uint32_t p1, uint32_t) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            r0[i] |= who & (uint32_t)__builtin_amdgcn_sbfe((int)p0, (uint32_t)i, 1u);
            r1[i] |= who & (uint32_t)__builtin_amdgcn_sbfe((int)p1, (uint32_t)i, 1u);
        }
#pragma unroll
        for (int i = 0; i < K; i++) skip[i] |= (uint32_t)i < lack ? who : 0u;
    });
    if (__ballot(bad != 0u) != 0ull) return false;
    const bool with_n = __ballot(any_n != 0u) != 0ull;
    const uint32_t none[1] = {0u};
    if (!with_n) {
        slice_sync();
        slice_columns<SL, R, kPlain>(a, lds, lane, r0, r1, none, skip);
        return true;
    }
    uint32_t rn[R];
#pragma unroll
    for (int i = 0; i < R; i++) rn[i] = 0u;
    each_read([&](uint32_t who, uint32_t, uint32_t, uint32_t, uint32_t pn) {
#pragma unroll
        for (int i = 0; i < R; i++) rn[i] |= who & (uint32_t)__builtin_amdgcn_sbfe((int)pn, (uint32_t)i, 1u);
    });
    slice_sync();
    if constexpr (S::rows_n(R)) {
        slice_columns<SL, R, kRowsN>(a, lds, lane, r0, r1, rn, skip);
    } else {
        // one word per row in this lane's column of the plane
        uint2 *plane = reinterpret_cast<uint2 *>(lds + S::kPlaneU4) + lane;
#pragma unroll
        for (int i = 0; i < R; i += 2)
            plane[(i / 2) * 64] = make_uint2(rn[i], i + 1 < R ? rn[i + 1 < R ? i + 1 : 0] : 0u);
        slice_columns<SL, R, kPlaneN>(a, lds, lane, r0, r1, none, skip);
    }
    return true;
}

// The bit-vector kernel over the same candidates, with the next width of these:
// every one up to kFallbackExact words, where it also runs bins of its own
// (small batches), above it those of the tuning table's bins, where a bin of
// several word counts gives many chunks that the sliced form does not take (200-1000
// bases, a launch per bin: 4.0 ms with 12, 16, 24 and 32, 3.7 ms).  Those that a
// form has no reads for are left out of its kernel.
constexpr uint32_t kFallbackExact = 7;
#define SLICE_FALLBACK_WIDTHS(X)                                                                 \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(9) X(10) X(13) X(16) X(19) X(22) X(25) X(29) X(32)
template <int SL>
__device__ __forceinline__ void slice_fallback(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                               uint32_t chunk, uint32_t words, uint4 *lds) {
    constexpr uint32_t kSub = 32u / (uint32_t)SL;
    const uint32_t lo = chunk * kSub, hi = min(lo + kSub, (count + 63u) / 64u);
#define SLICE_FALLBACK(WF)                                                                       \
    if constexpr ((WF) <= slice_max_words(SL) + 1) {                                             \
        if (words <= (WF)) {                                                                     \
            verify_chunks<1, (WF), false>(a, start, count, lo, hi, 1u, *reinterpret_cast<Workspace<1, (WF)> *>(lds)); \
            return;                                                                              \
        }                                                                                        \
    }
    SLICE_FALLBACK_WIDTHS(SLICE_FALLBACK)
#undef SLICE_FALLBACK
}

// Threshold mode.  An alignment's first rows cost no more than all of it, so a
// candidate whose first r rows' least score is above the threshold k of the
// whole read has no match.  Random text scores about 0.488 r; r rows as below
// rule out 98% of unrelated candidates (random DNA, 50-1000 bases, k of 0.05 to
// 0.3 m): 0.23 m to 0.3 m rows for k = 0.1 m, 0.44 m to 0.52 m for k = 0.2 m.
// The candidates kept start over with all rows, in a second launch of the
// kernel of longer reads (32 candidates per wave, so the few chunks take half
// as long).  Rows per lane, 0: not worth it.  11 candidates per read, one of
// them at its place, k = 0.2 m: 50K reads of 1000 bases 3.83 -> 2.79 ms, 100K of
// 600 bases 2.73 -> 2.43 ms; at 400 bases the work per column is most of a
// chunk and the second launch takes what the first gains (1.56 -> 1.75 ms).
// (k: the threshold of a read of max_words words)
template <int SL>
__host__ __device__ __forceinline__ uint32_t slice_first_rows(uint32_t max_words, float k) {
    const float m = 32.0f * (float)max_words;
    const uint32_t all = 32u * max_words / (uint32_t)SL;
    const float r = 2.05f * k + 0.75f * sqrtf(m) + 6.0f;
    const uint32_t rows = r >= m ? all : ((uint32_t)r + (uint32_t)SL) / (uint32_t)SL;
    return SL == 32 && max_words >= 18u && 10u * rows <= 7u * all ? rows : 0u;
}

// Verify chunk `chunk` (kCands candidates) of the slot range [start, start +
// count) of a bin whose reads have at most max_words words; of their first
// `first` rows per lane only (0: all rows).  kSliceRefused: nothing written, the
// chunk is one for the bit-vector kernel; kSliceShort: nothing written, some
// read has fewer rows than `first`.
enum SliceDone { kSliceDone, kSliceRefused, kSliceShort };
template <int SL>
__device__ __forceinline__ SliceDone verify_slice(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                                  uint32_t chunk, uint32_t max_words, uint32_t first, uint32_t variant,
                                                  uint4 *lds) {
    using S = SliceShape<SL>;
    const uint32_t lane = threadIdx.x, half = lane >> 5, ci = lane & 31u;
    const CandRec *__restrict__ cands = static_cast<const CandRec *>(a.cands);
    const uint2 *__restrict__ qinfo = reinterpret_cast<const uint2 *>(a.qinfo);
    uint32_t m_hi = 0, m_lo = 0xFFFFFFFFu, cols = 0, nreads = 0;
    // The table of the chunk's reads: a run of candidates of one read within a
    // group is one entry.
    uint32_t *first_read = reinterpret_cast<uint32_t *>(lds);
    uint32_t *cand = reinterpret_cast<uint32_t *>(lds + S::kFirstU4);
    uint4 *tab = lds + S::kTextU4;
    slice_sync();
#pragma unroll
    for (int k = 0; k < S::kBatches; k++) {
        const uint32_t slot = chunk * (uint32_t)S::kCands + 64u * (uint32_t)k + lane;
        uint32_t query = 0xFFFFFFFFu, m = 0, entry = 0, index = ~0u, block = 0, window = 0;
        bool live = false;
        if (slot < count) {
            index = a.order ? a.order[start + slot] : start + slot;
            const CandRec cr = cands[index];
            query = cr.query;
            if (query < a.num_queries) {
                const uint2 qi = qinfo[query];
                // the query must fit the bin and its Peq entries the batch
                if (qi.y <= 32u * max_words && (uint64_t)qi.x + ((qi.y + 127u) >> 7) <= (uint64_t)a.num_peq_entries) {
                    entry = qi.x;
                    m = qi.y;
                    const uint32_t n = window_len(m, a.distance);
                    // skip rule: src-api/coreMyersGPU-CC35.cu:142
                    live = cr.position < a.ref_size && a.ref_size - cr.position > (uint64_t)n;
                    if (live) {
                        // aligned window (src-api/coreMyersGPU-CC35.cu:132,144) or exact start:
                        // first text column (base 32 block + window % 32) and columns (window / 32)
                        const uint64_t from = a.mode == 0 ? (cr.position & ~7ull) : cr.position;
                        const uint32_t ncols = a.mode == 0 ? 8u * ((n >> 3) + ((n & 7u) ? 2u : 1u)) : n;
                        block = (uint32_t)(from >> 5);
                        window = ((uint32_t)from & 31u) | (ncols << 5);
                        m_hi = max(m_hi, max(m, 1u));
                        m_lo = min(m_lo, max(m, 1u));
                        cols = max(cols, ncols);
                    }
                }
            }
        }
        uint32_t *cd = cand + 64 * k + lane;
        cd[0] = block;
        cd[S::kCands] = window;
        cd[2 * S::kCands] = !live ? ~0u : first ? threshold_of(m, a.threshold) : m;
        cd[3 * S::kCands] = index;
        const uint32_t below = (uint32_t)__shfl_up((int)query, 1);
        const bool head = ci == 0u || below != query;
        const uint64_t heads64 = __ballot(head), live64 = __ballot(live);
        const uint32_t heads = half ? (uint32_t)(heads64 >> 32) : (uint32_t)heads64;
        const uint32_t lives = half ? (uint32_t)(live64 >> 32) : (uint32_t)live64;
        const uint32_t upto = (2u << ci) - 1u;          // bits 0 .. ci (all of them for ci = 31)
        const uint32_t after = heads & ~upto;
        const uint32_t run = (after ? (after & (0u - after)) - 1u : ~0u) & ~(upto >> 1);
        const uint32_t n_lo = (uint32_t)__builtin_popcount((uint32_t)heads64);
        const uint32_t at = nreads + (half ? n_lo : 0u);
        // the entry and m of a run are its first candidate's: one read has one
        if (head) tab[at + (uint32_t)__builtin_popcount(heads & upto) - 1u] = make_uint4(entry, first ? min(m, first * (uint32_t)SL) : m, run & lives, 0u);
        if (ci == 0u) first_read[(uint32_t)(2 * k) + half] = at;
        nreads += (uint32_t)__builtin_popcountll(heads64);
    }
    if (lane == 0u) first_read[S::kGroups] = nreads;
    slice_sync();
    m_hi = wave_max(m_hi);
    m_lo = ~wave_max(~m_lo);
    const uint32_t max_cols = wave_max(cols);
    if (m_hi == 0u) {                                   // every candidate skipped
#pragma unroll
        for (int k = 0; k < S::kBatches; k++) {
            const uint32_t index = cand[3 * S::kCands + 64 * k + (int)lane];
            if (index != ~0u) static_cast<uint2 *>(a.results)[index] = make_uint2(0u, kSkipScore);
        }
        return kSliceDone;
    }
    if (first) {
        if (m_lo < first * (uint32_t)SL) return kSliceShort;
        m_hi = m_lo = first * (uint32_t)SL;
    }
    if ((m_hi + 31u) >> 5 == (m_lo + 31u) >> 5 && max_cols < kSliceMaxCols) {
        const SliceBatch batch = {a.peq, a.planes, static_cast<uint2 *>(a.results), a.plane_blocks - 1u, a.threshold,
                                  nreads, max_cols, first ? a.list + start : nullptr,
                                  first ? a.list_ranges + 2u * variant + 1u : nullptr, first ? a.tally : nullptr};
        SliceLds *lds_at = (SliceLds *)lds;
        switch ((m_hi + (uint32_t)SL - 1u) / (uint32_t)SL) {
#define SLICE_CASE(R)                                                                            \
    case R:                                                                                      \
        if constexpr ((R) * SL <= 32 * slice_max_words(SL))                                      \
            return slice_run<SL, (R)>(batch, lds_at) ? kSliceDone : kSliceRefused;               \
        break;
            SLICE_CASE(1) SLICE_CASE(2) SLICE_CASE(3) SLICE_CASE(4) SLICE_CASE(5) SLICE_CASE(6) SLICE_CASE(7)
            SLICE_CASE(8) SLICE_CASE(9) SLICE_CASE(10) SLICE_CASE(11) SLICE_CASE(12) SLICE_CASE(13) SLICE_CASE(14)
            SLICE_CASE(15) SLICE_CASE(16) SLICE_CASE(17) SLICE_CASE(18) SLICE_CASE(19) SLICE_CASE(20) SLICE_CASE(21)
            SLICE_CASE(22) SLICE_CASE(23) SLICE_CASE(24) SLICE_CASE(25) SLICE_CASE(26) SLICE_CASE(27) SLICE_CASE(28)
            SLICE_CASE(29) SLICE_CASE(30) SLICE_CASE(31) SLICE_CASE(32)
#undef SLICE_CASE
            default:
                break;
        }
    }
    return kSliceRefused;
}

}  // namespace

#endif
