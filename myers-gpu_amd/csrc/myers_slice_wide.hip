// Reads of over 1024 bases in large batches: the candidate-sliced recurrence
// (myers_slice.h) on teams of waves.
#include "myers_slice.h"

namespace {

// A workgroup of 12 waves, one per CU (three waves per SIMD), is split into
// teams of 12, 4, 3, 2 or 1 waves, the same for a bin.  A team verifies 32
// candidates, lane b of its wave q holding R consecutive rows as in the forms of
// one wave.  Blocks of 32 steps are in step over the workgroup (one barrier each),
// and wave q runs kLag blocks behind wave q - 1, whose top lane's deltas of
// every step pass through a ring in LDS: lane 0 needs column c when the lane
// below it did it 63 steps later, at the end of the second block after this
// one.  Wave 0 brings in the text for the team (a ring of the columns between
// its first lane's block and the last wave's last lane), the top wave keeps the
// score row.
//
// Bound by VALU issue, as the forms of one wave.  Cells per second of large
// batches of one length (no N in the reads; with N): 2,000 bases (1 wave) -;
// 186e12, 6,144 (4 waves, 24 rows) 217e12; 197e12, 8,192 (4 waves, 32 rows)
// 232e12; 186e12, 12,288 (12 waves, 16 rows) 207e12; 180e12, 19,900 (12 waves,
// 26 rows) 232e12; 204e12; the multi-lane bit-vector kernels run 110-130e12.
// Few rows per lane pay for the steps' fixed part and the lag (96 steps per
// wave: 5% of 20,000 bases).  One workgroup for all teams, because launches of
// their own for each team size share two hardware queues and wait for each
// other (1000-4000 bases: 8.2 ms against 6.8).  Text at the start of a block
// and score at its end measured best (both at the end, with the text's loads a
// block ahead: 221e12 at 19,900 bases; both at the start: 213e12).
struct WideSlice {
    static constexpr uint32_t kCands = 32, kLag = 3, kMaxRows = 32, kWaves = MYERS_WIDE_SLICE_WAVES;
    // LDS, in 16-byte units.  Of the workgroup: the item, each team's number of
    // blocks.  Of a team: the text columns (a power of two of them), flags and a
    // zero, the candidates (block, window, length, column of the minimum, score,
    // deltas not searched yet, minimum, index; 32 words each), the table of
    // reads, and for each wave the ring of deltas, spare slots, and the N plane
    // (first the reads' Peq, staged).
    static constexpr uint32_t kHeadU4 = 4;
    static constexpr uint32_t kCandU4 = 2, kTabU4 = kCandU4 + 72, kSharedU4 = kTabU4 + 32;   // from the flags on
    static constexpr uint32_t kStageU4 = 32u * (kMaxRows / 2u);
    static constexpr __host__ __device__ uint32_t cols(uint32_t team) {
        uint32_t c = 128;
        while (c < 32u * (kLag * team + 1u)) c *= 2u;
        return c;
    }
    static constexpr __host__ __device__ uint32_t ring(uint32_t team) { return team == 1u ? 32u : 128u; }
    static constexpr __host__ __device__ uint32_t wave_u4(uint32_t team) { return ring(team) / 2u + 4u + kStageU4; }
    static constexpr __host__ __device__ uint32_t team_u4(uint32_t team) {
        return cols(team) + kSharedU4 + team * wave_u4(team);
    }
    static constexpr uint32_t ws_u4() {
        uint32_t most = 0;
        for (uint32_t team : {1u, 2u, 3u, 4u, 12u})
            most = kWaves / team * team_u4(team) > most ? kWaves / team * team_u4(team) : most;
        return kHeadU4 + most;
    }
};

// What the waves of a team share: its LDS, waves, this wave's number among them,
// and the workgroup's number of blocks (0: teams of one wave keep no step).
struct WideTeam {
    uint4 *lds;
    uint32_t waves, wave, blocks;
};

// slice_score with the score and the minimum in a word each.
__device__ __forceinline__ void slice_score_wide(uint32_t hp, uint32_t hm, uint32_t col0, uint32_t &score,
                                                 uint32_t &min_score, uint32_t &min_col, uint32_t &php, uint32_t &phm) {
    const int32_t begin = (int32_t)score, end = begin + (int32_t)__builtin_popcount(hp) - (int32_t)__builtin_popcount(hm);
    const int32_t least = begin - (int32_t)__builtin_popcount(php);
    int32_t low = (int32_t)min_score;
    if (__ballot(least < low && least <= end) != 0ull) slice_first_min(php, phm, begin, col0 - 32u, low, min_col);
    min_score = (uint32_t)low;
    php = hp;
    phm = hm;
    score = (uint32_t)end;
}

// Columns of one wave (kN: SliceN).
template <int R, int K, int kN>
__device__ __forceinline__ void wide_slice_columns(const SliceBatch &a, const WideTeam &tm, uint4 *own,
                                                   uint32_t lane, const uint32_t (&r0)[R],
                                                   const uint32_t (&r1)[R], const uint32_t (&rn)[kN == kRowsN ? R : 1],
                                                   const uint32_t (&skip)[K]) {
    using S = WideSlice;
    uint4 *lds = tm.lds;
    const uint32_t wave = tm.wave, waves = tm.waves;
    const uint32_t ring_cols = S::ring(waves), text_mask = 16u * S::cols(waves) - 1u;
    uint4 *shared = lds + S::cols(waves);
    uint32_t *cand = reinterpret_cast<uint32_t *>(shared + S::kCandU4);
    char *text = reinterpret_cast<char *>(lds);
    uint2 *ring = reinterpret_cast<uint2 *>(own);
    const uint2 *np = reinterpret_cast<const uint2 *>(own + ring_cols / 2u + 4u) + lane;
    // deltas entering lane 0: the ring of the wave below; the bottom wave reads
    // the zero behind the flags
    const uint2 *below = wave ? reinterpret_cast<const uint2 *>(own - S::wave_u4(waves))
                              : reinterpret_cast<const uint2 *>(shared + 1);
    const uint32_t below_mask = wave ? ring_cols - 1u : 0u;
    const bool top_wave = wave + 1u == waves;
    // before a lane's first column it reads text that matches no row (as above)
    if (wave == 0u) *reinterpret_cast<uint3 *>(text + ((16u * (lane - 64u)) & text_mask)) = make_uint3(~0u, 0u, ~0u);
    uint32_t Pv[R], Mv[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        Pv[i] = ~0u;
        Mv[i] = 0u;
    }
    uint32_t hp = 0, hm = 0;
    const uint32_t out_inc = lane == 63u ? 1u : 0u;
    const uint32_t nsteps = a.max_cols + 63u, nblocks = (nsteps + 31u) >> 5;
    uint32_t last0 = 0;
    __syncthreads();                                    // rings and flags are ready
    for (uint32_t at = 0; at < (tm.blocks ? tm.blocks : nblocks); at++) {
        const uint32_t blk = at - S::kLag * wave;       // wraps before this wave's first block
        if (blk < nblocks) {
            const uint32_t s0 = blk * 32u;
            uint32_t l = lane;
            asm volatile("" : "+v"(l));                 // (as in slice_columns)
            if (wave == 0u) {                           // (both halves hold the same candidates)
                const uint32_t *cd = cand + (l & 31u);
                const uint32_t b0 = cd[0] + blk, shift = cd[S::kCands];
                const uint3 cur = slice_planes(a.planes, b0, a.last_block);
                const uint3 nxt = slice_planes(a.planes, b0 + 1u, a.last_block);
                uint3 w;
                w.x = transpose32(__builtin_amdgcn_alignbit(nxt.x, cur.x, shift), l);
                w.y = transpose32(__builtin_amdgcn_alignbit(nxt.y, cur.y, shift), l);
                w.z = transpose32(__builtin_amdgcn_alignbit(nxt.z, cur.z, shift), l);
                if (l < 32u) *reinterpret_cast<uint3 *>(text + ((16u * (s0 + l)) & text_mask)) = w;
            }
            slice_sync();
            const uint32_t nj = min(32u, nsteps - s0);
            // lane 63 writes the ring, the others the spare slots behind it
            uint32_t oi = out_inc ? (s0 & (ring_cols - 1u)) : ring_cols + (l & 7u);
            const uint32_t in0 = s0 + 63u;
            uint32_t t_at = (16u * (s0 - l)) & text_mask;
            uint3 t = *reinterpret_cast<const uint3 *>(text + t_at);
            uint2 in = below[in0 & below_mask];
            for (uint32_t j = 0; j < nj; j += 2u) {
#pragma unroll
                for (uint32_t u = 0; u < 2u; u++) {
                    // (the last step of a block reads one past its columns: not used)
                    t_at = (t_at + 16u) & text_mask;
                    const uint3 t_next = *reinterpret_cast<const uint3 *>(text + t_at);
                    const uint2 in_next = below[(in0 + j + u + 1u) & below_mask];
                    hp = (uint32_t)__builtin_amdgcn_update_dpp((int)in.x, (int)hp, 0x138, 0xF, 0xF, false);
                    hm = (uint32_t)__builtin_amdgcn_update_dpp((int)in.y, (int)hm, 0x138, 0xF, 0xF, false);
                    slice_step<R, K, kN>(Pv, Mv, r0, r1, rn, skip, make_uint4(t.x, t.y, t.z, 0u), np, hp, hm);
                    ring[oi] = make_uint2(hp, hm);
                    oi += out_inc;
                    t = t_next;
                    in = in_next;
                    SLICE_FIX;
                }
            }
            if (top_wave) {
                slice_sync();
                asm volatile("" : "+v"(l));
                uint32_t *cd = cand + (l & 31u);
                // step s0 + j gave the score row's deltas of column s0 + j - 63
                const uint32_t col0 = s0 - 63u;         // wraps in the first two blocks
                // (signed: `s0 < 63u ? min(63u - s0, 32u) : 0u` makes clang 22 take
                // s0 <= 63 for granted after it)
                const uint32_t before = (uint32_t)min(max(63 - (int32_t)s0, 0), 32);
                const uint2 v = ring[(s0 & (ring_cols - 1u)) + (l & 31u)];
                uint32_t min_col = cd[3 * S::kCands], score = cd[4 * S::kCands], php = cd[5 * S::kCands];
                uint32_t phm = cd[6 * S::kCands], min_score = cd[7 * S::kCands];
                const uint32_t seen = col0 + before, ncols = cd[S::kCands] >> 5;
                const uint32_t left = ncols > seen ? ncols - seen : 0u;
                const uint32_t mask = before >= 32u ? 0u : (left >= 32u ? ~0u : (1u << left) - 1u) << before;
                slice_score_wide(transpose32(v.x, l) & mask, transpose32(v.y, l) & mask, col0, score, min_score, min_col,
                                 php, phm);
                cd[3 * S::kCands] = min_col;
                cd[4 * S::kCands] = score;
                cd[5 * S::kCands] = php;
                cd[6 * S::kCands] = phm;
                cd[7 * S::kCands] = min_score;
                last0 = col0;
            }
        }
        if (tm.blocks) __syncthreads();
    }
    if (!top_wave) return;
    const uint32_t *cd = cand + (lane & 31u);
    uint32_t min_col = cd[3 * S::kCands];
    const uint32_t score = cd[4 * S::kCands], php = cd[5 * S::kCands], phm = cd[6 * S::kCands];
    int32_t min_score = (int32_t)cd[7 * S::kCands];
    if (__ballot((int32_t)score - (int32_t)__builtin_popcount(php) < min_score) != 0ull)
        slice_first_min(php, phm, (int32_t)score, last0, min_score, min_col);
    const uint32_t m = cd[2 * S::kCands], index = cd[8 * S::kCands];
    if (lane >= 32u || index == ~0u) return;
    uint2 r = make_uint2(0u, kSkipScore);
    if (m != ~0u) {
        r = make_uint2(min_col, (uint32_t)min_score);
        if (a.threshold >= 0.0f && r.y > threshold_of(m, a.threshold)) r = make_uint2(kNoMatch, kNoMatch);
    }
    a.results[index] = r;
}

// A wave of a team without candidates keeps step with the others.
__device__ __forceinline__ void wide_slice_idle(uint32_t blocks) {
    for (uint32_t at = 0; at < 2u + blocks; at++) __syncthreads();
}

// The rows of one wave of a team of T waves whose 32 candidates' reads have
// between 64 T (R - K) and 64 T R bases, and their columns.  False (nothing
// written, in every wave of the team) if a read's Peq is not one code per base.
template <int R, int K>
__device__ __noinline__ bool wide_slice_run(SliceBatch a, SliceLds *lds_at, uint32_t waves_v, uint32_t wave_v, uint32_t blocks_v) {
    using S = WideSlice;
    a.peq = uniform_ptr(a.peq);
    a.planes = uniform_ptr(a.planes);
    a.results = uniform_ptr(a.results);
    a.last_block = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.last_block);
    a.threshold = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(a.threshold)));
    a.max_cols = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.max_cols);
    const uint32_t nreads = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.nreads);
    const uint32_t waves = (uint32_t)__builtin_amdgcn_readfirstlane((int)waves_v);
    const uint32_t lane = __lane_id();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_v);
    const uint32_t blocks = (uint32_t)__builtin_amdgcn_readfirstlane((int)blocks_v);
    uint4 *lds = (uint4 *)lds_at;
    const WideTeam tm = {lds, waves, wave, blocks};
    uint4 *shared = lds + S::cols(waves), *own = shared + S::kSharedU4 + wave * S::wave_u4(waves);
    uint32_t *flags = reinterpret_cast<uint32_t *>(shared);
    const uint4 *tab = shared + S::kTabU4;
    uint4 *stage = own + S::ring(waves) / 2u + 4u;
    constexpr uint32_t kWords = 2u * (uint32_t)R + 3u;  // a read's words that a wave's rows can touch
    constexpr uint32_t kPass = S::kStageU4 / kWords;
    const uint32_t lanes = 64u * waves, b = 64u * wave + lane, b0 = 64u * wave;
    uint32_t bad = 0, any_n = 0;
    // the p rows missing to 64 waves R, one or a few per lane: `lack` of them in
    // lane x, its row 0 at the read position returned
    auto place = [&](uint32_t m, uint32_t x, uint32_t &lack) {
        const uint32_t p = lanes * (uint32_t)R - m, each = p / lanes, more = p - each * lanes;
        lack = each + (x < more ? 1u : 0u);
        return (int32_t)(x * (uint32_t)R) - (int32_t)(x * each + min(x, more)) - (int32_t)lack;
    };
    auto each_read = [&](auto body) {
        for (uint32_t f0 = 0; f0 < nreads; f0 += kPass) {
            const uint32_t here = min(kPass, nreads - f0);
            slice_sync();
            for (uint32_t it = lane; it < here * kWords; it += 64u) {
                const uint4 rd = tab[f0 + it / kWords];
                uint32_t lack0 = 0;
                const int32_t first = place(rd.y, b0, lack0) >> 5;        // the wave's first word (-1: none there)
                const int32_t j = first + (int32_t)(it % kWords);
                uint4 w = make_uint4(0u, 0u, 0u, 0u);
                if (rd.z != 0u && j >= 0 && 32 * j < (int32_t)rd.y) {
                    const uint32_t *p = a.peq + (size_t)(rd.x + ((uint32_t)j >> 2)) * 20u + ((uint32_t)j & 3u);
                    const uint32_t pa = p[0], pc = p[4], pg = p[8], pt = p[12], pn = p[16];
                    const uint32_t rows = rd.y - 32u * (uint32_t)j >= 32u ? ~0u : (1u << (rd.y & 31u)) - 1u;
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
            for (uint32_t f = f0; f < f0 + here; f++) {
                const uint4 rd = tab[f];
                if (rd.z == 0u) continue;
                uint32_t lack = 0, lack0 = 0;
                const int32_t q0 = place(rd.y, b, lack), first = place(rd.y, b0, lack0) >> 5;
                const uint32_t sh = (uint32_t)q0 & 31u;
                const uint4 *sw = stage + (f - f0) * kWords + (uint32_t)((q0 >> 5) - first);
                const uint4 x = sw[0], y = sw[1];
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
    if (__ballot(bad != 0u) != 0ull && lane == 0u) flags[0] = 1u;
    __syncthreads();
    const bool refused = __builtin_amdgcn_readfirstlane((int)flags[0]) != 0;
    if (refused) {
        for (uint32_t at = 0; at < 1u + blocks; at++) __syncthreads();
        return false;
    }
    const uint32_t none[1] = {0u};
    if (__ballot(any_n != 0u) == 0ull) {
        wide_slice_columns<R, K, kPlain>(a, tm, own, lane, r0, r1, none, skip);
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
    if constexpr (5 * R + 4 <= 134) {
        wide_slice_columns<R, K, kRowsN>(a, tm, own, lane, r0, r1, rn, skip);
    } else {
        uint2 *plane = reinterpret_cast<uint2 *>(stage) + lane;
#pragma unroll
        for (int i = 0; i < R; i += 2)
            plane[(i / 2) * 64] = make_uint2(rn[i], i + 1 < R ? rn[i + 1 < R ? i + 1 : 0] : 0u);
        wide_slice_columns<R, K, kPlaneN>(a, tm, own, lane, r0, r1, none, skip);
    }
    return true;
}

// 32 candidates from slot `first` of a bin's slot range [start, start + count)
// on team `team` of the workgroup.  False: nothing written, the candidates are
// ones for the bit-vector kernel.
__device__ __forceinline__ bool verify_wide_slice(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                                  uint32_t first, uint32_t waves, uint32_t team, uint32_t wave,
                                                  uint4 *wg) {
    using S = WideSlice;
    const uint32_t lane = threadIdx.x & 63u, ci = lane & 31u;
    const CandRec *__restrict__ cands = static_cast<const CandRec *>(a.cands);
    const uint2 *__restrict__ qinfo = reinterpret_cast<const uint2 *>(a.qinfo);
    uint4 *lds = wg + S::kHeadU4 + team * S::team_u4(waves), *shared = lds + S::cols(waves);
    uint32_t *head = reinterpret_cast<uint32_t *>(wg);
    uint32_t *cand = reinterpret_cast<uint32_t *>(shared + S::kCandU4);
    uint32_t *flags = reinterpret_cast<uint32_t *>(shared);
    const uint32_t lanes = 64u * waves;
    // every wave looks at the candidates (both halves at the same ones); they
    // all write the same state and table
    const uint32_t slot = first + ci;
    uint32_t query = 0xFFFFFFFFu, m = 0, entry = 0, index = ~0u, block = 0, window = 0, cols = 0;
    bool live = false;
    if (slot < count) {
        index = a.order ? a.order[start + slot] : start + slot;
        const CandRec cr = cands[index];
        query = cr.query;
        if (query < a.num_queries) {
            const uint2 qi = qinfo[query];
            if (qi.y <= lanes * S::kMaxRows &&
                (uint64_t)qi.x + ((qi.y + 127u) >> 7) <= (uint64_t)a.num_peq_entries) {
                entry = qi.x;
                m = qi.y;
                const uint32_t n = window_len(m, a.distance);
                // skip rule: src-api/coreMyersGPU-CC35.cu:142
                live = cr.position < a.ref_size && a.ref_size - cr.position > (uint64_t)n;
                if (live) {
                    // aligned window (src-api/coreMyersGPU-CC35.cu:132,144) or exact start
                    const uint64_t at = a.mode == 0 ? (cr.position & ~7ull) : cr.position;
                    cols = a.mode == 0 ? 8u * ((n >> 3) + ((n & 7u) ? 2u : 1u)) : n;
                    block = (uint32_t)(at >> 5);
                    window = ((uint32_t)at & 31u) | (cols << 5);
                }
            }
        }
    }
    const uint32_t m_hi = wave_max(live ? max(m, 1u) : 0u), m_lo = ~wave_max(live ? ~max(m, 1u) : 0u);
    const uint32_t max_cols = wave_max(cols);
    const uint32_t prev = (uint32_t)__shfl_up((int)query, 1);
    const uint32_t heads = (uint32_t)__ballot(ci == 0u || prev != query);
    const uint32_t lives = (uint32_t)__ballot(live);
    const bool sliced = m_hi != 0u && max_cols < kSliceMaxCols;
    if (wave == 0u) {
        uint32_t *cd = cand + ci;
        cd[0] = block;
        cd[S::kCands] = window;
        cd[2 * S::kCands] = live ? m : ~0u;
        cd[3 * S::kCands] = 0u;
        cd[4 * S::kCands] = live ? m : 0u;
        cd[5 * S::kCands] = cd[6 * S::kCands] = 0u;
        cd[7 * S::kCands] = live ? m : 0u;
        cd[8 * S::kCands] = index;
        const uint32_t upto = (2u << ci) - 1u;
        const uint32_t after = heads & ~upto;
        const uint32_t run = (after ? (after & (0u - after)) - 1u : ~0u) & ~(upto >> 1);
        if ((heads >> ci) & 1u)
            (shared + S::kTabU4)[__builtin_popcount(heads & upto) - 1] = make_uint4(entry, m, run & lives, 0u);
        if (lane < 8u) flags[lane] = 0u;
        if (lane == 0u) head[1u + team] = sliced ? (max_cols + 63u + 31u) / 32u + S::kLag * (waves - 1u) : 0u;
    }
    __syncthreads();
    uint32_t blocks = 0;
    if (waves > 1u) {
        for (uint32_t i = 0; i < S::kWaves / waves; i++) blocks = max(blocks, head[1u + i]);
    }
    blocks = (uint32_t)__builtin_amdgcn_readfirstlane((int)blocks);
    if (!sliced) {
        wide_slice_idle(blocks);
        if (m_hi != 0u) return false;
        // every candidate skipped
        if (wave == 0u && lane < 32u && index != ~0u) static_cast<uint2 *>(a.results)[index] = make_uint2(0u, kSkipScore);
        return true;
    }
    const SliceBatch batch = {a.peq, a.planes, static_cast<uint2 *>(a.results), a.plane_blocks - 1u, a.threshold,
                              (uint32_t)__builtin_popcount(heads), max_cols, nullptr, nullptr, nullptr};
    SliceLds *lds_at = (SliceLds *)lds;
    const uint32_t rows = (m_hi + lanes - 1u) / lanes, lack = lanes * rows - m_lo;
    // (K rows that a lane may lack: two where the candidates are of about one
    // length)
#define WIDE_SLICE_CASE(R)                                                                       \
    case R:                                                                                      \
        if (lack <= 2u * lanes) return wide_slice_run<R, 2>(batch, lds_at, waves, wave, blocks);               \
        if (lack <= 8u * lanes) return wide_slice_run<R, 8>(batch, lds_at, waves, wave, blocks);               \
        break;
    switch (rows) {
        WIDE_SLICE_CASE(9) WIDE_SLICE_CASE(10) WIDE_SLICE_CASE(11) WIDE_SLICE_CASE(12) WIDE_SLICE_CASE(13) WIDE_SLICE_CASE(14) WIDE_SLICE_CASE(15)
        WIDE_SLICE_CASE(16) WIDE_SLICE_CASE(17) WIDE_SLICE_CASE(18) WIDE_SLICE_CASE(19) WIDE_SLICE_CASE(20)
        WIDE_SLICE_CASE(21) WIDE_SLICE_CASE(22) WIDE_SLICE_CASE(23) WIDE_SLICE_CASE(24) WIDE_SLICE_CASE(25)
        WIDE_SLICE_CASE(26) WIDE_SLICE_CASE(27) WIDE_SLICE_CASE(28) WIDE_SLICE_CASE(29) WIDE_SLICE_CASE(30)
        WIDE_SLICE_CASE(31) WIDE_SLICE_CASE(32)
        default:
            break;
    }
#undef WIDE_SLICE_CASE
    wide_slice_idle(blocks);
    return false;
}

// A team's 32 candidates on the bit-vector kernel, one candidate per wave (of
// as many waves as the team's LDS holds workspaces for).
template <int T>
__device__ __noinline__ void wide_slice_fallback(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                                 uint32_t first, uint32_t wave, SliceLds *lds_at) {
    using W = Workspace<64, T>;
    constexpr uint32_t kNeed = ((uint32_t)sizeof(W) + 15u) / 16u, kFit = WideSlice::team_u4(T) / kNeed;
    constexpr uint32_t kTeam = kFit < (uint32_t)T ? kFit : (uint32_t)T;
    static_assert(kTeam > 0u, "room for one wave's workspace");
    if (wave >= kTeam) return;
    W &ws = *reinterpret_cast<W *>((uint4 *)lds_at + wave * kNeed);
    zero_row_init<64, T, 2>(ws);
    wave_lds_sync();
    verify_chunks<64, T, false, 2>(a, start, count, first + wave, min(first + WideSlice::kCands, count), kTeam, ws);
}

// Every bin of the plan, 12 / T times 32 candidates at a time for teams of T
// waves, from a single counter in plan order (longest reads first).
__global__ __launch_bounds__(64 * (int)WideSlice::kWaves) __attribute__((amdgpu_waves_per_eu(3)))
void verify_wide_slice_kernel(myers_verify_args_t a, myers_queue_plan_t p) {
    extern __shared__ uint4 slice_lds[];
    using S = WideSlice;
    uint32_t *head = reinterpret_cast<uint32_t *>(slice_lds);
    const uint32_t wg_wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (;;) {
        if (threadIdx.x == 0) head[0] = atomicAdd(a.queue_heads + MYERS_QUEUE_HEAD(MYERS_QUEUE_WIDE), 1u);
        __syncthreads();
        const uint32_t item = (uint32_t)__builtin_amdgcn_readfirstlane((int)head[0]);
        uint32_t base = 0, start = 0, count = 0, waves = 1, per = S::kCands;
        bool found = false;
        for (uint32_t j = 0; j < p.n && !found; j++) {
            start = a.bin_ranges[2u * p.variant[j]];
            count = a.bin_ranges[2u * p.variant[j] + 1u];
            waves = p.key[j];
            per = S::kCands * (S::kWaves / waves);
            const uint32_t items = (count + per - 1u) / per;
            found = item - base < items;
            if (!found) base += items;
        }
        if (!found) break;                       // every bin drained: each wave exits here
        const uint32_t team = wg_wave / waves, wave = wg_wave - team * waves;
        const uint32_t first = (item - base) * per + team * S::kCands;
        const bool done = verify_wide_slice(a, start, count, first, waves, team, wave, slice_lds);
        __syncthreads();
        if (!done) {
            SliceLds *lds = (SliceLds *)(slice_lds + S::kHeadU4 + team * S::team_u4(waves));
            switch (waves) {
                case 1: wide_slice_fallback<1>(a, start, count, first, wave, lds); break;
                case 2: wide_slice_fallback<2>(a, start, count, first, wave, lds); break;
                case 3: wide_slice_fallback<3>(a, start, count, first, wave, lds); break;
                case 4: wide_slice_fallback<4>(a, start, count, first, wave, lds); break;
                default: wide_slice_fallback<12>(a, start, count, first, wave, lds); break;
            }
        }
    }
}

}  // namespace

extern "C" uint32_t myers_wide_slice_team(uint32_t words) {
    // one wave, or the fewest waves with at most 26 rows per lane (where a
    // read's N plane still fits the registers), or with 32
    for (uint32_t rows = 26u; rows <= WideSlice::kMaxRows; rows += 6u)
        for (uint32_t team : {1u, 2u, 3u, 4u})
            if (words <= team * 2u * (team == 1u ? WideSlice::kMaxRows : rows)) return team;
    return words <= 12u * 2u * WideSlice::kMaxRows ? 12u : 0u;
}

extern "C" int myers_launch_wide_slice(const myers_verify_args_t *args, const myers_queue_plan_t *plan, uint32_t grid,
                                       hipStream_t stream) {
    if (args == nullptr || plan == nullptr || grid == 0 || plan->n == 0 || plan->n > (uint32_t)MYERS_QUEUE_MAX ||
        args->planes == nullptr || args->plane_blocks == 0 || args->bin_ranges == nullptr ||
        args->queue_heads == nullptr || plan->cls != (uint32_t)MYERS_QUEUE_WIDE)
        return -1;
    for (uint32_t j = 0; j < plan->n; j++) {
        myers_variant_desc_t d;
        if (myers_variant_desc(plan->variant[j], &d) != 0) return -1;
        const uint32_t team = myers_wide_slice_team(d.total_words);
        if (team == 0u || plan->key[j] != team) return -1;
    }
    const size_t lds = (size_t)WideSlice::ws_u4() * 16u;
    const void *fn = reinterpret_cast<const void *>(&verify_wide_slice_kernel);
    // above 64 KiB a launch needs the kernel's limit raised (as myers_launch_long)
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    void *kargs[] = {const_cast<myers_verify_args_t *>(args), const_cast<myers_queue_plan_t *>(plan)};
    return (int)hipLaunchKernel(fn, dim3(grid), dim3(64u * WideSlice::kWaves), kargs, lds, stream);
}
