// Long reads in small batches: one candidate's rows split over waves anywhere
// on the chip.
//
// A batch of few long reads is bound by one candidate's chain of column steps.
// A wave alone on its SIMD issues one instruction every few clocks whatever it
// does, so a step's time is its instruction count: 64 lanes of W words each
// hold a part of 2048 W rows, and the parts of a candidate are items of their
// own, pulled from one counter by waves that know nothing of each other.  A
// part's top lane hands its horizontal deltas on through memory, 32 columns per
// 64-bit word, and the part above follows a few blocks behind.
//
//   * Hand-over.  The deltas of a column are 0, +1 or -1; a word holds the
//     complements (~p, ~m), so that no written word is zero and zero means "not
//     there yet": one relaxed 64-bit store and load at device scope, no flag.
//     The reader puts zero back, so the words are clear for the next use.
//   * Waits end.  Items are pulled in order, candidate by candidate and part
//     after part, so whatever a wave waits for is done by a wave that pulled
//     earlier: by induction it runs or has finished, whichever workgroups are
//     resident.  Slots (one boundary between two parts each) are used in turn;
//     the next writer and reader of a slot wait until its earlier reader counted
//     itself done.
//   * A step.  Text arrives by a lane shift like the deltas, its new column from
//     a register that holds the block's columns in its lanes; deltas travel as one
//     register (+1 in bit 31, -1 in bit 0).  Part p starts P - 1 - p columns
//     early, which lines its blocks up with the words it reads and writes.
//
// Bound by single-wave issue: 22 to 24 VALU operations per step of one word (32
// to 34 of two) at about 5 clocks each, 52 and 70 ns per step; the workgroup of
// four waves and three words per lane that took such reads before needs 118 ns
// (46 operations per step, a barrier every 8 steps).  Four words per lane take
// 105 ns, or 85 ns of a SIMD's time with two waves on it: 98e12 cells per second
// against 60e12 with two words, for batches of some hundred long reads.  One
// candidate of 20,000 bases: 6.4 ms on one wave, 2.9 on such a workgroup, 1.57
// here (10 parts).  Blocks of 64 steps because a word's way through memory takes
// about 2 us: with blocks of 32 steps, one ahead, the loads stalled 0.4 us per
// block (1.98 ms).
#include "myers_device.h"

namespace {

constexpr uint32_t kSplitWaves = 4;                     // independent waves per workgroup, one per SIMD

template <int W>
struct SplitLds {
    uint32_t eq[6 * 64 * W];                            // [row][lane][word]: A C G T N, zero
};

// What the waves of a candidate share.
struct SplitCand {
    uint64_t nib0;                                      // first column's base
    uint32_t entry, m, ncols;
};

// Wait until a boundary's slot has been read `times` times.
__device__ __forceinline__ void split_wait_done(uint32_t *done, uint32_t times) {
    while ((uint32_t)__builtin_amdgcn_readfirstlane(
               (int)__hip_atomic_load(done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT)) < times)
        __builtin_amdgcn_s_sleep(8);
}

// The first minimum of a block of 32 columns (deltas p, m, score `begin` before
// them), if it is below low.  Uniform.
__device__ __forceinline__ void split_first_min(uint32_t p, uint32_t m, uint32_t begin, uint32_t col0, uint32_t &low,
                                                uint32_t &min_col) {
    const uint32_t j = __lane_id() & 31u, upto = (2u << j) - 1u;
    const uint32_t s = begin + (uint32_t)__builtin_popcount(p & upto) - (uint32_t)__builtin_popcount(m & upto);
    const uint32_t key = ~wave_max(~((s << 6) | j));
    if ((key >> 6) < low) {
        low = key >> 6;
        min_col = col0 + (key & 63u);
    }
}

// The columns of one part on one wave.  in / out: words of the boundary below
// and above (kBelow, kAbove).  Returns {min_col, min_score} of the top part.
template <int W, bool kBelow, bool kAbove>
__device__ __forceinline__ uint2 split_columns(const myers_verify_args_t &a, const SplitCand &c, uint32_t ahead,
                                               const uint32_t *eq_lane, uint64_t *in, uint64_t *out) {
    const uint32_t lane = __lane_id();
    const uint32_t *__restrict__ ref = a.ref;
    const int64_t last_word = (int64_t)a.ref_words - 1;
    constexpr uint32_t kRow = 64u * (uint32_t)W * 4u;   // bytes
    // a column's base code in the low bits, and the LDS offset of its Eq row
    // (the zero row before the first column)
    auto text_of = [&](int32_t col) {
        const int64_t nib = (int64_t)c.nib0 + (int64_t)max(col, 0);
        return ref[min(nib >> 3, last_word)] >> (4u * ((uint32_t)nib & 7u));
    };
    auto row_of = [&](uint32_t text, int32_t col) {
        const uint32_t code = text & 7u;
        return (col < 0 ? 5u : code > 4u ? 0u : code) * kRow;
    };
    auto eq_of = [&](uint32_t off, uint32_t (&e)[W]) {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(eq_lane) + off);
#pragma unroll
        for (int k = 0; k < W; k++) e[k] = p[k];
    };
    // lane b is at column s - ahead - b at step s; its Eq words are read two
    // steps before
    const int32_t first = -(int32_t)ahead - (int32_t)lane;
    uint32_t e0[W], e1[W], e2[W];
    eq_of(row_of(text_of(first), first), e0);
    eq_of(row_of(text_of(first + 1), first + 1), e1);
    uint32_t off = row_of(text_of(first + 2), first + 2);
    uint32_t Pv[W], Mv[W];
#pragma unroll
    for (int k = 0; k < W; k++) {
        Pv[k] = ~0u;
        Mv[k] = 0u;
    }
    // blocks of 64 steps, two words of deltas each
    const uint32_t nblocks = (c.ncols + 63u + ahead + 63u) >> 6;
    const uint32_t blocks_in = (c.ncols + ahead + 63u) >> 6, blocks_out = (c.ncols + ahead - 1u + 63u) >> 6;
    // lane l: the column whose Eq row lane 0 starts on at step 64 b + l
    int32_t feed_col = 3 + (int32_t)lane - (int32_t)ahead;
    uint32_t feed_text = text_of(feed_col);
    // the half of the block that this lane's step is in
    const uint32_t half = lane >> 5, bit = lane & 31u;
    auto deltas = [&](uint32_t b) {
        return __hip_atomic_load(in + 2u * b + half, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    uint64_t word = kBelow ? deltas(0u) : 0ull;
    uint32_t h = 0, acc_p = 0, acc_m = 0;
    uint32_t score = c.m, low = c.m, min_col = 0, pend_p = 0, pend_m = 0, pend_col = 0;
    for (uint32_t b = 0; b < nblocks; b++) {
        uint32_t feed = row_of(feed_text, feed_col);
        feed_col += 64;
        feed_text = text_of(feed_col);
        uint32_t feed_h = 0;
        if constexpr (kBelow) {
            if (b < blocks_in) {
                while (__ballot(word == 0ull) != 0ull) {
                    __builtin_amdgcn_s_sleep(2);
                    word = deltas(b);
                }
                if (bit == 0u) __hip_atomic_store(in + 2u * b + half, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t p = ~(uint32_t)(word >> 32), m = ~(uint32_t)word;
                feed_h = ((p >> bit) << 31) | ((m >> bit) & 1u);
                if (b + 1u < blocks_in) word = deltas(b + 1u);
            }
        }
        uint32_t p0 = 0, m0 = 0;                        // the top lane's deltas of this lane's half, first step in bit 0
#pragma unroll 1
        for (uint32_t q = 0; q < 2u; q++) {
#pragma unroll 8
        for (uint32_t j = 0; j < 32u; j++) {
            eq_of(off, e2);
            off = (uint32_t)__builtin_amdgcn_update_dpp((int)feed, (int)off, 0x138, 0xF, 0xF, false);         // wave_shr:1
            feed = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)feed, 0x130, 0xF, 0xF, true);                // wave_shl:1
            uint32_t hi;
            if constexpr (kBelow) {
                hi = (uint32_t)__builtin_amdgcn_update_dpp((int)feed_h, (int)h, 0x138, 0xF, 0xF, false);
                feed_h = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)feed_h, 0x130, 0xF, 0xF, true);
            } else {
                hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)h, 0x138, 0xF, 0xF, true);
            }
            // one column (src/myers-4bits.c:115-134 block form)
            const uint32_t hm = hi & 1u;
            uint32_t carry = 0, ph_prev = hi, mh_prev = 0;
#pragma unroll
            for (int k = 0; k < W; k++) {
                const uint32_t pv = Pv[k], mv = Mv[k], e = e0[k];
                const uint32_t xv = e | mv, eq = k == 0 ? e | hm : e;
                uint32_t c_out;
                const uint32_t sum = __builtin_addc(eq & pv, pv, carry, &c_out);
                carry = c_out;
                const uint32_t xh = __builtin_amdgcn_bitop3_b32(sum, pv, eq, kXorOr);
                const uint32_t ph = __builtin_amdgcn_bitop3_b32(mv, xh, pv, kOrNor);
                const uint32_t mh = pv & xh;
                const uint32_t php = __builtin_amdgcn_alignbit(ph, ph_prev, 31u);
                const uint32_t mhp = k == 0 ? (mh << 1) | hm : __builtin_amdgcn_alignbit(mh, mh_prev, 31u);
                ph_prev = ph;
                mh_prev = mh;
                Pv[k] = __builtin_amdgcn_bitop3_b32(mhp, xv, php, kOrNor);
                Mv[k] = php & xv;
            }
            h = (ph_prev & 0x80000000u) | (mh_prev >> 31);
            acc_p = __builtin_amdgcn_alignbit(acc_p, ph_prev, 31u);
            acc_m = __builtin_amdgcn_alignbit(acc_m, mh_prev, 31u);
#pragma unroll
            for (int k = 0; k < W; k++) {
                e0[k] = e1[k];
                e1[k] = e2[k];
            }
        }
            const uint32_t pq = __builtin_bitreverse32((uint32_t)__builtin_amdgcn_readlane((int)acc_p, 63));
            const uint32_t mq = __builtin_bitreverse32((uint32_t)__builtin_amdgcn_readlane((int)acc_m, 63));
            if constexpr (kAbove) {
                p0 = half == q ? pq : p0;
                m0 = half == q ? mq : m0;
            } else {
                // 32 columns (ahead is 0 here)
                const int32_t col0 = 64 * (int32_t)b + 32 * (int32_t)q - 63;
                const uint32_t before = (uint32_t)min(max(-col0, 0), 32);
                const uint32_t left = (uint32_t)min(max((int32_t)c.ncols - col0, 0), 32);  // columns below ncols
                const uint32_t mask = (uint32_t)(((1ull << left) - 1ull) & ~((1ull << before) - 1ull));
                const uint32_t pw = pq & mask, mw = mq & mask;
                // the columns before are searched only if they may hold a new
                // minimum that no later score is below
                const uint32_t end = score + (uint32_t)__builtin_popcount(pw) - (uint32_t)__builtin_popcount(mw);
                const int32_t least = (int32_t)score - (int32_t)__builtin_popcount(pend_p);
                if (least < (int32_t)low && least <= (int32_t)end)
                    split_first_min(pend_p, pend_m, (uint32_t)least + (uint32_t)__builtin_popcount(pend_m), pend_col,
                                    low, min_col);
                score = end;
                pend_p = pw;
                pend_m = mw;
                pend_col = (uint32_t)col0;
            }
        }
        if constexpr (kAbove) {
            if (b >= 1u && b - 1u < blocks_out && bit == 0u)
                __hip_atomic_store(out + 2u * (b - 1u) + half, ((uint64_t)~p0 << 32) | (uint64_t)~m0, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (!kAbove)
        split_first_min(pend_p, pend_m,
                        score - (uint32_t)__builtin_popcount(pend_p) + (uint32_t)__builtin_popcount(pend_m), pend_col,
                        low, min_col);
    return make_uint2(min_col, low);
}

// Peq words of part `part` of P for this wave's lanes, top-justified over all
// parts (as stage_peq has them), each lane its own words.
template <int W>
__device__ __forceinline__ void split_stage(const myers_verify_args_t &a, const SplitCand &c, uint32_t part,
                                            uint32_t parts, SplitLds<W> &lds) {
    const uint32_t lane = __lane_id();
    const int32_t pad = (int32_t)(parts * 2048u * (uint32_t)W) - (int32_t)c.m;
    const int32_t nq = (int32_t)((c.m + 31u) >> 5);
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < W; k++) {
        const int32_t b0 = 32 * (int32_t)((part * 64u + lane) * (uint32_t)W + (uint32_t)k) - pad;
        const int32_t lo = b0 >> 5;
        const uint32_t sh = (uint32_t)b0 & 31u;
        for (uint32_t r = 0; r < 5u; r++) {
            const uint32_t *base = a.peq + (size_t)c.entry * 20u + 4u * r;
            uint32_t wlo = 0, whi = 0;
            if (lo >= 0 && lo < nq) wlo = base[(uint32_t)(lo >> 2) * 20u + (uint32_t)(lo & 3)];
            if (lo + 1 >= 0 && lo + 1 < nq) whi = base[(uint32_t)((lo + 1) >> 2) * 20u + (uint32_t)((lo + 1) & 3)];
            lds.eq[(r * 64u + lane) * (uint32_t)W + (uint32_t)k] = __builtin_amdgcn_alignbit(whi, wlo, sh);
        }
        lds.eq[(5u * 64u + lane) * (uint32_t)W + (uint32_t)k] = 0u;
    }
    wave_lds_sync();
}

// Every bin of the plan, one part per wave.
template <int W>
__global__ __launch_bounds__(64 * (int)kSplitWaves) void verify_split_kernel(myers_verify_args_t a,
                                                                             myers_split_plan_t p) {
    __shared__ __attribute__((aligned(16))) SplitLds<W> split_lds[kSplitWaves];
    const uint32_t lane = threadIdx.x & 63u;
    SplitLds<W> &lds = split_lds[__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))];
    uint32_t *counter = a.queue_heads + MYERS_SPLIT_HEAD;
    set_wave_prio<64>();
    // one bin of one part per candidate needs no ranges and no counter: each wave
    // takes every (waves of the grid)th candidate
    const bool plain = a.bin_ranges == nullptr;
    uint32_t next = blockIdx.x * kSplitWaves + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t total = 0;                                 // boundaries of the launch
    for (uint32_t j = 0; j < p.n && !plain; j++) total += a.bin_ranges[2u * p.variant[j] + 1u] * (p.parts[j] - 1u);
    for (;;) {
        uint32_t got = next;
        next += gridDim.x * kSplitWaves;
        if (!plain && lane == 0u) got = atomicAdd(counter, 1u);
        const uint32_t item = (uint32_t)__builtin_amdgcn_readfirstlane((int)got);
        uint32_t base = 0, bound = 0, start = a.start, count = a.count, parts = 1;
        bool found = plain && item < count;
        for (uint32_t j = 0; j < p.n && !found && !plain; j++) {
            start = a.bin_ranges[2u * p.variant[j]];
            count = a.bin_ranges[2u * p.variant[j] + 1u];
            parts = p.parts[j];
            found = item - base < count * parts;
            if (!found) {
                base += count * parts;
                bound += count * (parts - 1u);
            }
        }
        if (!found) break;                              // every bin drained: each wave exits here
        const uint32_t ci = (item - base) / parts, part = (item - base) - ci * parts;
        const bool top = part + 1u == parts;
        // the boundaries above and below this part
        const uint32_t above = bound + ci * (parts - 1u) + part, below = above - 1u;
        const uint32_t slot_above = above % p.nslots, slot_below = below % p.nslots;
        // every lane reads the same candidate: all values below are uniform
        const uint32_t cand = a.order ? a.order[start + ci] : start + ci;
        const CandRec cr = static_cast<const CandRec *>(a.cands)[cand];
        SplitCand c = {0ull, 0u, 0u, 0u};
        bool live = false;
        if (cr.query < a.num_queries) {
            const uint2 qi = reinterpret_cast<const uint2 *>(a.qinfo)[cr.query];
            c.entry = qi.x;
            c.m = qi.y;
            const uint32_t n = window_len(c.m, a.distance);
            // skip rule: src-api/coreMyersGPU-CC35.cu:142
            live = c.m <= parts * 2048u * (uint32_t)W &&
                   (uint64_t)qi.x + ((qi.y + 127u) >> 7) <= (uint64_t)a.num_peq_entries && cr.position < a.ref_size &&
                   a.ref_size - cr.position > (uint64_t)n;
            // aligned window (src-api/coreMyersGPU-CC35.cu:132,144) or exact start
            c.nib0 = a.mode == 0 ? (cr.position & ~7ull) : cr.position;
            c.ncols = a.mode == 0 ? 8u * ((n >> 3) + ((n & 7u) ? 2u : 1u)) : n;
            // (the slots are as large as the longest read of a bin needs)
            live = live && 2u * ((c.ncols + parts + 63u) >> 6) <= p.stride;
        }
        c.entry = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.entry);
        c.m = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.m);
        c.ncols = (uint32_t)__builtin_amdgcn_readfirstlane((int)c.ncols);
        // the slot below is this part's when its earlier readers are done
        if (part != 0u) split_wait_done(p.done + slot_below, below / p.nslots);
        uint2 r = make_uint2(0u, kSkipScore);
        if (live) {
            split_stage<W>(a, c, part, parts, lds);
            const uint32_t *eq_lane = lds.eq + lane * (uint32_t)W;
            uint64_t *in = p.pool + (size_t)slot_below * p.stride, *out = p.pool + (size_t)slot_above * p.stride;
            const uint32_t ahead = parts - 1u - part;
            if (!top) split_wait_done(p.done + slot_above, above / p.nslots);
            if (part == 0u) {
                if (top) r = split_columns<W, false, false>(a, c, ahead, eq_lane, in, out);
                else split_columns<W, false, true>(a, c, ahead, eq_lane, in, out);
            } else if (top) {
                r = split_columns<W, true, false>(a, c, ahead, eq_lane, in, out);
            } else {
                split_columns<W, true, true>(a, c, ahead, eq_lane, in, out);
            }
        }
        // the boundary below has been read, its words are zero again; the slot's
        // last reader of the launch leaves the count at zero too
        if (part != 0u && lane == 0u) {
            const uint32_t times = below + p.nslots >= total ? 0u : below / p.nslots + 1u;
            __hip_atomic_store(p.done + slot_below, times, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (top && lane == 0u) {
            if (live && a.threshold >= 0.0f && r.y > threshold_of(c.m, a.threshold)) r = make_uint2(kNoMatch, kNoMatch);
            static_cast<uint2 *>(a.results)[cand] = r;
        }
    }
}

}  // namespace

extern "C" int myers_launch_split(const myers_verify_args_t *args, const myers_split_plan_t *plan, uint32_t words,
                                  uint32_t grid, hipStream_t stream) {
    if (args == nullptr || plan == nullptr || grid == 0 || plan->n == 0 || plan->n > (uint32_t)MYERS_QUEUE_MAX ||
        (words != 1u && words != 2u && words != 4u) || (plan->pool == nullptr) != (plan->done == nullptr) ||
        plan->nslots < (uint32_t)MYERS_SPLIT_MIN_SLOTS || plan->nslots > (uint32_t)MYERS_SPLIT_MAX_SLOTS ||
        plan->stride == 0 || (uint64_t)plan->nslots * plan->stride * 2u > (uint64_t)MYERS_SPLIT_POOL_WORDS)
        return -1;
    if (args->bin_ranges == nullptr ? plan->n != 1u || plan->parts[0] != 1u : args->queue_heads == nullptr) return -1;
    for (uint32_t j = 0; j < plan->n; j++) {
        myers_variant_desc_t d;
        if (myers_variant_desc(plan->variant[j], &d) != 0 || plan->parts[j] * 64u * words < d.total_words ||
            plan->parts[j] >= (uint32_t)MYERS_SPLIT_MIN_SLOTS || (plan->parts[j] > 1u && plan->pool == nullptr))
            return -1;
    }
    const void *k = words == 1u   ? reinterpret_cast<const void *>(&verify_split_kernel<1>)
                    : words == 2u ? reinterpret_cast<const void *>(&verify_split_kernel<2>)
                                  : reinterpret_cast<const void *>(&verify_split_kernel<4>);
    void *kargs[] = {const_cast<myers_verify_args_t *>(args), const_cast<myers_split_plan_t *>(plan)};
    return (int)hipLaunchKernel(k, dim3(grid), dim3(64u * kSplitWaves), kargs, 0, stream);
}
