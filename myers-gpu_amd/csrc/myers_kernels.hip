// Multi-lane and multi-wave verification kernels, binning and the launch shims
// (the column recurrence and the one-wave chunk loop are in myers_device.h,
// reads of up to 1024 bases in myers_slice.hip, the resident serving kernel in
// myers_serve_kernel.hip).
#include "myers_device.h"

namespace {

// Plain launch: a fixed grid strides over the chunks of one slot range.
template <int L, int W, bool kCut>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWavesPerEU<L, W, kCut, false>)))
void verify_kernel(myers_verify_args_t a) {
    using S = Shape<L, W>;
    __shared__ Workspace<L, W> ws;
    set_wave_prio<L>();
    uint32_t start = a.start, count = a.count;
    if (a.bin_ranges != nullptr) {
        start = a.bin_ranges[2 * a.variant];
        count = a.bin_ranges[2 * a.variant + 1];
    }
    const uint32_t nchunks = (count + S::kSlots - 1) / S::kSlots;
    zero_row_init<L, W>(ws);
    // Workgroups are dispatched round-robin over the 8 XCDs; renumber them so
    // that each XCD (own L2) takes a contiguous run of chunks, which keeps the
    // candidates of one query -- and their Peq -- in one L2.
    uint32_t first = blockIdx.x;
    if ((gridDim.x & 7u) == 0u) first = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    verify_chunks<L, W, kCut>(a, start, count, first, nchunks, gridDim.x, ws);
}

// Persistent launch: a resident grid pulls ranges of chunks (at least
// `chunk_factor`) from the variant's device queue (part heads reset by the
// binning) until the bin is drained; every wave reaches the exit test.
template <int L, int W, bool kCut>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWavesPerEU<L, W, kCut, true>)))
void verify_persistent_kernel(myers_verify_args_t a) {
    using S = Shape<L, W>;
    __shared__ Workspace<L, W> ws;
    __shared__ uint32_t item_sh, item_hi_sh;
    const uint32_t start = a.bin_ranges[2 * a.variant];
    const uint32_t count = a.bin_ranges[2 * a.variant + 1];
    const uint32_t nchunks = (count + S::kSlots - 1) / S::kSlots;
    const uint32_t cf = a.chunk_factor ? a.chunk_factor : 1u;
    uint32_t *heads = a.queue_heads + a.variant * (uint32_t)(MYERS_QUEUE_PARTS * MYERS_QUEUE_STRIDE);
    uint32_t part = 0;
    if (blockIdx.x >= nchunks) return;      // more workgroups than chunks: the others cover them
    set_wave_prio<L>();
    zero_row_init<L, W>(ws);
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t lo = 0, hi = 0;
            if (!pull_work(heads, nchunks, cf, part, lo, hi)) lo = hi = 0xFFFFFFFFu;
            item_sh = lo;
            item_hi_sh = hi;
        }
        __syncthreads();
        const uint32_t lo = __builtin_amdgcn_readfirstlane(item_sh);
        const uint32_t hi = __builtin_amdgcn_readfirstlane(item_hi_sh);
        if (lo == 0xFFFFFFFFu) break;
        verify_chunks<L, W, kCut>(a, start, count, lo, hi, 1u, ws);
    }
}

// ------------------------------------------------- multi-wave candidates
// A wave issues one instruction every few clocks, so the time of one long
// candidate grows with the steps times the words each lane carries: a
// 20,000-base read on one wave (64 lanes x 10 words) takes ~5-10 ms.  For
// latency, a candidate can span Q waves of one workgroup (64Q lanes, W words
// each).  Lanes run diagonally as in one wave (lane d computes column t - d);
// at a wave boundary the bottom lane's hin is the top lane of the wave below,
// passed through LDS: wave q runs kWaveLag steps behind wave q-1 on top of the
// per-lane lag, each wave's top lane packs its (Ph, Mh) top bits of a block
// of 8 steps into one word of an LDS ring, and one barrier per block orders
// writes and reads.  Every wave runs the same number of blocks.

constexpr uint32_t kWaveLag = 8;
constexpr uint32_t kRingWords = 4;

template <int Q, int W>
struct WideShape {
    static constexpr int kLanes = 64 * Q;               // lanes per candidate
    static constexpr int kGroups = (W + 3) / 4;
    static constexpr int kTotal = kLanes * W;           // words per candidate
    static constexpr int kRows = 6;                     // A C G T N + zero row
    static constexpr int kRowU4 = kLanes;
    static constexpr int kLdsU4 = kGroups * kRows * kRowU4;
    static constexpr uint32_t kMaxLag = (uint32_t)kLanes - 1u + kWaveLag * (uint32_t)(Q - 1);
};

template <int Q, int W>
struct WideWorkspace {
    uint4 lds[WideShape<Q, W>::kLdsU4];
    uint32_t ring[Q - 1][kRingWords];
};

// Peq of one read, top-justified, transposed for 64Q lanes (the layout of
// stage_peq with one slot).
template <int Q, int W>
__device__ __forceinline__ void stage_peq_wide(uint4 *lds, uint2 qi, const uint32_t *__restrict__ peq,
                                               uint32_t tid) {
    using S = WideShape<Q, W>;
    uint32_t *l32 = reinterpret_cast<uint32_t *>(lds);
    const int32_t pad = 32 * S::kTotal - (int32_t)qi.y;
    const int32_t nq = (int32_t)((qi.y + 31u) >> 5);
    for (uint32_t idx = tid; idx < 5u * (uint32_t)S::kTotal; idx += (uint32_t)S::kLanes) {
        const uint32_t gw = idx % (uint32_t)S::kTotal;
        const uint32_t c = idx / (uint32_t)S::kTotal;
        const int32_t b0 = 32 * (int32_t)gw - pad;
        const int32_t lo = b0 >> 5;
        const uint32_t sh = (uint32_t)b0 & 31u;
        const uint32_t *base = peq + (size_t)qi.x * 20u + 4u * c;
        uint32_t wlo = 0, whi = 0;
        if (lo >= 0 && lo < nq) wlo = base[(uint32_t)(lo >> 2) * 20u + (uint32_t)(lo & 3)];
        if (lo + 1 >= 0 && lo + 1 < nq) whi = base[(uint32_t)((lo + 1) >> 2) * 20u + (uint32_t)((lo + 1) & 3)];
        const uint32_t k = gw % (uint32_t)W, gl = gw / (uint32_t)W;
        const uint32_t u4 = ((k >> 2) * (uint32_t)S::kRows + c) * (uint32_t)S::kRowU4 + gl;
        l32[u4 * 4u + (k & 3u)] = (uint32_t)((((uint64_t)whi << 32) | wlo) >> sh);
    }
}

// One candidate's columns on wave wq of its workgroup (Q > 1).  A wave's
// role is fixed for the whole loop, so each role is its own instantiation:
// kBelow -- lane 0's hin is the top lane of the wave below, read from the LDS
// ring; kAbove -- this wave's top lane feeds the wave above; kTop -- the top
// wave keeps the score row.  Ring word of block b: the top lane's Ph bit 31
// of step 8b+i at bit i, its Mh bit 31 at bit 8+i.  Returns {min_col,
// min_score}, meaningful on lane 63 of the top wave.
template <int Q, int W, bool kBelow, bool kAbove, bool kTop>
__device__ __forceinline__ uint2 wide_columns(WideWorkspace<Q, W> &ws, uint32_t wq, uint32_t tid,
                                              const uint32_t *__restrict__ ref, int32_t last_word,
                                              uint64_t nib0, uint32_t lag, uint32_t ncols, uint32_t m) {
    using S = WideShape<Q, W>;
    constexpr uint32_t kGS = (uint32_t)(S::kRows * S::kRowU4);
    const uint32_t lane = tid & 63u;
    const uint4 *lds_lane = ws.lds + tid;
    const uint32_t nblocks = (ncols + S::kMaxLag + 7u) >> 3;
    const int64_t qn = (int64_t)nib0 - (int64_t)lag;
    const int32_t w0 = (int32_t)(qn >> 3);
    const uint32_t shift = (uint32_t)(qn & 7) * 4u;

    uint32_t Pv[W], Mv[W];
#pragma unroll
    for (int k = 0; k < W; k++) {
        Pv[k] = ~0u;
        Mv[k] = 0u;
    }
    // Score row and its first minimum.  Before its first column the top lane
    // keeps its initial state (every lane below it is before its own first
    // column too), so the score stays m and those steps never win; only the
    // last block can reach columns past the window and checks them.  Windows
    // of at most 65,536 columns keep the minimum as one key, (score << 16) |
    // column (score <= m <= 24,576): the smaller key is the smaller score, then
    // the earlier column; a column past the window is masked to all ones.
    int32_t score = (int32_t)m, min_score = (int32_t)m;
    uint32_t min_col = 0, min_key = m << 16;
    uint32_t ph_top = 0, mh_top = 0, acc_p = 0, acc_m = 0;
    auto text_word = [&](int32_t k) { return ref[min(max(w0 + k, 0), last_word)]; };
    auto text_block = [&](uint32_t lo, uint32_t hi, uint32_t b) {
        uint32_t t = sanitize_text(__builtin_amdgcn_alignbit(hi, lo, shift));
        // steps before this lane's first column read the zero row
        const int32_t early = (int32_t)lag - 8 * (int32_t)b;
        if (early > 0) {
            const uint32_t low = early >= 8 ? ~0u : ((1u << (4 * early)) - 1u);
            t = (t & ~low) | (0x55555555u & low);
        }
        return t;
    };
    const uint32_t tw0 = text_word(0);
    const uint32_t tw1 = text_word(1);
    uint32_t tw2 = text_word(2);
    uint32_t tw3 = text_word(3);
    uint32_t text = text_block(tw0, tw1, 0);
    uint32_t text_next = text_block(tw1, tw2, 1);
    uint32_t cur_off = (text & 7u) * (uint32_t)S::kRowU4;
    uint4 eq4 = lds_lane[cur_off];
    auto block = [&](uint32_t b, auto last, auto keyed) {
        constexpr bool kLast = decltype(last)::value;
        constexpr bool kKeyed = decltype(keyed)::value;
        const uint32_t tw4 = text_word((int32_t)b + 4);
        // ring words of the wave below: its top lane's steps 8b-9 .. 8b-2,
        // written in blocks b-2 and b-1 (the same value in every lane)
        uint32_t w1 = 0, w2 = 0;
        if constexpr (kBelow) {
            if (b >= 1u) w1 = ws.ring[wq - 1u][(b - 1u) % kRingWords];
            if (b >= 2u) w2 = ws.ring[wq - 1u][(b - 2u) % kRingWords];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t cn = (i < 7) ? ((text >> (4 * (i + 1))) & 7u) : (text_next & 7u);
            const uint32_t next_off = cn * (uint32_t)S::kRowU4;
            const uint4 eq4n = lds_lane[next_off];
            // hin from the lane below (DPP wave_shr:1); lane 0 keeps the fill:
            // 0 on the bottom wave, else the wave below's bit of step 8b+i-9
            // moved to bit 31 (only bit 31 of a hin is read)
            uint32_t fill_p = 0u, fill_m = 0u;
            if constexpr (kBelow) {
                fill_p = i == 0 ? (w2 << 24) : (w1 << (32 - i));
                fill_m = i == 0 ? (w2 << 16) : (w1 << (24 - i));
            }
            const uint32_t ph_in = (uint32_t)__builtin_amdgcn_update_dpp((int)fill_p, (int)ph_top, 0x138, 0xF, 0xF, false);
            const uint32_t mh_in = (uint32_t)__builtin_amdgcn_update_dpp((int)fill_m, (int)mh_top, 0x138, 0xF, 0xF, false);
            column_grp<W, true, kGS, false>(Pv, Mv, eq4, lds_lane, cur_off, ph_in, mh_in, ph_top, mh_top);
            eq4 = eq4n;
            if constexpr (kAbove) {
                acc_p = (acc_p >> 1) | (ph_top & 0x80000000u);
                acc_m = (acc_m >> 1) | (mh_top & 0x80000000u);
            }
            if constexpr (kTop) {
                // score row: the top lane of the top wave, at column t - kMaxLag
                score += (int32_t)(ph_top >> 31) - (int32_t)(mh_top >> 31);
                const uint32_t col = 8u * b + (uint32_t)i - S::kMaxLag;
                if constexpr (kKeyed) {
                    const uint32_t c = kLast ? (col < ncols ? col : ~0u) : col;
                    min_key = min(min_key, ((uint32_t)score << 16) | c);
                } else {
                    const bool better = kLast ? (score < min_score) && (col < ncols) : (score < min_score);
                    min_col = better ? col : min_col;
                    min_score = better ? score : min_score;
                }
            }
            cur_off = next_off;
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kAbove) {
            if (lane == 63u) ws.ring[wq][b % kRingWords] = (acc_p >> 24) | ((acc_m >> 16) & 0xFF00u);
        }
        __syncthreads();
        text = text_next;
        text_next = text_block(tw2, tw3, b + 2);
        tw2 = tw3;
        tw3 = tw4;
    };
    auto run = [&](auto keyed) {
        for (uint32_t b = 0; b + 1u < nblocks; b++) block(b, std::false_type{}, keyed);
        if (nblocks) block(nblocks - 1u, std::true_type{}, keyed);
    };
    if (kTop && ncols <= 0x10000u) {
        run(std::true_type{});
        return make_uint2(min_key & 0xFFFFu, min_key >> 16);
    }
    run(std::false_type{});
    return make_uint2(min_col, (uint32_t)min_score);
}

// Candidates cand_lo, cand_lo + stride, ... < cand_hi of the slot range
// [start, start + count), one per workgroup at a time.
template <int Q, int W>
__device__ __forceinline__ void verify_wide(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                            uint32_t cand_lo, uint32_t cand_hi, uint32_t stride,
                                            WideWorkspace<Q, W> &ws, uint32_t &staged_query) {
    using S = WideShape<Q, W>;
    const uint32_t tid = threadIdx.x;
    const uint32_t wq = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave of the workgroup
    const uint32_t lag = tid + kWaveLag * wq;                      // this lane's column lag
    const uint32_t *__restrict__ ref = a.ref;
    const int32_t last_word = (int32_t)(a.ref_words - 1);
    const CandRec *__restrict__ cands = static_cast<const CandRec *>(a.cands);
    const uint2 *__restrict__ qinfo = reinterpret_cast<const uint2 *>(a.qinfo);
    uint2 *__restrict__ results = static_cast<uint2 *>(a.results);

    for (uint32_t ci = cand_lo; ci < cand_hi && ci < count; ci += stride) {
        // every lane reads the same candidate: all values below are uniform
        const uint32_t cand = a.order ? a.order[start + ci] : start + ci;
        const CandRec cr = cands[cand];
        uint32_t m = 0, pos_entry = 0;
        bool sane = false;
        if (cr.query < a.num_queries) {
            const uint2 qi = qinfo[cr.query];
            pos_entry = qi.x;
            m = qi.y;
            sane = m <= 32u * S::kTotal && (uint64_t)pos_entry + ((m + 127u) >> 7) <= (uint64_t)a.num_peq_entries;
        }
        if (!sane) m = 0;
        const uint32_t n = window_len(m, a.distance);
        const bool live = sane && cr.position < a.ref_size && (a.ref_size - cr.position) > (uint64_t)n;
        if (!live) {
            if (tid == 0u) results[cand] = make_uint2(0u, kSkipScore);
            continue;
        }
        uint64_t nib0;
        uint32_t ncols;
        if (a.mode == 0) {
            nib0 = cr.position & ~7ull;
            ncols = 8u * ((n >> 3) + ((n & 7u) ? 2u : 1u));
        } else {
            nib0 = cr.position;
            ncols = n;
        }
        // consecutive candidates of one read keep its Peq in LDS
        if (cr.query != staged_query) {
            __syncthreads();
            stage_peq_wide<Q, W>(ws.lds, make_uint2(pos_entry, m), a.peq, tid);
            __syncthreads();
            staged_query = cr.query;
        }
        uint2 r;
        if (wq == 0u) {
            r = wide_columns<Q, W, false, true, false>(ws, wq, tid, ref, last_word, nib0, lag, ncols, m);
        } else if (wq + 1u < (uint32_t)Q) {
            r = wide_columns<Q, W, true, true, false>(ws, wq, tid, ref, last_word, nib0, lag, ncols, m);
        } else {
            r = wide_columns<Q, W, true, false, true>(ws, wq, tid, ref, last_word, nib0, lag, ncols, m);
        }
        if (tid == (uint32_t)S::kLanes - 1u) {
            if (a.threshold >= 0.0f && r.y > threshold_of(m, a.threshold)) r = make_uint2(kNoMatch, kNoMatch);
            results[cand] = r;
        }
    }
}

template <int Q, int W>
__device__ __forceinline__ void zero_row_init_wide(WideWorkspace<Q, W> &ws) {
    using S = WideShape<Q, W>;
    uint32_t *l32 = reinterpret_cast<uint32_t *>(ws.lds);
    for (uint32_t i = threadIdx.x; i < (uint32_t)(S::kGroups * S::kRowU4 * 4); i += (uint32_t)S::kLanes) {
        const uint32_t u4 = i >> 2, g = u4 / S::kRowU4, r = u4 % S::kRowU4;
        l32[((g * S::kRows + kZeroRow) * S::kRowU4 + r) * 4u + (i & 3u)] = 0u;
    }
    __syncthreads();
}

template <int Q, int W>
__global__ __launch_bounds__(64 * Q) void verify_wide_kernel(myers_verify_args_t a) {
    __shared__ WideWorkspace<Q, W> ws;
    uint32_t start = a.start, count = a.count;
    if (a.bin_ranges != nullptr) {
        start = a.bin_ranges[2 * a.variant];
        count = a.bin_ranges[2 * a.variant + 1];
    }
    set_wave_prio<64 * Q>();
    zero_row_init_wide<Q, W>(ws);
    uint32_t first = blockIdx.x;
    if ((gridDim.x & 7u) == 0u) first = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    uint32_t staged = 0xFFFFFFFFu;
    verify_wide<Q, W>(a, start, count, first, count, gridDim.x, ws, staged);
}

template <int Q, int W>
__global__ __launch_bounds__(64 * Q) void verify_wide_persistent_kernel(myers_verify_args_t a) {
    __shared__ WideWorkspace<Q, W> ws;
    __shared__ uint32_t item_sh, item_hi_sh;
    const uint32_t start = a.bin_ranges[2 * a.variant];
    const uint32_t count = a.bin_ranges[2 * a.variant + 1];
    const uint32_t cf = a.chunk_factor ? a.chunk_factor : 1u;
    uint32_t *heads = a.queue_heads + a.variant * (uint32_t)(MYERS_QUEUE_PARTS * MYERS_QUEUE_STRIDE);
    uint32_t part = 0;
    if (blockIdx.x >= count) return;        // more workgroups than candidates: the others cover them
    set_wave_prio<64 * Q>();
    zero_row_init_wide<Q, W>(ws);
    uint32_t staged = 0xFFFFFFFFu;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t lo = 0, hi = 0;
            if (!pull_work(heads, count, cf, part, lo, hi)) lo = hi = 0xFFFFFFFFu;
            item_sh = lo;
            item_hi_sh = hi;
        }
        __syncthreads();
        const uint32_t lo = __builtin_amdgcn_readfirstlane(item_sh);
        const uint32_t hi = __builtin_amdgcn_readfirstlane(item_hi_sh);
        if (lo == 0xFFFFFFFFu) break;
        verify_wide<Q, W>(a, start, count, lo, hi, 1u, ws, staged);
    }
}

// ------------------------------------------------- long-read bins, one launch
// A bin of long reads holds few candidates, and each takes one chain of
// dependent column steps: its time is the chain, not the chip's throughput.
// Separate launches per bin stack such waves on shared SIMDs, where they
// slow each other.  One launch of MYERS_LONG_WAVES-wave workgroups (the
// waves of a workgroup sit on different SIMDs of one CU) runs all of them:
// each wave pulls the next chunk from one counter over the bins in plan
// order, longest reads first, so the longest chains start first and a SIMD
// holds one long chain at a time.
#define MYERS_LONG_CASE(L, W)                                                                    \
    case ((L) << 8) | (W):                                                                       \
        if constexpr ((L) >= 4 && (L) <= 64) {                                                   \
            auto &w = *reinterpret_cast<Workspace<(L), (W)> *>(ws);                              \
            if (prepared != j) {                                                                 \
                zero_row_init<(L), (W), MYERS_LONG_WAVES>(w);                                    \
                prepared = j;                                                                    \
            }                                                                                    \
            verify_chunks<(L), (W), false, MYERS_LONG_WAVES>(a, start, count, chunk, chunk + 1u, 1u, w); \
        }                                                                                        \
        break;

using LongWide = WideWorkspace<MYERS_LONG_WAVES, MYERS_WIDE_MAX_WORDS>;
static_assert(sizeof(WideWorkspace<MYERS_LONG_WAVES, 2>) == sizeof(LongWide) &&
                  WideShape<MYERS_LONG_WAVES, 2>::kGroups == WideShape<MYERS_LONG_WAVES, 3>::kGroups,
              "wide candidates of 2 and 3 words share one LDS layout");

__global__ __launch_bounds__(64 * MYERS_LONG_WAVES) void verify_long_kernel(myers_verify_args_t a,
                                                                           myers_long_plan_t p) {
    extern __shared__ uint4 long_lds[];
    __shared__ uint32_t wide_item_sh;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;
    set_wave_prio<64>();
    // Phase 1: the wide bins, one candidate per workgroup (longest reads).
    if (p.n_wide) {
        LongWide &wws = *reinterpret_cast<LongWide *>(long_lds);
        zero_row_init_wide<MYERS_LONG_WAVES, MYERS_WIDE_MAX_WORDS>(wws);
        uint32_t staged = 0xFFFFFFFFu;
        const uint32_t grid = gridDim.x;
        uint32_t witem = (blockIdx.x + grid - (p.rotate / (uint32_t)MYERS_LONG_WAVES) % grid) % grid;
        for (bool first = true;; first = false) {
            if (!first) {
                if (threadIdx.x == 0) wide_item_sh = atomicAdd(a.queue_heads + MYERS_WIDE_HEAD, 1u);
                __syncthreads();
                witem = grid + (uint32_t)__builtin_amdgcn_readfirstlane((int)wide_item_sh);
                __syncthreads();                 // every wave has read it before the next pull
            }
            uint32_t j = 0, base = 0, start = 0, count = 0;
            bool found = false;
            for (; j < p.n_wide; j++) {
                const uint32_t v = p.wide_variant[j];
                const uint32_t c = a.bin_ranges[2u * v + 1u];
                if (witem - base < c) {
                    start = a.bin_ranges[2u * v];
                    count = c;
                    found = true;
                    break;
                }
                base += c;
            }
            if (!found) break;                   // every wide bin drained
            const uint32_t slot = witem - base;
            if (p.wide_words[j] == 2u) {
                verify_wide<MYERS_LONG_WAVES, 2>(a, start, count, slot, slot + 1u, 1u,
                                                 *reinterpret_cast<WideWorkspace<MYERS_LONG_WAVES, 2> *>(long_lds),
                                                 staged);
            } else {
                verify_wide<MYERS_LONG_WAVES, 3>(a, start, count, slot, slot + 1u, 1u, wws, staged);
            }
        }
        __syncthreads();                         // phase 2 reuses the LDS
    }
    // Phase 2: the other bins, one chunk per wave.  The first round gives one
    // item to each wave free at the start -- past the workgroups that took a
    // wide candidate in phase 1's first round (from workgroup rotate / waves
    // on) -- so that the longest of these items start at once; later items
    // are pulled from the counter.
    uint4 *ws = long_lds + wave * p.ws_u4;
    uint32_t *counter = a.queue_heads + MYERS_LONG_HEAD;
    uint32_t prepared = 0xFFFFFFFFu;
    uint32_t wide_first = 0;
    for (uint32_t j = 0; j < p.n_wide; j++) wide_first += a.bin_ranges[2u * p.wide_variant[j] + 1u];
    wide_first = min(wide_first, gridDim.x);
    const uint32_t nw = gridDim.x * (uint32_t)MYERS_LONG_WAVES;
    const uint32_t free_waves = nw - wide_first * (uint32_t)MYERS_LONG_WAVES;
    const uint32_t slot = blockIdx.x * (uint32_t)MYERS_LONG_WAVES + wave;
    const uint32_t rel = (slot + nw - (p.rotate + wide_first * (uint32_t)MYERS_LONG_WAVES) % nw) % nw;
    uint32_t item = rel;
    for (bool first = rel < free_waves;; first = false) {
        if (!first) {
            uint32_t got = 0;
            if (lane == 0u) got = atomicAdd(counter, 1u);
            item = free_waves + (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)got, 0));
        }
        uint32_t j = 0, base = 0, start = 0, count = 0;
        bool found = false;
        for (; j < p.n; j++) {
            const uint32_t v = p.variant[j];
            const uint32_t c = a.bin_ranges[2u * v + 1u];
            const uint32_t slots = 64u / (p.key[j] >> 8);
            const uint32_t chunks = (c + slots - 1u) / slots;
            if (item - base < chunks) {
                start = a.bin_ranges[2u * v];
                count = c;
                found = true;
                break;
            }
            base += chunks;
        }
        if (!found) break;                       // every bin drained
        const uint32_t chunk = item - base;
        switch (p.key[j]) {
            MYERS_VARIANT_LIST(MYERS_LONG_CASE)
            default:
                break;
        }
    }
}

// ------------------------------------------------- one launch over all bins
// The queue launch of the multi-lane bins: a resident grid of two-wave
// workgroups takes one pair of chunks at a time from a single counter over
// the bins in plan order (the host orders them longest reads first, so the
// grid's tail is short chunks), and runs it with its bin's variant.  No launch
// boundary separates the bins: a workgroup that finishes the last pair of one
// bin takes the next bin's first.
constexpr int kQueueWaves = 2;

#define MYERS_QUEUE_CASE(L, W)                                                                   \
    case ((L) << 8) | (W):                                                                       \
        if constexpr (kQueueClass<(L), (W)> == MYERS_QUEUE_MULTI_LANE) {                                    \
            auto &w = *reinterpret_cast<Workspace<(L), (W)> *>(queue_lds + kXchgU4);             \
            if (prepared != key) {                                                               \
                set_wave_prio<(L)>();                                                            \
                zero_row_init<(L), (W), 1, 64u * kShare>(w);                                     \
                prepared = key;                                                                  \
            }                                                                                    \
            verify_chunks<(L), (W), kCut && kHasCut<(L), (W)>, 1, false, kShare>(a, start, count, chunk, \
                                                                                 chunk + 1u, 1u, w, xchg); \
        }                                                                                        \
        break;

template <bool kCut>
__global__ __launch_bounds__(64 * kQueueWaves) __attribute__((amdgpu_waves_per_eu(3)))
void verify_queue_kernel(myers_verify_args_t a, myers_queue_plan_t p) {
    extern __shared__ uint4 queue_lds[];
    // The waves of a workgroup share one workspace (verify_chunks, kShare = 2),
    // after one uint4 of hand-over words; the item counter counts chunk pairs.
    constexpr int kShare = kQueueWaves;
    constexpr uint32_t kXchgU4 = 1u;
    uint32_t *xchg = reinterpret_cast<uint32_t *>(queue_lds);
    uint32_t *counter = a.queue_heads + MYERS_QUEUE_HEAD(MYERS_QUEUE_MULTI_LANE);
    uint32_t prepared = 0xFFFFFFFFu;
    for (;;) {
        if (threadIdx.x == 0) xchg[3] = atomicAdd(counter, 1u);
        __syncthreads();
        const uint32_t item = __builtin_amdgcn_readfirstlane(xchg[3]);
        __syncthreads();                         // read by all before the next claim
        uint32_t j = 0, base = 0, start = 0, count = 0;
        bool found = false;
        for (; j < p.n; j++) {
            const uint32_t v = p.variant[j];
            const uint32_t c = a.bin_ranges[2u * v + 1u];
            const uint32_t slots = 64u / (p.key[j] >> 8);
            const uint32_t chunks = (c + slots * (uint32_t)kShare - 1u) / (slots * (uint32_t)kShare);
            if (item - base < chunks) {
                start = a.bin_ranges[2u * v];
                count = c;
                found = true;
                break;
            }
            base += chunks;
        }
        if (!found) break;                       // every bin drained: each wave exits here
        const uint32_t chunk = item - base;
        const uint32_t key = p.key[j];
        switch (key) {
            MYERS_VARIANT_LIST(MYERS_QUEUE_CASE)
            default:
                break;
        }
    }
}

// ---------------------------------------------------------------- binning

constexpr uint32_t kTooLong = 0xFFFFFFFFu;
constexpr uint32_t kBadQuery = 0xFFFFFFFEu;

__device__ __forceinline__ uint32_t variant_of(const uint2 *qinfo, uint32_t num_queries, const CandRec *cands,
                                               uint32_t i, const uint8_t *bin_of_words, uint32_t max_words) {
    const uint32_t q = cands[i].query;
    if (q >= num_queries) return kBadQuery;
    const uint32_t w = (qinfo[q].y + 31u) >> 5;
    return w <= max_words ? (uint32_t)bin_of_words[w] : kTooLong;
}

// Binning is a stable partition of the candidates by variant with no global
// atomics: block b of the count and scatter kernels owns the contiguous span
// [b*span, (b+1)*span); bin_count writes each block's per-variant counts
// (variant-major, and behind them the errors it met), bin_scan (one block per
// variant, one for the errors) turns them into each block's first slot within
// the variant, and bin_scatter lays the variants' ranges end to end (every block
// for itself; the first one writes them down) and writes every candidate's id at
// its slot in input order.  A read's candidates, adjacent in the input, stay
// adjacent in their bin.  Three launches: with the ranges, a reset of the error
// word and its copy to the host as launches of their own, a binned batch took
// 25 us longer.

__device__ __forceinline__ uint32_t bin_span(uint32_t n) {
    const uint32_t span = (n + gridDim.x - 1u) / gridDim.x;
    return (span + 255u) & ~255u;
}

__global__ __launch_bounds__(256) void bin_count_kernel(const uint2 *qinfo, uint32_t num_queries,
                                                        const CandRec *cands,
                                                        uint32_t n, const uint8_t *bin_of_words,
                                                        uint32_t max_words, uint32_t nv,
                                                        uint32_t *block_counts) {
    __shared__ uint32_t hist[MYERS_MAX_VARIANTS];      // and the errors at nv
    for (uint32_t i = threadIdx.x; i <= nv; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    const uint32_t span = bin_span(n);
    const uint32_t lo = blockIdx.x * span, hi = min(n, lo + span);
    for (uint32_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        const uint32_t v = variant_of(qinfo, num_queries, cands, i, bin_of_words, max_words);
        if (v < nv) {
            atomicAdd(&hist[v], 1u);
        } else {
            atomicOr(&hist[nv], v == kBadQuery ? 2u : 1u);
        }
    }
    __syncthreads();
    for (uint32_t v = threadIdx.x; v <= nv; v += blockDim.x) block_counts[v * gridDim.x + blockIdx.x] = hist[v];
}

// One block of 256 threads per variant: an exclusive scan of the variant's
// per-block counts (16 consecutive blocks per thread, then a scan of the 256
// thread sums), in place, giving each count block's first slot relative to
// the variant's range; the variant's total goes to ranges[2v+1].  The last
// block joins the errors, for the host to read (host memory).
__global__ __launch_bounds__(256) void bin_scan_kernel(uint32_t *block_counts, uint32_t nblocks,
                                                       uint32_t *ranges, uint32_t *host_err) {
    __shared__ uint32_t part[256];
    const uint32_t t = threadIdx.x, v = blockIdx.x;
    const uint32_t per = (nblocks + 255u) / 256u;
    uint32_t *row = block_counts + v * nblocks;
    if (v + 1u == gridDim.x) {
        uint32_t any = 0;
        for (uint32_t b = t; b < nblocks; b += 256u) any |= row[b];
        any = (__ballot(any & 1u) != 0ull ? 1u : 0u) | (__ballot(any & 2u) != 0ull ? 2u : 0u);
        if ((t & 63u) == 0u) part[t >> 6] = any;
        __syncthreads();
        if (t == 0u)
            __hip_atomic_store(host_err, part[0] | part[1] | part[2] | part[3], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        return;
    }
    uint32_t sum = 0;
    for (uint32_t k = 0; k < per; k++) {
        const uint32_t b = t * per + k;
        if (b < nblocks) sum += row[b];
    }
    part[t] = sum;
    __syncthreads();
    for (uint32_t o = 1; o < 256u; o <<= 1) {       // inclusive scan (Hillis-Steele)
        const uint32_t x = t >= o ? part[t - o] : 0u;
        __syncthreads();
        part[t] += x;
        __syncthreads();
    }
    uint32_t run = part[t] - sum;
    for (uint32_t k = 0; k < per; k++) {
        const uint32_t b = t * per + k;
        if (b < nblocks) {
            const uint32_t c = row[b];
            row[b] = run;
            run += c;
        }
    }
    if (t == 255u) ranges[2 * v + 1] = part[255];
}

// Write each candidate's id at its slot: per 256-candidate round, ranks within
// a wave come from ballots, the waves' counts are added in wave order in LDS,
// and the block's running first slot per variant advances by the round's
// counts.
__global__ __launch_bounds__(256) void bin_scatter_kernel(const uint2 *qinfo, uint32_t num_queries,
                                                          const CandRec *cands,
                                                          uint32_t n, const uint8_t *bin_of_words,
                                                          uint32_t max_words, uint32_t nv,
                                                          const uint32_t *block_first, uint32_t *ranges,
                                                          uint32_t *queue_heads, uint32_t *order, uint2 *results) {
    __shared__ uint32_t next[MYERS_MAX_VARIANTS];
    __shared__ uint32_t wave_cnt[4][MYERS_MAX_VARIANTS];
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    if (wave == 0u) {
        // the variants' ranges from their totals (only the first block writes
        // them, and nothing that the others read)
        const uint32_t total = lane < nv ? ranges[2 * lane + 1] : 0u;
        uint32_t end = total;
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)end, o);
            end += lane >= o ? y : 0u;
        }
        if (lane < nv) next[lane] = end - total + block_first[lane * gridDim.x + blockIdx.x];
        if (blockIdx.x == 0u && lane < nv) {
            ranges[2 * lane] = end - total;
            // empty lists of a second launch
            ranges[MYERS_WORK_LIST + 2 * lane] = end - total;
            ranges[MYERS_WORK_LIST + 2 * lane + 1] = 0u;
        }
        if (blockIdx.x == 0u && lane < 2u) ranges[MYERS_WORK_TALLY + lane] = 0u;
    } else if (blockIdx.x == 0u) {
        // the queues' heads
        const uint32_t t = threadIdx.x - 64u;
        for (uint32_t i = t; i < nv * (uint32_t)MYERS_QUEUE_PARTS; i += 192u)
            queue_heads[i * (uint32_t)MYERS_QUEUE_STRIDE] = 0;
        if (t < (uint32_t)MYERS_QUEUE_PARTS) {
            // one line each, two words used
            queue_heads[MYERS_LONG_HEAD + t * (uint32_t)MYERS_QUEUE_STRIDE] = 0;
            queue_heads[MYERS_LONG_HEAD + t * (uint32_t)MYERS_QUEUE_STRIDE + 1u] = 0;
        }
    }
    __syncthreads();
    const uint32_t span = bin_span(n);
    const uint32_t lo = blockIdx.x * span, hi = min(n, lo + span);
    for (uint32_t r = lo; r < hi; r += 256u) {
        for (uint32_t i = threadIdx.x; i < 4u * nv; i += blockDim.x) wave_cnt[i / nv][i % nv] = 0;
        __syncthreads();
        const uint32_t i = r + threadIdx.x;
        const uint32_t v = i < hi ? variant_of(qinfo, num_queries, cands, i, bin_of_words, max_words) : kTooLong;
        if (i < hi && v >= nv) results[i] = make_uint2(0u, kSkipScore);
        uint32_t rank = 0;
        uint64_t pending = __ballot(v < nv);
        while (pending) {
            const uint32_t leader = (uint32_t)__builtin_ctzll(pending);
            const uint32_t vv = (uint32_t)__shfl((int)v, (int)leader);
            const uint64_t mine = __ballot(v == vv);
            if (v == vv) rank = (uint32_t)__builtin_popcountll(mine & below);
            if (lane == leader) wave_cnt[wave][vv] = (uint32_t)__builtin_popcountll(mine);
            pending &= ~mine;
        }
        __syncthreads();
        if (v < nv) {
            uint32_t slot = next[v] + rank;
            for (uint32_t w = 0; w < wave; w++) slot += wave_cnt[w][v];
            order[slot] = i;
        }
        __syncthreads();
        for (uint32_t vv = threadIdx.x; vv < nv; vv += blockDim.x)
            next[vv] += wave_cnt[0][vv] + wave_cnt[1][vv] + wave_cnt[2][vv] + wave_cnt[3][vv];
        __syncthreads();
    }
}

// ---------------------------------------------------- reads with N together
// A chunk of the sliced kernel takes an eighth operation per 32 cells if one
// of its reads holds an N (and from 27 rows per lane on reads the N plane from
// LDS): 1.34x the time of a chunk without.  Six 1000-base reads to a chunk, N
// in 12% of them, more than half the chunks are such; put together within
// spans of slots, a seventh is (1.1M candidates: 7.25 -> 6.3 ms).
//
// read_n_kernel: results[i].x of candidate i of a read of min_m to max_m bases
// becomes 1 if the read holds an N, else 0.  Neighbouring candidates of one
// read share the loads of its Peq entries' N words.
__global__ __launch_bounds__(256) void read_n_kernel(myers_verify_args_t a, uint32_t n, uint32_t min_m, uint32_t max_m) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, lane = __lane_id();
    uint32_t query = 0xFFFFFFFFu, m = 0, entry = 0;
    if (i < n) {
        query = static_cast<const CandRec *>(a.cands)[i].query;
        if (query < a.num_queries) {
            const uint2 qi = reinterpret_cast<const uint2 *>(a.qinfo)[query];
            if (qi.y >= min_m && qi.y <= max_m && (uint64_t)qi.x + ((qi.y + 127u) >> 7) <= (uint64_t)a.num_peq_entries) {
                entry = qi.x;
                m = qi.y;
            }
        }
    }
    const uint64_t heads = __ballot(lane == 0u || (uint32_t)__shfl_up((int)query, 1) != query);
    const uint64_t upto = lane == 63u ? ~0ull : (2ull << lane) - 1ull;
    const uint32_t first = 63u - (uint32_t)__builtin_clzll(heads & upto);
    const uint64_t after = heads & ~upto;
    const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
    // lane k of a run of L lanes looks at the read's words k, k + L, ...
    uint32_t any = 0;
    for (uint32_t w = lane - first; 32u * w < m; w += end - first) {
        const uint32_t rows = m - 32u * w >= 32u ? ~0u : (1u << (m & 31u)) - 1u;
        any |= a.peq[(size_t)(entry + (w >> 2)) * 20u + 16u + (w & 3u)] & rows;
    }
    const uint64_t run = (end == 64u ? ~0ull : (1ull << end) - 1ull) & ~((1ull << first) - 1ull);
    const uint64_t found = __ballot(any != 0u) & run;
    if (i < n) static_cast<uint2 *>(a.results)[i].x = found ? 1u : 0u;
}

// Stable partition of each span of kNSpan slots of a variant's range (from
// the range's start): candidates of reads with N first, so that the grid's
// tail is the shorter chunks.  One block per span.
constexpr uint32_t kNSpan = 4096u, kNRounds = kNSpan / 256u;
__global__ __launch_bounds__(256) void group_n_kernel(const uint32_t *ranges, uint32_t nv, uint64_t mask,
                                                      uint32_t *order, const uint2 *results) {
    __shared__ uint32_t before[kNRounds * 4u];          // with N: per round of 256 slots and wave, then those before it
    __shared__ uint32_t total;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t spans = 0;                                 // of the variants before v
    for (uint32_t v = 0; v < nv && v < 64u; v++) {
        if (!((mask >> v) & 1ull)) continue;
        const uint32_t start = ranges[2 * v], count = ranges[2 * v + 1];
        const uint32_t here = (count + kNSpan - 1u) / kNSpan;
        // block b takes the spans b, b + gridDim, .. of all variants' spans
        const uint32_t skip = (blockIdx.x + gridDim.x - spans % gridDim.x) % gridDim.x;
        for (uint32_t sp = skip; sp < here; sp += gridDim.x) {
            const uint32_t s0 = start + sp * kNSpan, len = min(kNSpan, count - sp * kNSpan);
            uint32_t cand[kNRounds], is_n = 0;
            __syncthreads();                            // the previous span's counts have been read
#pragma unroll
            for (uint32_t r = 0; r < kNRounds; r++) {
                const uint32_t at = r * 256u + threadIdx.x;
                cand[r] = at < len ? order[s0 + at] : 0u;
                const bool with_n = at < len && (results[cand[r]].x & 1u) != 0u;
                is_n |= with_n ? 1u << r : 0u;
                const uint64_t b = __ballot(with_n);
                if (lane == 0u) before[4u * r + wave] = (uint32_t)__builtin_popcountll(b);
            }
            __syncthreads();
            if (wave == 0u) {                           // exclusive scan of the 64 counts
                const uint32_t own = before[lane];
                uint32_t sum = own;
                for (uint32_t o = 1; o < 64u; o <<= 1) {
                    const uint32_t y = (uint32_t)__shfl_up((int)sum, o);
                    sum += lane >= o ? y : 0u;
                }
                before[lane] = sum - own;
                if (lane == 63u) total = sum;
            }
            __syncthreads();
            const uint32_t nn = total;
            if (nn == 0u) continue;                     // no N in the span (the same for the block)
#pragma unroll
            for (uint32_t r = 0; r < kNRounds; r++) {
                const uint32_t at = r * 256u + threadIdx.x;
                const bool with_n = (is_n >> r) & 1u;
                const uint64_t b = __ballot(with_n);
                const uint32_t rank = before[4u * r + wave] + (uint32_t)__builtin_popcountll(b & below);
                if (at < len) order[s0 + (with_n ? rank : nn + (at - rank))] = cand[r];
            }
        }
        spans += here;
    }
}

// Sort each span of kLenSpan slots of a variant's range: reads with N first
// (read_n_kernel), then by read length, longest first, then by slot (so a
// read's candidates stay together).  A bitonic network over keys of the three
// in LDS, one block per span.
constexpr uint32_t kLenSpan = 4096u;
__global__ __launch_bounds__(1024) void sort_len_kernel(myers_verify_args_t a, const uint32_t *ranges, uint32_t nv,
                                                        uint64_t mask, uint32_t *order) {
    __shared__ uint32_t key[kLenSpan], cand[kLenSpan];
    uint32_t spans = 0;                                 // of the variants before v
    for (uint32_t v = 0; v < nv && v < 64u; v++) {
        if (!((mask >> v) & 1ull)) continue;
        const uint32_t start = ranges[2 * v], count = ranges[2 * v + 1];
        const uint32_t here = (count + kLenSpan - 1u) / kLenSpan;
        // block b takes the spans b, b + gridDim, .. of all variants' spans
        const uint32_t skip = (blockIdx.x + gridDim.x - spans % gridDim.x) % gridDim.x;
        for (uint32_t sp = skip; sp < here; sp += gridDim.x) {
            const uint32_t s0 = start + sp * kLenSpan, len = min(kLenSpan, count - sp * kLenSpan);
            uint32_t n = 2;                             // keys sorted: a power of two
            while (n < len) n *= 2u;
            __syncthreads();                            // the previous span is written
            for (uint32_t at = threadIdx.x; at < n; at += 1024u) {
                uint32_t k = ~0u;
                if (at < len) {
                    const uint32_t c = order[s0 + at], query = static_cast<const CandRec *>(a.cands)[c].query;
                    const uint32_t m = query < a.num_queries ? reinterpret_cast<const uint2 *>(a.qinfo)[query].y : 0u;
                    cand[at] = c;
                    const uint32_t n_last = static_cast<const uint2 *>(a.results)[c].x & 1u ? 0u : 1u << 31;
                    k = n_last | ((0x7FFFFu - min(m, 0x7FFFFu)) << 12) | at;
                }
                key[at] = k;
            }
            __syncthreads();
            for (uint32_t size = 2; size <= n; size *= 2u) {
                for (uint32_t d = size / 2u; d > 0u; d /= 2u) {
                    for (uint32_t i = threadIdx.x; i < n / 2u; i += 1024u) {
                        const uint32_t lo = 2u * i - (i & (d - 1u)), hi = lo + d;
                        const uint32_t x = key[lo], y = key[hi];
                        if ((x > y) == ((lo & size) == 0u)) {
                            key[lo] = y;
                            key[hi] = x;
                        }
                    }
                    __syncthreads();
                }
            }
            for (uint32_t at = threadIdx.x; at < len; at += 1024u) order[s0 + at] = cand[key[at] & (kLenSpan - 1u)];
        }
        spans += here;
    }
}

}  // namespace

// ------------------------------------------------------------ variant table


namespace {
struct VariantEntry {
    uint32_t lanes, words;
    const void *fn;
    const void *persistent_fn;
    const void *cut_fn;              // threshold mode with the cut-off, or null
    const void *cut_persistent_fn;
    uint32_t block;                  // threads per workgroup
};
template <int L, int W>
constexpr const void *cut_kernel(bool persistent) {
    if constexpr (kHasCut<L, W>) {
        return persistent ? reinterpret_cast<const void *>(&verify_persistent_kernel<L, W, true>)
                          : reinterpret_cast<const void *>(&verify_kernel<L, W, true>);
    } else {
        return nullptr;
    }
}
// One-lane variants run the kernels of myers_slice.hip; those of the shortest
// reads have a plain bit-vector kernel for small batches of one length too
// (110K candidates of 100 bases: 32 us, the sliced form 41), and some wide ones
// the cut-off kernel for low thresholds (launch_bin).
constexpr int kPlainOneLane = 7;
template <int W>
constexpr bool kCutOneLane = W == 19 || W == 22 || W == 25 || W == 29 || W == 32;
template <int L, int W>
constexpr VariantEntry variant_entry() {
    if constexpr (L == 1 && W <= kPlainOneLane) {
        return {1u, (uint32_t)W, reinterpret_cast<const void *>(&verify_kernel<1, W, false>), nullptr, nullptr, nullptr, 64u};
    } else if constexpr (L == 1 && kCutOneLane<W>) {
        return {1u, (uint32_t)W, nullptr, nullptr, reinterpret_cast<const void *>(&verify_kernel<1, W, true>), nullptr, 64u};
    } else if constexpr (L == 1) {
        return {1u, (uint32_t)W, nullptr, nullptr, nullptr, nullptr, 64u};
    } else {
        return {(uint32_t)L, (uint32_t)W, reinterpret_cast<const void *>(&verify_kernel<L, W, false>),
                reinterpret_cast<const void *>(&verify_persistent_kernel<L, W, false>), cut_kernel<L, W>(false),
                cut_kernel<L, W>(true), 64u};
    }
}
#define MYERS_VARIANT_ENTRY(L, W) variant_entry<L, W>(),
#define MYERS_WIDE_ENTRY(Q, W)                                                                   \
    {64u * (Q), W, reinterpret_cast<const void *>(&verify_wide_kernel<Q, W>),                   \
     reinterpret_cast<const void *>(&verify_wide_persistent_kernel<Q, W>), nullptr, nullptr, 64u * (Q)},
const VariantEntry kVariants[] = {MYERS_VARIANT_LIST(MYERS_VARIANT_ENTRY) MYERS_WIDE_LIST(MYERS_WIDE_ENTRY)};
constexpr uint32_t kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
static_assert(kNumVariants < MYERS_MAX_VARIANTS, "variant table too large (the last queue row is the long-read counter)");
#define MYERS_COUNT_LONG(L, W) +((L) >= 4 && (L) <= 64 ? 1 : 0)
static_assert(0 MYERS_VARIANT_LIST(MYERS_COUNT_LONG) <= MYERS_LONG_MAX,
              "one long-read plan can hold a bin of every long-read variant");
#define MYERS_WS_U4(L, W) (uint32_t)((sizeof(Workspace<L, W>) + 15u) / 16u),
const uint32_t kWorkspaceU4[] = {MYERS_VARIANT_LIST(MYERS_WS_U4)};
}  // namespace

extern "C" uint32_t myers_num_variants(void) { return kNumVariants; }

extern "C" int myers_variant_desc(uint32_t v, myers_variant_desc_t *out) {
    if (v >= kNumVariants || out == nullptr) return -1;
    const uint32_t L = kVariants[v].lanes, W = kVariants[v].words;
    out->lanes = L;
    out->words = W;
    out->total_words = L * W;
    out->slots = L <= 64u ? 64u / L : 1u;
    out->block = kVariants[v].block;
    if (L == 1u) {
        out->lds_bytes = myers_slice_ws_u4(32u, W) * 16u;
        return 0;
    }
    hipFuncAttributes attr;
    out->lds_bytes = hipFuncGetAttributes(&attr, kVariants[v].fn) == hipSuccess ? (uint32_t)attr.sharedSizeBytes : 0u;
    return 0;
}

extern "C" int myers_variant_occupancy(uint32_t v, int *wg_per_cu) {
    if (v >= kNumVariants || wg_per_cu == nullptr) return -1;
    if (kVariants[v].lanes == 1u) return myers_slice_occupancy(32u, myers_slice_ws_u4(32u, kVariants[v].words) * 16u, wg_per_cu);
    int blocks = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kVariants[v].fn, (int)kVariants[v].block, 0);
    if (e != hipSuccess) return (int)e;
    *wg_per_cu = blocks;
    return 0;
}

extern "C" int myers_variant_occupancy_persistent(uint32_t v, int *wg_per_cu) {
    if (v >= kNumVariants || wg_per_cu == nullptr) return -1;
    if (kVariants[v].lanes == 1u) return myers_slice_occupancy(32u, myers_slice_ws_u4(32u, kVariants[v].words) * 16u, wg_per_cu);
    int blocks = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kVariants[v].persistent_fn,
                                                                (int)kVariants[v].block, 0);
    if (e != hipSuccess) return (int)e;
    *wg_per_cu = blocks;
    return 0;
}

extern "C" int myers_launch_verify(uint32_t v, const myers_verify_args_t *args, uint32_t grid,
                                   int persistent, hipStream_t stream) {
    if (v >= kNumVariants || args == nullptr || grid == 0) return -1;
    if (persistent && (args->bin_ranges == nullptr || args->queue_heads == nullptr)) return -1;
    void *kargs[] = {const_cast<myers_verify_args_t *>(args)};
    const VariantEntry &ve = kVariants[v];
    const bool cut = args->threshold >= 0.0f && ve.cut_fn != nullptr;
    const void *fn = cut ? (persistent ? ve.cut_persistent_fn : ve.cut_fn) : (persistent ? ve.persistent_fn : ve.fn);
    if (fn == nullptr) return -1;
    hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(ve.block), kargs, 0, stream);
    return (int)e;
}

extern "C" int myers_variant_cut_ok(uint32_t v) {
    return v < kNumVariants && kVariants[v].lanes == 1u && kVariants[v].cut_fn != nullptr;
}

extern "C" int myers_variant_long_ok(uint32_t v, uint32_t *ws_u4) {
    constexpr uint32_t kOneWave = sizeof(kWorkspaceU4) / sizeof(kWorkspaceU4[0]);
    if (v >= kOneWave || kVariants[v].lanes < 4u || kVariants[v].lanes > 64u) return 0;
    if (ws_u4) *ws_u4 = kWorkspaceU4[v];
    return 1;
}

extern "C" uint32_t myers_long_wide_lds_bytes(void) { return (uint32_t)sizeof(LongWide); }

namespace {
#define MYERS_QUEUE_CLASS_OF(L, W) kQueueClass<L, W>,
const int kQueueClassOf[] = {MYERS_VARIANT_LIST(MYERS_QUEUE_CLASS_OF)};
const void *queue_kernel(bool cut) {
    return cut ? reinterpret_cast<const void *>(&verify_queue_kernel<true>)
               : reinterpret_cast<const void *>(&verify_queue_kernel<false>);
}
}  // namespace

extern "C" int myers_variant_queue_class(uint32_t v, uint32_t *ws_u4) {
    constexpr uint32_t kOneWave = sizeof(kQueueClassOf) / sizeof(kQueueClassOf[0]);
    if (v >= kOneWave || kQueueClassOf[v] < 0) return -1;
    // the multi-lane class's workgroups keep one uint4 of hand-over words first
    if (ws_u4) *ws_u4 = kWorkspaceU4[v] + (kQueueClassOf[v] == MYERS_QUEUE_MULTI_LANE ? 1u : 0u);
    return kQueueClassOf[v];
}

extern "C" int myers_queue_occupancy(int cut, uint32_t lds_bytes, int *wg_per_cu) {
    if (wg_per_cu == nullptr) return -1;
    int blocks = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, queue_kernel(cut != 0), 64 * kQueueWaves,
                                                                (size_t)lds_bytes);
    if (e != hipSuccess) return (int)e;
    *wg_per_cu = blocks;
    return 0;
}

extern "C" int myers_launch_queue(const myers_verify_args_t *args, const myers_queue_plan_t *plan, uint32_t grid,
                                  hipStream_t stream) {
    if (args == nullptr || plan == nullptr || grid == 0 || plan->cls != (uint32_t)MYERS_QUEUE_MULTI_LANE ||
        plan->n == 0 || plan->n > (uint32_t)MYERS_QUEUE_MAX || args->bin_ranges == nullptr ||
        args->queue_heads == nullptr)
        return -1;
    uint32_t need = 0;
    for (uint32_t j = 0; j < plan->n; j++) {
        uint32_t u4 = 0;
        const uint32_t v = plan->variant[j];
        if (myers_variant_queue_class(v, &u4) != (int)plan->cls ||
            plan->key[j] != ((kVariants[v].lanes << 8) | kVariants[v].words))
            return -1;
        need = u4 > need ? u4 : need;
    }
    if (plan->ws_u4 < need || plan->ws_u4 * 16u > 64u * 1024u) return -1;
    void *kargs[] = {const_cast<myers_verify_args_t *>(args), const_cast<myers_queue_plan_t *>(plan)};
    return (int)hipLaunchKernel(queue_kernel(args->threshold >= 0.0f), dim3(grid), dim3(64u * kQueueWaves),
                                kargs, (size_t)plan->ws_u4 * 16u, stream);
}

extern "C" int myers_launch_long(const myers_verify_args_t *args, const myers_long_plan_t *plan, uint32_t grid,
                                 hipStream_t stream) {
    if (args == nullptr || plan == nullptr || grid == 0 || plan->n > (uint32_t)MYERS_LONG_MAX ||
        plan->n_wide > (uint32_t)MYERS_LONG_MAX || plan->n + plan->n_wide == 0 ||
        args->bin_ranges == nullptr || args->queue_heads == nullptr)
        return -1;
    uint32_t need = 0;
    for (uint32_t j = 0; j < plan->n_wide; j++) {
        const uint32_t v = plan->wide_variant[j], w = plan->wide_words[j];
        if (!myers_variant_long_ok(v, nullptr) || (w != 2u && w != 3u) ||
            kVariants[v].lanes * kVariants[v].words > 64u * MYERS_LONG_WAVES * w)
            return -1;
        need = (uint32_t)((sizeof(LongWide) + 16u * MYERS_LONG_WAVES - 1u) / (16u * MYERS_LONG_WAVES));
    }
    for (uint32_t j = 0; j < plan->n; j++) {
        uint32_t u4 = 0;
        if (!myers_variant_long_ok(plan->variant[j], &u4) ||
            plan->key[j] != ((kVariants[plan->variant[j]].lanes << 8) | kVariants[plan->variant[j]].words))
            return -1;
        need = u4 > need ? u4 : need;
    }
    if (plan->ws_u4 < need) return -1;
    const size_t lds = (size_t)plan->ws_u4 * 16u * MYERS_LONG_WAVES;
    if (lds > 64u * 1024u) {
        // above 64 KiB a launch needs the kernel's limit raised (gfx950: 160 KiB per workgroup)
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&verify_long_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    void *kargs[] = {const_cast<myers_verify_args_t *>(args), const_cast<myers_long_plan_t *>(plan)};
    return (int)hipLaunchKernel(reinterpret_cast<const void *>(&verify_long_kernel), dim3(grid),
                                dim3(64u * MYERS_LONG_WAVES), kargs, lds, stream);
}

// ------------------------------------------------- static device workspace
// The allocation-free entry point's workspace.  In host code the name
// `scratch` stands for the variable, not a device address: the address on
// each GPU comes from hipGetSymbolAddress, resolved once per device and kept.
static __device__ __align__(256) uint32_t scratch[MYERS_SCRATCH_WORDS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint32_t *g_scratch_ptr[kMaxDevices];
}  // namespace

extern "C" int myers_scratch_init(int device, uint32_t **ptr) {
    if (device < 0 || device >= kMaxDevices || ptr == nullptr) return (int)hipErrorInvalidValue;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device] == nullptr) {
        int current = -1;
        hipError_t e = hipGetDevice(&current);
        if (e != hipSuccess) return (int)e;
        if (current != device) return (int)hipErrorInvalidDevice;
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (p == nullptr) return (int)hipErrorInvalidSymbol;
        g_scratch_ptr[device] = static_cast<uint32_t *>(p);
    }
    *ptr = g_scratch_ptr[device];
    return 0;
}

extern "C" int myers_launch_binning(const uint32_t *qinfo, uint32_t num_queries, const void *cands,
                                    uint32_t num_cands,
                                    const uint8_t *bin_of_words, uint32_t max_words,
                                    uint32_t num_variants, uint32_t *block_counts, uint32_t *ranges,
                                    uint32_t *order, uint32_t *host_err, void *results, uint32_t *queue_heads,
                                    hipStream_t stream) {
    if (num_variants == 0 || num_variants >= MYERS_MAX_VARIANTS || host_err == nullptr) return -1;
    const uint2 *qi = reinterpret_cast<const uint2 *>(qinfo);
    const CandRec *cr = static_cast<const CandRec *>(cands);
    uint32_t grid = (num_cands + 1023u) / 1024u;           // about 4 rounds of 256 per block
    if (grid > (uint32_t)MYERS_BIN_BLOCKS) grid = (uint32_t)MYERS_BIN_BLOCKS;
    if (grid == 0u) grid = 1u;
    hipLaunchKernelGGL(bin_count_kernel, dim3(grid), dim3(256), 0, stream, qi, num_queries, cr, num_cands,
                       bin_of_words, max_words, num_variants, block_counts);
    hipLaunchKernelGGL(bin_scan_kernel, dim3(num_variants + 1u), dim3(256), 0, stream, block_counts, grid, ranges,
                       host_err);
    hipLaunchKernelGGL(bin_scatter_kernel, dim3(grid), dim3(256), 0, stream, qi, num_queries, cr, num_cands,
                       bin_of_words, max_words, num_variants, block_counts, ranges, queue_heads, order,
                       static_cast<uint2 *>(results));
    return (int)hipGetLastError();
}

extern "C" int myers_launch_read_n(const myers_verify_args_t *args, uint32_t num_cands, uint32_t min_m,
                                   uint32_t max_m, hipStream_t stream) {
    if (args == nullptr || args->results == nullptr || num_cands == 0u) return -1;
    hipLaunchKernelGGL(read_n_kernel, dim3((num_cands + 255u) / 256u), dim3(256), 0, stream, *args, num_cands, min_m,
                       max_m);
    return (int)hipGetLastError();
}

extern "C" int myers_launch_group_n(const uint32_t *ranges, uint32_t num_variants, uint64_t variants,
                                    uint32_t num_cands, uint32_t *order, const void *results, hipStream_t stream) {
    if (ranges == nullptr || order == nullptr || results == nullptr || num_variants > MYERS_MAX_VARIANTS) return -1;
    uint32_t grid = num_cands / kNSpan + 1u;
    if (grid > 2048u) grid = 2048u;
    hipLaunchKernelGGL(group_n_kernel, dim3(grid), dim3(256), 0, stream, ranges, num_variants, variants, order,
                       static_cast<const uint2 *>(results));
    return (int)hipGetLastError();
}

extern "C" int myers_launch_sort_len(const myers_verify_args_t *args, const uint32_t *ranges, uint32_t num_variants,
                                     uint64_t variants, uint32_t num_cands, uint32_t *order, hipStream_t stream) {
    if (args == nullptr || ranges == nullptr || order == nullptr || num_variants > MYERS_MAX_VARIANTS) return -1;
    uint32_t grid = num_cands / kLenSpan + (uint32_t)__builtin_popcountll(variants);
    if (grid > 1024u) grid = 1024u;
    if (grid == 0u) return 0;
    hipLaunchKernelGGL(sort_len_kernel, dim3(grid), dim3(1024), 0, stream, *args, ranges, num_variants, variants, order);
    return (int)hipGetLastError();
}
