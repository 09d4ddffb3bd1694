// Candidate-verification kernels for MI355X (gfx950, wave64).
//
// Each candidate is verified by the Myers/Hyyro bit-vector recurrence over
// its reference window (reference kernel: src-api/coreMyersGPU-CC35.cu:110-240;
// CPU form: src/myers-4bits.c:111-135).  All work is integer VALU (no MFMA).
//
//   * A kernel variant <L, W> gives each candidate L lanes of a wave64 and
//     each lane W u32 words of the query bit-vector (32*L*W rows in all).
//     Inside a lane the W words form one full-width vector (add carries and
//     Ph/Mh shifts run through all of them).  Between the lanes of a group
//     the block form of the recurrence applies (src/myers-4bits.c:115-134):
//     a lane needs only the horizontal delta hin at its bottom boundary,
//     which is the top bit of the Ph/Mh of the lane below in the same
//     column.  The lanes run diagonally: lane b of a group computes column
//     t - b at step t, so its hin is the lower lane's output of step t - 1,
//     moved up one lane by a single DPP shift.  No carry crosses lanes, no
//     ballot, no branch.  A lane before its first column reads an all-zero
//     Peq row; with Eq = 0 and hin = 0 the initial state Pv = ~0, Mv = 0 is
//     a fixed point emitting no delta, so late-starting lanes need no reset.
//     L = 1 is the special case with hin = 0 and no lag.
//   * Query bit-vectors are top-justified: a query of m bases occupies the
//     top m rows and the rows below it never match (their Peq bits are 0).
//     Such rows stay at the same fixed point, so they emit no horizontal
//     delta and the query rows see the semi-global boundary D[0][j]=0.  The
//     score row m-1 is therefore bit 31 of the top lane's top word for every
//     m the variant covers.
//   * Peq masks are staged into LDS once per distinct read of a wave, as
//     [ceil(W/4) groups][read slot][rows][L lanes] x 128-bit (rows = 5 bases,
//     plus a zero row for L > 1), so one column's Eq words are ceil(W/4)
//     ds_read_b128 at an address chosen by the column's base code, and the
//     (slot, base) pairs of a wave fall on consecutive 16-byte bank groups.
//   * The packed reference (8 bases per u32) streams through a register
//     window per lane, two 8-column blocks ahead of use; exact-start windows
//     and the diagonal lag use a per-lane funnel shift.
//   * Per word and column the recurrence is 10 VALU ops: and, add-with-carry,
//     3 three-input logic ops, 2 funnel shifts, or, and, and.  and/or/bitop3
//     issue at twice the rate of the funnel shifts and the carry add on
//     gfx950, so variants are sized for at least two waves per SIMD.
#ifndef MYERS_DEVICE_H
#define MYERS_DEVICE_H
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "myers_kernels.h"

namespace {

struct CandRec {
    uint32_t query;
    uint32_t pad;
    uint64_t position;
};

constexpr uint32_t kSkipScore = 0xFFFFFFFFu;
constexpr uint32_t kNoMatch = 0xFFFFFFFFu;  // threshold mode: {column, score} of a candidate above it
constexpr uint32_t kZeroRow = 5u;          // LDS row of all-zero Peq words (L > 1)

// n = (uint32)(m * (1 + 2*d)) in float32 with round-to-nearest steps
// (src-api/coreMyersGPU-CC35.cu:131).
__device__ __forceinline__ uint32_t window_len(uint32_t m, float d) {
    float f = __fmul_rn((float)m, __fadd_rn(1.0f, __fmul_rn(2.0f, d)));
    return (uint32_t)f;
}

// Rows 5..7 of the Peq do not exist; the reference kernel's selectEq maps
// them to row 0 (src-api/coreMyersGPU-CC35.cu:82-95).  Applied to all eight
// nibbles of a text word at once: clear bit 3, then zero codes 5..7.
__device__ __forceinline__ uint32_t sanitize_text(uint32_t w) {
    uint32_t c = w & 0x77777777u;
    uint32_t hi = (c >> 2) & 0x11111111u;
    uint32_t lo = (c | (c >> 1)) & 0x11111111u;
    return c & ~((hi & lo) * 7u);
}

// Under-threshold bound k = (uint32)((float)m * e) (src/checksum-2.c:88); the host
// passes no e above MYERS_MAX_THRESHOLD, so that sums with k stay within 31 bits.
__device__ __forceinline__ uint32_t threshold_of(uint32_t m, float e) {
    return (uint32_t)__fmul_rn((float)m, e);
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o));
    return __builtin_amdgcn_readfirstlane(v);
}

template <int L, int W>
struct Shape {
    static constexpr int kGroups = (W + 3) / 4;        // 128-bit LDS groups per lane
    static constexpr int kTotal = L * W;                // words per candidate
    static constexpr int kSlots = 64 / L;               // candidates per wave
    static constexpr int kRows = L > 1 ? 6 : 5;         // A C G T N (+ zero row)
    // Peq is staged once per distinct query of the wave ("query slot"), not
    // once per candidate; up to kQSlots queries per pass.  LDS layout
    // [group][slot][row][lane] x 128 bit: the uint4s one column reads for
    // the (slot, base) pairs of a wave are consecutive in slot*rows + base,
    // so they spread evenly over the LDS banks.
    static constexpr int kQSlotsMax = L == 1 ? 16 : 8;
    static constexpr int kQSlots = kSlots < kQSlotsMax ? kSlots : kQSlotsMax;
    static constexpr int kRowU4 = L;                    // uint4 between rows of a slot
    static constexpr int kSlotU4 = kRows * L;           // uint4 between slots
    static constexpr int kGroupU4 = kQSlots * kSlotU4;  // uint4 between groups
    static constexpr int kLdsU4 = kGroups * kGroupU4;
};

// Loads and stores of a batch's arrays.  kHost: the arrays are host memory
// rewritten while a resident kernel runs (the serving arena), which the GPU
// may hold in its L2; system-scope accesses go around that cache, so a load
// never sees a line cached for an earlier request and a store reaches the
// host once it completes.  Otherwise plain (cached) accesses.
template <bool kHost>
__device__ __forceinline__ uint32_t ld32(const uint32_t *p) {
    if constexpr (kHost) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else return *p;
}
template <bool kHost>
__device__ __forceinline__ uint64_t ld64(const uint64_t *p) {
    if constexpr (kHost) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else return *p;
}
template <bool kHost>
__device__ __forceinline__ void st_result(uint2 *p, uint2 v) {
    if constexpr (kHost) {
        __hip_atomic_store(reinterpret_cast<uint64_t *>(p), ((uint64_t)v.y << 32) | v.x, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    } else {
        *p = v;
    }
}

// Stage the Peq words of the wave's query slots into LDS, top-justified,
// with all 64 lanes sharing the work.  Word gw (0 <= gw < L*W) of a slot
// holds virtual rows [32gw, 32gw+32); virtual row r is query row r - pad,
// pad = 32*L*W - m, so it is the funnel of query words lo and lo+1
// (lo = floor((32gw - pad)/32)) shifted right by (-pad) mod 32.  Query word
// j (rows 32j..32j+31) of base c is bitmap[c][j%4] of entry posEntry + j/4;
// words outside the query read 0.  Lane gl = gw / W of the group reads word
// k = gw % W at LDS uint4 (k/4)*kGroupU4 + slot*kSlotU4 + c*L + gl, lane k%4.
template <int L, int W, bool kHost = false, uint32_t kThreads = 64>
__device__ __forceinline__ void stage_peq(uint4 *lds, const uint2 *qtab, uint32_t nslots,
                                          const uint32_t *__restrict__ peq, uint32_t lane) {
    using S = Shape<L, W>;
    uint32_t *l32 = reinterpret_cast<uint32_t *>(lds);
    const uint32_t total = nslots * 5u * (uint32_t)S::kTotal;
    for (uint32_t idx = lane; idx < total; idx += kThreads) {
        const uint32_t gw = idx % (uint32_t)S::kTotal;
        const uint32_t rest = idx / (uint32_t)S::kTotal;
        const uint32_t c = rest % 5u;
        const uint32_t slot = rest / 5u;
        const uint2 qi = qtab[slot];                   // {posEntry, m}
        const int32_t pad = 32 * S::kTotal - (int32_t)qi.y;
        const int32_t nq = (int32_t)((qi.y + 31u) >> 5);
        const int32_t b0 = 32 * (int32_t)gw - pad;
        const int32_t lo = b0 >> 5;                    // floor division
        const uint32_t sh = (uint32_t)b0 & 31u;
        const uint32_t *base = peq + (size_t)qi.x * 20u + 4u * c;
        uint32_t wlo = 0, whi = 0;
        if (lo >= 0 && lo < nq) wlo = ld32<kHost>(base + (uint32_t)(lo >> 2) * 20u + (uint32_t)(lo & 3));
        if (lo + 1 >= 0 && lo + 1 < nq)
            whi = ld32<kHost>(base + (uint32_t)((lo + 1) >> 2) * 20u + (uint32_t)((lo + 1) & 3));
        const uint32_t k = gw % (uint32_t)W, gl = gw / (uint32_t)W;
        const uint32_t u4 = (k >> 2) * (uint32_t)S::kGroupU4 + slot * (uint32_t)S::kSlotU4 + c * (uint32_t)L + gl;
        l32[u4 * 4u + (k & 3u)] = (uint32_t)((((uint64_t)whi << 32) | wlo) >> sh);
    }
}

// Truth tables of v_bitop3_b32(a, b, c): bit (4a+2b+c) of the immediate is
// f(a, b, c); with a = 0xF0, b = 0xCC, c = 0xAA the table is f applied
// bitwise to those constants.
constexpr uint32_t kXorOr = (0xF0u ^ 0xCCu) | 0xAAu;          // (a ^ b) | c
constexpr uint32_t kOrNor = (0xF0u | ~(0xCCu | 0xAAu)) & 0xFFu;  // a | ~(b | c)

// The lower lane's value of the previous step: DPP row_shr:1 (within rows
// of 16) or wave_shr:1, with 0 on the first lane of every group.
template <int L>
__device__ __forceinline__ uint32_t from_lower_lane(uint32_t v, uint32_t not_first) {
    if constexpr (L > 16) {
        v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);   // wave_shr:1
    } else {
        v = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);   // row_shr:1
    }
    if constexpr (L != 16 && L != 64) v &= not_first;   // rows and the wave already start at 0
    return v;
}

// One group of four words (g) of a one-lane column (L = 1), for the cut-off
// column below: the recurrence over words 4g..4g+3 with the Eq words e
// (src/myers-4bits.c:115-134 block form), in the phased order of column_grp.
// carry is the add's carry between words; ph_prev / mh_prev the Ph / Mh
// (before the shift) of the word below, whose top bit shifts into this
// group's first word.
template <int W>
__device__ __forceinline__ void group_update(int g, uint32_t (&Pv)[W], uint32_t (&Mv)[W], const uint4 &e,
                                             uint32_t &carry, uint32_t &ph_prev, uint32_t &mh_prev) {
    const uint32_t e4[4] = {e.x, e.y, e.z, e.w};
    const int k0 = 4 * g;
    const int n = (W - k0) < 4 ? (W - k0) : 4;
    uint32_t t[4], xv[4], sum[4], xh[4], ph[4], mh[4], php[4], mhp[4];
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) {
        t[j] = e4[j] & Pv[k0 + j];
        xv[j] = e4[j] | Mv[k0 + j];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) {
        uint32_t c_out;
        sum[j] = __builtin_addc(t[j], Pv[k0 + j], carry, &c_out);
        carry = c_out;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) xh[j] = __builtin_amdgcn_bitop3_b32(sum[j], Pv[k0 + j], e4[j], kXorOr);
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) {
        ph[j] = __builtin_amdgcn_bitop3_b32(Mv[k0 + j], xh[j], Pv[k0 + j], kOrNor);
        mh[j] = Pv[k0 + j] & xh[j];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) {
        const int k = k0 + j;
        php[j] = k == 0 ? (ph[j] << 1) : __builtin_amdgcn_alignbit(ph[j], ph_prev, 31u);
        mhp[j] = k == 0 ? (mh[j] << 1) : __builtin_amdgcn_alignbit(mh[j], mh_prev, 31u);
        ph_prev = ph[j];
        mh_prev = mh[j];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4 && j < n; j++) {
        Pv[k0 + j] = __builtin_amdgcn_bitop3_b32(mhp[j], xv[j], php[j], kOrNor);
        Mv[k0 + j] = php[j] & xv[j];
    }
    __builtin_amdgcn_sched_barrier(0);
}

// One column for one lane's W words.  Eq words stream from LDS one group of
// four words ahead of use (group g+1 is read while group g computes; the
// caller reads the next column's group 0 at the start of the column), so 12
// Eq registers are live instead of 2W.  For L > 1, ph_in / mh_in carry the
// lower lane's hin in bit 31 (src/myers-4bits.c:115-134 block form).  The
// top word's Ph / Mh (before the shift) come back in ph_top / mh_top.
//
// kPhased: issue each group's word updates in phases (below).  With several
// waves per SIMD this raises the share of quad-cycles that issue two VALU
// instructions (18% -> 35% on 1000-base reads, 11% faster); a wave that runs
// a long chain alone on its SIMD (the long-read launch, multi-wave
// candidates) is 5-10% faster with the compiler's interleaved order, which
// overlaps the carry chain with the other words' operations.  The phased
// body is also group_update's; calling group_update here measured 2% slower
// (the compiler sinks Xv into the last phase), and pinning Xv in the first
// phase makes the cut-off column spill.
template <int W, bool kHin, uint32_t kGS, bool kPhased = true>
__device__ __forceinline__ void column_grp(uint32_t (&Pv)[W], uint32_t (&Mv)[W], const uint4 &e0,
                                           const uint4 *lds_lane, uint32_t cur_off, uint32_t ph_in,
                                           uint32_t mh_in, uint32_t &ph_top, uint32_t &mh_top) {
    constexpr int kG = (W + 3) / 4;     // kGS: uint4 between groups in LDS
    uint32_t carry = 0, ph_prev = ph_in, mh_prev = mh_in;
    uint4 cur = e0, nxt = e0;
#pragma unroll
    for (int g = 0; g < kG; g++) {
        {
            if (g + 1 < kG) nxt = lds_lane[cur_off + (uint32_t)(g + 1) * kGS];
            const uint32_t e4[4] = {cur.x, cur.y, cur.z, cur.w};
            if constexpr (kPhased) {
                const int k0 = 4 * g;
                const int n = (W - k0) < 4 ? (W - k0) : 4;
                uint32_t eqv[4], t[4], xv[4], sum[4], xh[4], ph[4], mh[4], php[4], mhp[4];
                // The group's words go through the recurrence in phases, each
                // phase over all of its words, so that the double-rate bit
                // operations of independent words issue back to back (a SIMD
                // issues two of them in one quad-cycle) and the single-rate ones
                // (add with carry, funnel shifts) come in runs:
                //   Eq & Pv, Xv | carry chain | Xh, Ph, Mh | shifts | Pv, Mv.
                // sched_barrier keeps the compiler from interleaving the phases.
    #pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (j >= n) break;
                    const int k = k0 + j;
                    eqv[j] = (kHin && k == 0) ? (e4[0] | (mh_in >> 31)) : e4[j];
                    t[j] = eqv[j] & Pv[k];
                    xv[j] = e4[j] | Mv[k];
                }
                __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (j >= n) break;
                    uint32_t c_out;
                    sum[j] = __builtin_addc(t[j], Pv[k0 + j], carry, &c_out);
                    carry = c_out;
                }
                __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                for (int j = 0; j < 4 && j < n; j++) xh[j] = __builtin_amdgcn_bitop3_b32(sum[j], Pv[k0 + j], eqv[j], kXorOr);
    #pragma unroll
                for (int j = 0; j < 4 && j < n; j++) {
                    ph[j] = __builtin_amdgcn_bitop3_b32(Mv[k0 + j], xh[j], Pv[k0 + j], kOrNor);
                    mh[j] = Pv[k0 + j] & xh[j];
                }
                __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                for (int j = 0; j < 4 && j < n; j++) {
                    const int k = k0 + j;
                    php[j] = (!kHin && k == 0) ? (ph[j] << 1) : __builtin_amdgcn_alignbit(ph[j], ph_prev, 31u);
                    mhp[j] = (!kHin && k == 0) ? (mh[j] << 1) : __builtin_amdgcn_alignbit(mh[j], mh_prev, 31u);
                    ph_prev = ph[j];
                    mh_prev = mh[j];
                }
                __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                for (int j = 0; j < 4 && j < n; j++) {
                    Pv[k0 + j] = __builtin_amdgcn_bitop3_b32(mhp[j], xv[j], php[j], kOrNor);
                    Mv[k0 + j] = php[j] & xv[j];
                }
                __builtin_amdgcn_sched_barrier(0);
            } else {
#pragma unroll
                for (int k = 4 * g; k < 4 * g + 4 && k < W; k++) {
                    const uint32_t pv = Pv[k], mv = Mv[k];
                    const uint32_t xv = e4[k - 4 * g] | mv;
                    const uint32_t eq = (kHin && k == 0) ? (e4[0] | (mh_in >> 31)) : e4[k - 4 * g];
                    uint32_t c_out;
                    const uint32_t sum = __builtin_addc(eq & pv, pv, carry, &c_out);
                    carry = c_out;
                    const uint32_t xh = __builtin_amdgcn_bitop3_b32(sum, pv, eq, kXorOr);
                    const uint32_t ph = __builtin_amdgcn_bitop3_b32(mv, xh, pv, kOrNor);
                    const uint32_t mh = pv & xh;
                    const uint32_t php = (!kHin && k == 0) ? (ph << 1) : __builtin_amdgcn_alignbit(ph, ph_prev, 31u);
                    const uint32_t mhp = (!kHin && k == 0) ? (mh << 1) : __builtin_amdgcn_alignbit(mh, mh_prev, 31u);
                    ph_prev = ph;
                    mh_prev = mh;
                    Pv[k] = __builtin_amdgcn_bitop3_b32(mhp, xv, php, kOrNor);
                    Mv[k] = php & xv;
                }
            }
            cur = nxt;
        }
    }
    ph_top = ph_prev;
    mh_top = mh_prev;
}

// The same column (L = 1) with the Ukkonen cut-off of threshold mode (Myers
// 1999, blocks model; GEMTools gt_map_align_bpm.c:141-214): only groups
// 0..ga-1 are advanced, ga being the same in every lane of the wave.  Group
// G+1 runs inside group G's (scalar) branch, so a skipped group costs a
// compare and a branch, the carry stays in its scalar register, and no
// value needs merging between groups; ph_top / mh_top are those of group
// ga-1's top word.
template <int G, int W, uint32_t kGS>
__device__ __forceinline__ void column_cut(uint32_t (&Pv)[W], uint32_t (&Mv)[W], const uint4 &cur,
                                           const uint4 *lds_lane, uint32_t cur_off, uint32_t ga,
                                           uint32_t carry, uint32_t ph_prev, uint32_t mh_prev,
                                           uint32_t &ph_top, uint32_t &mh_top) {
    constexpr int kG = (W + 3) / 4;
    uint4 nxt = cur;
    if constexpr (G + 1 < kG) nxt = lds_lane[cur_off + (uint32_t)(G + 1) * kGS];
    group_update<W>(G, Pv, Mv, cur, carry, ph_prev, mh_prev);
    if constexpr (G + 1 < kG) {
        if ((uint32_t)(G + 1) < ga) {
            column_cut<G + 1, W, kGS>(Pv, Mv, nxt, lds_lane, cur_off, ga, carry, ph_prev, mh_prev, ph_top, mh_top);
            return;
        }
    }
    ph_top = ph_prev;
    mh_top = mh_prev;
}

template <int L, int W>
struct Workspace {
    uint4 lds[Shape<L, W>::kLdsU4];
    uint2 qtab[Shape<L, W>::kQSlots];
};

// LDS hand-over between the lanes of one wave when a workgroup holds several
// independent waves: a wave's LDS accesses execute in order, so it is enough
// to wait for them and keep the compiler from moving accesses across.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// Workgroups of kWaves independent waves (1: the workgroup is the wave).
template <int kWaves>
__device__ __forceinline__ void chunk_sync() {
    if constexpr (kWaves == 1) {
        __syncthreads();
    } else {
        wave_lds_sync();
    }
}

template <int kWaves>
__device__ __forceinline__ uint32_t wave_lane() {
    return kWaves == 1 ? threadIdx.x : (threadIdx.x & 63u);
}

// kThreads: the threads sharing the workspace (64, or 128 for a workgroup of
// two waves that stage together).
template <int L, int W, int kWaves = 1, uint32_t kThreads = 64>
__device__ __forceinline__ void zero_row_init(Workspace<L, W> &ws) {
    using S = Shape<L, W>;
    if constexpr (S::kRows > 5) {
        // the all-zero row read by lanes before their first column
        uint32_t *l32 = reinterpret_cast<uint32_t *>(ws.lds);
        constexpr uint32_t kPerGroup = (uint32_t)(S::kQSlots * L);    // (slot, lane) pairs
        const uint32_t t0 = kThreads == 64u ? wave_lane<kWaves>() : threadIdx.x;
        for (uint32_t i = t0; i < (uint32_t)S::kGroups * kPerGroup * 4u; i += kThreads) {
            const uint32_t u4 = i >> 2, g = u4 / kPerGroup, r = u4 % kPerGroup;
            const uint32_t slot = r / (uint32_t)L, gl = r % (uint32_t)L;
            l32[(g * (uint32_t)S::kGroupU4 + slot * (uint32_t)S::kSlotU4 + kZeroRow * (uint32_t)L + gl) * 4u +
                (i & 3u)] = 0u;
        }
    }
}

// Verify chunks chunk_lo, chunk_lo + stride, ... < chunk_hi of the slot range
// [start, start + count); a chunk is the kSlots candidates of one wave.
// kCut: threshold mode.  L = 1 (W >= 8): the Ukkonen cut-off; L > 1: a
// wave stops once its candidates cannot get under the threshold.  kHost: the
// batch's arrays are host memory of the resident server (ld32 / st_result).
// kShare = 2: a workgroup of two waves verifies chunk pairs (2c, 2c+1) with
// one workspace: the distinct reads of both waves' candidates share its
// query slots (one pass while they number at most kQSlots), so each wave
// needs half the LDS of a wave of its own.  xchg: three words of LDS for the
// hand-over between the waves (the last read of wave 0, each wave's count of
// reads).
template <int L, int W, bool kCut, int kWaves = 1, bool kHost = false, int kShare = 1>
__device__ __forceinline__ void verify_chunks(const myers_verify_args_t &a, uint32_t start, uint32_t count,
                                              uint32_t chunk_lo, uint32_t chunk_hi, uint32_t stride,
                                              Workspace<L, W> &ws, uint32_t *xchg = nullptr) {
    static_assert(kShare == 1 || (kShare == 2 && kWaves == 1 && !kHost), "shared workspace: one-wave chunks");
    using S = Shape<L, W>;
    constexpr bool kUkk = kCut && L == 1;       // the cut-off
    constexpr bool kStop = kCut && L > 1;       // the early stop
    uint4 *lds = ws.lds;
    uint2 *qtab = ws.qtab;
    const uint32_t lane = kShare == 1 ? wave_lane<kWaves>() : (threadIdx.x & 63u);
    const uint32_t wave = kShare == 1 ? 0u : (threadIdx.x >> 6);
    const uint32_t gl = lane % L;                      // lane within the candidate's group
    const uint32_t *__restrict__ ref = a.ref;
    const int32_t last_word = (int32_t)(a.ref_words - 1);
    const CandRec *__restrict__ cands = static_cast<const CandRec *>(a.cands);
    const uint2 *__restrict__ qinfo = reinterpret_cast<const uint2 *>(a.qinfo);
    uint2 *__restrict__ results = static_cast<uint2 *>(a.results);
    const uint32_t not_first = gl != 0u ? ~0u : 0u;
    const uint64_t lanes_upto = lane == 63u ? ~0ull : ((2ull << lane) - 1ull);

    for (uint32_t chunk = chunk_lo; chunk < chunk_hi; chunk += stride) {
        const uint32_t slot = (chunk * (uint32_t)kShare + wave) * S::kSlots + lane / L;
        const bool valid = slot < count;
        uint32_t cand = 0, m = 0, pos_entry = 0, query = 0xFFFFFFFFu;
        uint64_t pos = 0;
        bool sane = false;
        if (valid) {
            const uint32_t s = start + slot;
            cand = a.order ? ld32<kHost>(a.order + s) : s;
            if constexpr (kHost) {
                pos = ld64<true>(&cands[cand].position);
                query = ld32<true>(&cands[cand].query);
            } else {
                const CandRec cr = cands[cand];
                pos = cr.position;
                query = cr.query;
            }
            if (query < a.num_queries) {
                const uint64_t qi = ld64<kHost>(reinterpret_cast<const uint64_t *>(qinfo + query));
                pos_entry = (uint32_t)qi;
                m = (uint32_t)(qi >> 32);
                // the query must fit this variant and its Peq entries the batch
                sane = m <= 32u * S::kTotal &&
                       (uint64_t)pos_entry + ((m + 127u) >> 7) <= (uint64_t)a.num_peq_entries;
            }
        }
        if (!sane) m = 0;
        const uint32_t n = window_len(m, a.distance);
        // skip rule: src-api/coreMyersGPU-CC35.cu:142
        const bool live = valid && sane && pos < a.ref_size && (a.ref_size - pos) > (uint64_t)n;
        uint64_t nib0 = 0;
        uint32_t ncols_live = 0;
        if (live) {
            if (a.mode == 0) {
                // aligned window: src-api/coreMyersGPU-CC35.cu:132,144
                nib0 = pos & ~7ull;
                ncols_live = 8u * ((n >> 3) + ((n & 7u) ? 2u : 1u));
            } else {
                nib0 = pos;
                ncols_live = n;
            }
        }

        // Query slots: consecutive candidates of one query share a slot (the
        // callers' batches and the binning keep a query's candidates adjacent).
        uint32_t query_below = (uint32_t)__shfl_up((int)query, L);
        if constexpr (kShare == 2) {
            // wave 1's first candidate continues wave 0's last read or heads a new one
            if (wave == 0u && lane == 63u) xchg[0] = query;
            __syncthreads();
            if (wave == 1u && lane < (uint32_t)L) query_below = xchg[0];
        }
        const bool first = kShare == 1 ? lane < (uint32_t)L : (wave == 0u && lane < (uint32_t)L);
        const bool head = (first || query_below != query) && gl == 0u;
        const uint64_t heads = __ballot(head);
        uint32_t slot_base = 0u, nqslots = (uint32_t)__builtin_popcountll(heads);
        if constexpr (kShare == 2) {
            if (lane == 0u) xchg[1u + wave] = nqslots;
            __syncthreads();
            const uint32_t h0 = xchg[1], h1 = xchg[2];
            slot_base = wave == 0u ? 0u : h0;
            nqslots = h0 + h1;
        }
        const uint32_t qslot = slot_base + (uint32_t)__builtin_popcountll(heads & lanes_upto) - 1u;

        // More distinct queries than LDS slots: one pass per kQSlots queries.
        for (uint32_t base_slot = 0; base_slot < nqslots; base_slot += S::kQSlots) {
            const bool in_pass = qslot >= base_slot && qslot < base_slot + S::kQSlots;
            const uint32_t my_slot = in_pass ? qslot - base_slot : 0u;
            chunk_sync<kWaves>();                        // previous readers of qtab / lds are done
            if (in_pass && head) qtab[my_slot] = make_uint2(pos_entry, m);
            chunk_sync<kWaves>();
            stage_peq<L, W, kHost, 64u * kShare>(lds, qtab, min(nqslots - base_slot, (uint32_t)S::kQSlots), a.peq,
                                                 kShare == 1 ? lane : threadIdx.x);
            chunk_sync<kWaves>();
            const uint4 *lds_lane = lds + my_slot * (uint32_t)S::kSlotU4 + gl;
            const uint32_t ncols = in_pass ? ncols_live : 0u;
            // threshold of the group's top lane (-1: no early stop for this lane)
            int32_t kthr = -1;
            if constexpr (kStop) {
                if (a.threshold >= 0.0f && live && in_pass && gl == (uint32_t)(L - 1))
                    kthr = (int32_t)threshold_of(m, a.threshold);
            }

            // Steps: the top lane of a group finishes column ncols-1 at step
            // ncols-1 + L-1.  Lane gl reads text from nibble nib0 - gl.
            const uint32_t max_cols = wave_max(ncols);
            const uint32_t nblocks = (max_cols + (uint32_t)(L - 1) + 7u) >> 3;
            const int64_t q = (int64_t)nib0 - (int64_t)gl;
            const int32_t w0 = (int32_t)(q >> 3);            // floor
            const uint32_t shift = (uint32_t)(q & 7) * 4u;

            uint32_t Pv[W], Mv[W];
#pragma unroll
            for (int k = 0; k < W; k++) {
                Pv[k] = ~0u;
                Mv[k] = 0u;
            }
            int32_t score = (int32_t)m, min_score = (int32_t)m;
            uint32_t min_col = 0;
            uint32_t ph_top = 0, mh_top = 0;
            // Cut-off state: rows with D <= k (k + pad in layout rows, where
            // the pad rows below the query hold D = row) must lie in the
            // first ga groups, 8 rows below its top.  Groups hold 128 rows,
            // the top one 32 (W - 4 (kG - 1)).  Start with every lane's rows
            // 0..kv+8 covered; D at the top row R of group ga-1 is then R.
            constexpr uint32_t kG = (uint32_t)((W + 3) / 4);
            constexpr int32_t kTopRows = 32 * (W - 4 * ((W + 3) / 4 - 1));
            int32_t kv = 0;
            uint32_t ga = kG;
            if constexpr (kUkk) {
                kv = (int32_t)threshold_of(m, a.threshold) + (32 * W - (int32_t)m);
                ga = min(wave_max(ncols > 0u ? ((uint32_t)kv + 135u) / 128u : 1u), kG);
                score = ga == kG ? 32 * W : 128 * (int32_t)ga;
            }

            // Text words stream through registers two blocks (16 columns) ahead
            // of their use; the Eq words of step t+1 are read from LDS while
            // step t computes.  Reads outside the stored reference are clamped
            // to its first / last (all-N guard) word; they only feed steps that
            // no lane keeps.
            auto text_word = [&](int32_t k) { return ref[min(max(w0 + k, 0), last_word)]; };
            auto text_block = [&](uint32_t lo, uint32_t hi, uint32_t b) {
                uint32_t t = sanitize_text(__builtin_amdgcn_alignbit(hi, lo, shift));
                if constexpr (L > 1) {
                    // steps before this lane's first column read the zero row
                    const int32_t early = (int32_t)gl - 8 * (int32_t)b;     // such steps in this block
                    if (early > 0) {
                        const uint32_t low = early >= 8 ? ~0u : ((1u << (4 * early)) - 1u);
                        t = (t & ~low) | (0x55555555u & low);
                    }
                }
                return t;
            };
            const uint32_t tw0 = text_word(0);
            const uint32_t tw1 = text_word(1);
            uint32_t tw2 = text_word(2);
            uint32_t tw3 = text_word(3);
            uint32_t text = text_block(tw0, tw1, 0);
            uint32_t text_next = text_block(tw1, tw2, 1);
            uint32_t cur_off = (text & 7u) * S::kRowU4;
            uint4 eq4 = lds_lane[cur_off];
            for (uint32_t b = 0; b < nblocks; b++) {
                const uint32_t tw4 = text_word((int32_t)b + 4);
                if constexpr (kUkk) {
                    // The extent changes only between blocks of 8 columns.  A row
                    // with D <= k in column j + t lies at most t + 1 rows above
                    // the last such row of column j - 1, so the extent must keep
                    // 8 rows of headroom over it: rows R-7..R with D <= k force
                    // D(R) <= k + 7 (one group is added), and a group can go
                    // when its rows and the 8 below it exceed k: D(R) > k + 135
                    // (for the shorter top group a stricter test than needed).
                    const bool on = 8u * b < ncols;
                    if (ga < kG && __ballot(on && score <= kv + 7) != 0ull) {
                        // new group: D rises by one per row above R (Pv = ~0, Mv = 0)
#pragma unroll
                        for (int g = 1; g < (int)kG; g++) {
                            const bool sel = (uint32_t)g == ga;
#pragma unroll
                            for (int k = 4 * g; k < 4 * g + 4 && k < W; k++) {
                                Pv[k] = sel ? ~0u : Pv[k];
                                Mv[k] = sel ? 0u : Mv[k];
                            }
                        }
                        score += ga + 1u == kG ? kTopRows : 128;
                        ga++;
                    } else if (ga > 1u && __ballot(on && score <= kv + 135) == 0ull) {
                        // drop group ga-1: S moves down by its vertical deltas
#pragma unroll
                        for (int g = 1; g < (int)kG; g++) {
                            if ((uint32_t)g + 1u == ga) {
                                int32_t dv = 0;
#pragma unroll
                                for (int k = 4 * g; k < 4 * g + 4 && k < W; k++)
                                    dv += __builtin_popcount(Pv[k]) - __builtin_popcount(Mv[k]);
                                score -= dv;
                            }
                        }
                        ga--;
                    }
                }
                const uint32_t ga_s = __builtin_amdgcn_readfirstlane(ga);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint32_t cn = (i < 7) ? ((text >> (4 * (i + 1))) & 7u) : (text_next & 7u);
                    const uint32_t next_off = cn * S::kRowU4;
                    if constexpr (L == 1) {
                        const uint4 eq4n = lds_lane[next_off];        // next column, group 0
                        if constexpr (kUkk) {
                            column_cut<0, W, (uint32_t)S::kGroupU4>(Pv, Mv, eq4, lds_lane, cur_off, ga_s, 0u, 0u,
                                                                   0u, ph_top, mh_top);
                        } else {
                            column_grp<W, false, (uint32_t)S::kGroupU4>(Pv, Mv, eq4, lds_lane, cur_off, 0u, 0u,
                                                                       ph_top, mh_top);
                        }
                        eq4 = eq4n;
                        score += (int32_t)(ph_top >> 31) - (int32_t)(mh_top >> 31);
                        const uint32_t col = 8u * b + (uint32_t)i;
                        const bool on = col < ncols;
                        if constexpr (!kUkk) {
                            // first minimum of the score row (src-api/coreMyersGPU-CC35.cu:205-207,227-228)
                            const bool better = (score < min_score) && on;
                            min_col = better ? col : min_col;
                            min_score = better ? score : min_score;
                        } else {
                            if (ga == kG) {
                                // score is D at row m plus the pad rows below the query
                                const int32_t d = score - (32 * W - (int32_t)m);
                                const bool better = (d < min_score) && on;
                                min_col = better ? col : min_col;
                                min_score = better ? d : min_score;
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    } else {
                        const uint4 eq4n = lds_lane[next_off];        // next column, group 0
                        const uint32_t ph_in = from_lower_lane<L>(ph_top, not_first);
                        const uint32_t mh_in = from_lower_lane<L>(mh_top, not_first);
                        column_grp<W, true, (uint32_t)S::kGroupU4, kWaves == 1>(
                            Pv, Mv, eq4, lds_lane, cur_off, ph_in, mh_in, ph_top, mh_top);
                        eq4 = eq4n;
                        // score row and first minimum (src-api/coreMyersGPU-CC35.cu:205-207,227-228);
                        // only the group's top lane keeps them, at column t - (L-1)
                        score += (int32_t)(ph_top >> 31) - (int32_t)(mh_top >> 31);
                        const uint32_t col = 8u * b + (uint32_t)i - (uint32_t)(L - 1);
                        const bool better = (score < min_score) && (col < ncols);
                        min_col = better ? col : min_col;
                        min_score = better ? score : min_score;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    cur_off = next_off;
                }
                text = text_next;
                text_next = text_block(tw2, tw3, b + 2);
                tw2 = tw3;
                tw3 = tw4;
                if constexpr (kStop) {
                    // Threshold mode: the score row moves by at most 1 per column, so a
                    // candidate whose minimum so far and whose score less the columns
                    // left both exceed the threshold cannot get under it.  The wave
                    // stops once each of its candidates has finished or is in that state.
                    if (a.threshold >= 0.0f) {
                        const int32_t col = (int32_t)(8u * b + 7u) - (L - 1);
                        const bool hopeless = col >= 0 && min_score > kthr &&
                                              score - ((int32_t)ncols - 1 - col) > kthr;
                        const bool running = kthr >= 0 && col < (int32_t)ncols - 1 && !hopeless;
                        if (__ballot(running) == 0ull) break;
                    }
                }
            }

            if (in_pass && valid && gl == (uint32_t)(L - 1)) {
                uint2 r = live ? make_uint2(min_col, (uint32_t)min_score) : make_uint2(0u, kSkipScore);
                // threshold mode: score <= (uint32)((float)m * e) (src/checksum-2.c:88,104-105)
                if (live && a.threshold >= 0.0f && (uint32_t)min_score > threshold_of(m, a.threshold))
                    r = make_uint2(kNoMatch, kNoMatch);
                st_result<kHost>(results + cand, r);
            }
        }
    }
}

// Take the next range of work items [lo, hi) for a persistent workgroup from
// the variant's queue: items [0, n) are split into one part per XCD, a
// workgroup starts on the part of the XCD it runs on (workgroups are
// dispatched round-robin over the 8 XCDs) and moves on to the other parts
// when its own is drained, so the atomics of one part stay within one XCD
// until the tail.  Each pull takes a guided share of what is left in the
// part, an eighth of an even split over the part's workgroups (at least
// min_take items), so long-running items still balance at the tail.  Thread 0 only; *part counts the parts
// this workgroup has found drained.  Returns false when all are.
__device__ __forceinline__ bool pull_work(uint32_t *heads, uint32_t n, uint32_t min_take, uint32_t &part,
                                          uint32_t &lo, uint32_t &hi) {
    const uint32_t xcd = blockIdx.x % (uint32_t)MYERS_QUEUE_PARTS;
    const uint32_t workers = max(1u, gridDim.x / (uint32_t)MYERS_QUEUE_PARTS);
    while (part < (uint32_t)MYERS_QUEUE_PARTS) {
        const uint32_t x = (xcd + part) % (uint32_t)MYERS_QUEUE_PARTS;
        const uint32_t p_lo = (uint32_t)(((uint64_t)n * x) / MYERS_QUEUE_PARTS);
        const uint32_t p_hi = (uint32_t)(((uint64_t)n * (x + 1u)) / MYERS_QUEUE_PARTS);
        uint32_t *head = heads + x * (uint32_t)MYERS_QUEUE_STRIDE;
        const uint32_t seen = __hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t left = (p_hi - p_lo) > seen ? (p_hi - p_lo) - seen : 0u;
        if (left == 0u) {                               // drained: no atomic needed
            part++;
            continue;
        }
        const uint32_t take = max(min_take, left / (8u * workers));
        const uint32_t got = atomicAdd(head, take);
        if (got < p_hi - p_lo) {
            lo = p_lo + got;
            hi = min(p_hi, lo + take);
            return true;
        }
        part++;
    }
    return false;
}

// Waves per SIMD the register allocator must leave room for (1 = no limit).
// The wide one-lane kernels fit 3 (<= 168 VGPRs) or 4 (<= 128); more
// resident waves keep the double-rate logic ops issuing.  The cut-off
// kernels for W >= 28 then spill a few per-chunk values, outside the column
// loop.
template <int L, int W, bool kCut, bool kPersistent>
constexpr int kWavesPerEU = L != 1 ? 1 : (W >= 28 ? 3 : (W >= 20 ? ((!kPersistent && !kCut) ? 4 : 3) : 1));

// Variants with a threshold-mode kernel: the cut-off (L = 1, W >= 8) or the
// early stop (multi-lane).
template <int L, int W>
constexpr bool kHasCut = (L == 1 && W >= 8) || (L > 1 && L <= 64);

// Issue priority of a variant's waves (s_setprio).  A wave of a long read
// runs one candidate's chain of dependent column steps, and the chain of the
// longest candidate sets the time of its batch; so the arbiter of a shared
// SIMD serves waves of longer reads first and short-read waves fill the other
// issue slots.  Where every wave of a SIMD is of one kind nothing changes.
template <int L>
constexpr int kWavePrio = L >= 64 ? 3 : (L >= 16 ? 2 : (L >= 4 ? 1 : 0));

template <int L>
__device__ __forceinline__ void set_wave_prio() {
    if constexpr (kWavePrio<L> > 0) __builtin_amdgcn_s_setprio(kWavePrio<L>);
}

// (L, W) pairs compiled into the library.  L = 1 covers queries up to
// 32*32 = 1024 bases in one lane; L > 1 covers long reads (up to 64*12*32 =
// 24576 bases).
#define MYERS_VARIANT_LIST(X)                                                                    \
    X(1, 1) X(1, 2) X(1, 3) X(1, 4) X(1, 5) X(1, 6) X(1, 7) X(1, 8) X(1, 9) X(1, 10) X(1, 11)     \
    X(1, 12) X(1, 13) X(1, 14) X(1, 15) X(1, 16) X(1, 17) X(1, 18) X(1, 19) X(1, 20) X(1, 21)    \
    X(1, 22) X(1, 23) X(1, 24) X(1, 25) X(1, 26) X(1, 27) X(1, 28) X(1, 29) X(1, 30) X(1, 31)    \
    X(1, 32)                                                                                     \
    X(2, 8) X(2, 12) X(2, 16) X(4, 8) X(4, 12) X(4, 16) X(8, 8) X(8, 12) X(8, 16)                \
    X(16, 8) X(16, 9) X(16, 10) X(16, 11) X(16, 12) X(16, 16) X(32, 7) X(32, 8) X(32, 9)          \
    X(32, 10) X(32, 11) X(32, 12) X(32, 16) X(64, 7) X(64, 8) X(64, 9) X(64, 10) X(64, 12)

// Multi-wave variants (lanes = 64 Q per candidate, one candidate per
// workgroup of Q waves): long reads with lower per-candidate latency.
#define MYERS_WIDE_LIST(X) X(2, 4) X(2, 6) X(4, 2) X(4, 3)

// Classes of the queue launches: one-lane variants (myers_slice.hip) and
// multi-lane ones of up to 12 words per lane (W = 16 would leave two waves
// per SIMD for every bin of the launch).
template <int L, int W>
constexpr int kQueueClass = L == 1 ? MYERS_QUEUE_ONE_LANE : ((L <= 64 && W <= 12) ? MYERS_QUEUE_MULTI_LANE : -1);


}  // namespace

#endif
