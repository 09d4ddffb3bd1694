// Reads of up to 1024 bases: the candidate-sliced kernel (myers_slice.h), the
// bit planes of the reference it reads, and their launch shims.
#include "myers_slice.h"

namespace {

// One kernel per form (SL lanes per group) for every engine.  It is compiled for
// three waves per SIMD (168 VGPRs): 32 rows per lane take 128, and three waves
// issue the double-rate operations at 0.41 per clock against 0.35 with two.
//   MYERS_SLICE_PLAIN  one bin, a fixed grid strides over its chunks
//   MYERS_SLICE_RANGES one bin, a resident grid pulls guided ranges of chunks
//   MYERS_SLICE_QUEUE  every bin of the plan, one chunk at a time from a
//                      single counter in plan order (longest reads first, so
//                      the grid's tail is short chunks)
template <int SL>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
void verify_slice_kernel(myers_verify_args_t a, myers_queue_plan_t p, uint32_t mode) {
    extern __shared__ uint4 slice_lds[];
    constexpr uint32_t kCands = (uint32_t)SliceShape<SL>::kCands;
    constexpr uint32_t kHead = MYERS_QUEUE_HEAD(SL == 16 ? MYERS_QUEUE_ONE_LANE_16 : MYERS_QUEUE_ONE_LANE);
    uint32_t next = blockIdx.x, lo = 0, hi = 0, part = 0;
    if (mode == (uint32_t)MYERS_SLICE_PLAIN && (gridDim.x & 7u) == 0u) {
        // Workgroups are dispatched round-robin over the 8 XCDs; renumber them so
        // that each XCD (own L2) takes a contiguous run of chunks.  Not where the
        // bin has fewer chunks than the grid workgroups: the first XCDs would take
        // them all (200K candidates of 36-400 bases, a launch per bin: 1.0 ms, 0.56).
        const uint32_t n = a.bin_ranges != nullptr ? a.bin_ranges[2u * p.variant[0] + 1u] : a.count;
        if (n > (gridDim.x - 1u) * kCands) next = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    }
    for (;;) {
        uint32_t j = 0, start = a.start, count = a.count, chunk = 0;
        if (mode == (uint32_t)MYERS_SLICE_QUEUE) {
            uint32_t got = 0;
            if (threadIdx.x == 0) got = atomicAdd(a.queue_heads + kHead, 1u);
            const uint32_t item = (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)got, 0));
            uint32_t base = 0;
            bool found = false;
            for (; j < p.n; j++) {
                const uint32_t c = a.bin_ranges[2u * p.variant[j] + 1u];
                const uint32_t chunks = (c + kCands - 1u) / kCands;
                if (item - base < chunks) {
                    start = a.bin_ranges[2u * p.variant[j]];
                    count = c;
                    found = true;
                    break;
                }
                base += chunks;
            }
            if (!found) break;                   // every bin drained: each wave exits here
            chunk = item - base;
        } else {
            if (a.bin_ranges != nullptr) {
                start = a.bin_ranges[2u * p.variant[0]];
                count = a.bin_ranges[2u * p.variant[0] + 1u];
            }
            const uint32_t chunks = (count + kCands - 1u) / kCands;
            if (mode == (uint32_t)MYERS_SLICE_PLAIN) {
                if (next >= chunks) break;
                chunk = next;
                next += gridDim.x;
            } else {
                if (lo >= hi) {
                    uint32_t got_lo = 0, got_hi = 0;
                    uint32_t *heads = a.queue_heads + p.variant[0] * (uint32_t)(MYERS_QUEUE_PARTS * MYERS_QUEUE_STRIDE);
                    if (threadIdx.x == 0 && !pull_work(heads, chunks, max(a.chunk_factor, 1u), part, got_lo, got_hi))
                        got_lo = got_hi = 0u;
                    lo = (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)got_lo, 0));
                    hi = (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)got_hi, 0));
                    if (lo >= hi) break;         // drained
                }
                chunk = lo++;
            }
        }
        // bins of form 1 run the bit-vector kernel (chunks of 64, as form 32)
        const uint32_t words = p.key[j] & 0xFFu;
        SliceDone done = kSliceRefused;
        if (p.key[j] >> 8 != 1u) {
            // first rows only, while they rule out enough: of `tally`'s
            // candidates a share below 0.75 of what the rows left out would cost
            uint32_t first = a.list != nullptr ? slice_first_rows<SL>(words, (float)threshold_of(32u * words, a.threshold)) : 0u;
            if (first != 0u) {
                const uint32_t tried = __hip_atomic_load(a.tally, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t kept = __hip_atomic_load(a.tally + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const float share = 0.75f * (1.0f - (float)(first * (uint32_t)SL) / (32.0f * (float)words));
                const bool go = tried < 16384u || (float)kept < share * (float)tried;
                first = (uint32_t)__builtin_amdgcn_readfirstlane(go ? (int)first : 0);
            }
            done = verify_slice<SL>(a, start, count, chunk, words, first, p.variant[j], slice_lds);
            if (done == kSliceShort) done = verify_slice<SL>(a, start, count, chunk, words, 0u, p.variant[j], slice_lds);
        }
        if (done != kSliceDone)
            slice_fallback<SL>(a, start, count, chunk, words, slice_lds);
    }
}

const void *slice_kernel(uint32_t lanes) {
    return lanes == 16u ? reinterpret_cast<const void *>(&verify_slice_kernel<16>)
                        : reinterpret_cast<const void *>(&verify_slice_kernel<32>);
}

uint32_t fallback_u4(uint32_t words) {
    size_t b = 0;
#define SLICE_FALLBACK_SIZE(WF) if (b == 0 && words <= (WF)) b = sizeof(Workspace<1, (WF)>);
    SLICE_FALLBACK_WIDTHS(SLICE_FALLBACK_SIZE)
#undef SLICE_FALLBACK_SIZE
    return (uint32_t)((b + 15u) / 16u);
}

// Bit planes of the packed reference: three words per block of 32 bases, the
// code's bit 0 and bit 1 (codes 5..7 read as A, sanitize_text) and the N flag.
// Words past the stored ones count as N.
__global__ __launch_bounds__(256) void planes_kernel(const uint32_t *ref, uint64_t ref_words, uint32_t *planes,
                                                     uint32_t nblocks) {
    const uint32_t blk = blockIdx.x * 256u + threadIdx.x;
    if (blk >= nblocks) return;
    uint32_t p[3] = {0u, 0u, 0u};
    for (uint32_t w = 0; w < 4u; w++) {
        const uint64_t at = 4ull * blk + w;
        const uint32_t t = sanitize_text(at < ref_words ? ref[at] : 0x44444444u);
        for (uint32_t q = 0; q < 3u; q++) {
            // bits 0, 4, .., 28 to bits 0..7
            uint32_t v = (t >> q) & 0x11111111u;
            v = (v | (v >> 3)) & 0x03030303u;
            v = (v | (v >> 6)) & 0x000F000Fu;
            p[q] |= ((v | (v >> 12)) & 0xFFu) << (8u * w);
        }
    }
    for (uint32_t q = 0; q < 3u; q++) planes[3ull * blk + q] = p[q];
}

}  // namespace

extern "C" uint32_t myers_slice_max_words(uint32_t lanes) {
    if (lanes == 1u) return kFallbackExact;
    return lanes == 16u || lanes == 32u ? (uint32_t)slice_max_words((int)lanes) : 0u;
}

extern "C" uint32_t myers_slice_first_rows(uint32_t words, float threshold) {
    return slice_first_rows<32>(words, floorf(32.0f * (float)words * threshold));
}

extern "C" uint32_t myers_slice_ws_u4(uint32_t lanes, uint32_t words) {
    if (words == 0u || words > myers_slice_max_words(lanes)) return 0u;
    if (lanes == 1u) return fallback_u4(words);
    const uint32_t u4 = (uint32_t)(lanes == 16u ? SliceShape<16>::ws_u4((int)words * 2) : SliceShape<32>::ws_u4((int)words));
    const uint32_t fb = fallback_u4(words);
    return u4 > fb ? u4 : fb;
}

extern "C" int myers_slice_occupancy(uint32_t lanes, uint32_t lds_bytes, int *wg_per_cu) {
    if (wg_per_cu == nullptr) return -1;
    int blocks = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, slice_kernel(lanes), 64, (size_t)lds_bytes);
    if (e != hipSuccess) return (int)e;
    *wg_per_cu = blocks;
    return 0;
}

extern "C" int myers_launch_slice(const myers_verify_args_t *args, const myers_queue_plan_t *plan, uint32_t mode,
                                  uint32_t grid, hipStream_t stream) {
    if (args == nullptr || plan == nullptr || grid == 0 || plan->n == 0 || plan->n > (uint32_t)MYERS_QUEUE_MAX ||
        args->planes == nullptr || args->plane_blocks == 0)
        return -1;
    if (mode > (uint32_t)MYERS_SLICE_QUEUE || (mode != (uint32_t)MYERS_SLICE_QUEUE && plan->n != 1u)) return -1;
    if (args->list != nullptr && (mode != (uint32_t)MYERS_SLICE_QUEUE || args->threshold < 0.0f ||
                                  args->list_ranges == nullptr || args->tally == nullptr))
        return -1;
    if (mode != (uint32_t)MYERS_SLICE_PLAIN && (args->bin_ranges == nullptr || args->queue_heads == nullptr)) return -1;
    const uint32_t lanes = plan->key[0] >> 8;
    if (plan->cls != (uint32_t)(lanes == 16u ? MYERS_QUEUE_ONE_LANE_16 : MYERS_QUEUE_ONE_LANE)) return -1;
    for (uint32_t j = 0; j < plan->n; j++) {
        if ((plan->key[j] >> 8 == 16u) != (lanes == 16u)) return -1;     // chunks of 128, or of 64
        const uint32_t need = myers_slice_ws_u4(plan->key[j] >> 8, plan->key[j] & 0xFFu);
        if (need == 0u || plan->ws_u4 < need || plan->variant[j] >= (uint32_t)MYERS_MAX_VARIANTS) return -1;
    }
    if (plan->ws_u4 * 16u > 64u * 1024u) return -1;
    void *kargs[] = {const_cast<myers_verify_args_t *>(args), const_cast<myers_queue_plan_t *>(plan), &mode};
    return (int)hipLaunchKernel(slice_kernel(lanes), dim3(grid), dim3(64), kargs, (size_t)plan->ws_u4 * 16u, stream);
}

extern "C" int myers_launch_planes(const uint32_t *ref, uint64_t ref_words, uint32_t *planes, uint32_t nblocks,
                                   hipStream_t stream) {
    if (ref == nullptr || planes == nullptr || nblocks == 0) return -1;
    hipLaunchKernelGGL(planes_kernel, dim3((nblocks + 255u) / 256u), dim3(256), 0, stream, ref, ref_words, planes,
                       nblocks);
    return (int)hipGetLastError();
}
