// GPU-built SG lists for GFD Direct: the pattern of the reference's
// examples/03_gpu_planned_transfer.cu:32-66, where kernels select the tokens
// routed to one expert and write the SGEntry list straight into pinned host
// memory, and the host then hands that list to submit_direct.
//
// MI355X design: up to 8 workgroups of 16 waves own one range of tokens each,
// and a wave one run of its workgroup's range.  A wave reads its run kUnroll
// loads at a time and counts its matches by ballots; the workgroup counts the
// matches ahead of its range by itself (16-byte loads, so no scratch memory
// and no second launch); one exchange of the waves' counts gives every wave
// its first slot.  The list is in token order (stable) and the same on every
// run; the reference compacts with an atomicAdd per match, which orders slots
// by arrival.  Bound by the latency of the reads and of the records' way to
// pinned memory.  A call of 4096 tokens and 8 experts takes 4.6 us, of 65536
// 8.6; with one workgroup that took 1024 tokens at a time, two barriers each,
// 5.4 and 63.8 (a table in host memory: 6.5 and 27 against 9.6 and 131).  8
// workgroups at most, because each reads the table up to its own range, and
// the table may lie in host memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "gfd_capi.h"

namespace {

constexpr int kPlanWaves = 16, kPlanBlock = kPlanWaves * 64, kPlanGroups = 8, kUnroll = 8;

// Workgroup b owns tokens [b * range, (b + 1) * range); range is a multiple of kPlanBlock.
__global__ __launch_bounds__(kPlanBlock) void plan_expert_entries_kernel(
    const int* __restrict__ routing, int num_tokens, int range, int expert, uint64_t cpu_base, uint64_t stride,
    uint64_t gpu_dst, uint64_t token_size, gfd_sg_entry* __restrict__ entries, int* __restrict__ count) {
    typedef int int4v __attribute__((ext_vector_type(4), aligned(4)));
    __shared__ int wave_before[kPlanWaves], wave_hits[kPlanWaves];
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    const int first = (int)blockIdx.x * range;  // below num_tokens (0 if there are none)
    const int last = first + min(num_tokens - first, range);
    const int per = range / kPlanBlock;  // groups of 64 tokens of a wave's run
    const int run = first + wave * per * 64;

    int r[kUnroll];
    auto read = [&](int g) {
#pragma unroll
        for (int k = 0; k < kUnroll; k++) {
            const uint32_t t = (uint32_t)(run + lane) + (uint32_t)(g + k) * 64u;
            const bool in = g + k < per && t < (uint32_t)last;
            // Past the run: token 0, whose value is not kept (none at all without tokens).
            const int v = num_tokens > 0 ? routing[in ? t : 0u] : 0;
            r[k] = in ? (v == expert) : 0;
        }
    };
    read(0);
    // Matches ahead of the range, by all waves together.
    int before = 0;
    const int quads = first / 4;
    for (int q = 0; q < quads; q += kPlanBlock * kUnroll) {
        int4v v[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; k++)
            v[k] = *reinterpret_cast<const int4v*>(routing + 4 * min(q + k * kPlanBlock + (int)threadIdx.x, quads - 1));
#pragma unroll
        for (int k = 0; k < kUnroll; k++) {
            const int hits = (v[k].x == expert) + (v[k].y == expert) + (v[k].z == expert) + (v[k].w == expert);
            before += q + k * kPlanBlock + (int)threadIdx.x < quads ? hits : 0;
        }
    }
    int hits = 0;
    for (int g = 0; g < per; g += kUnroll) {
        if (g > 0) read(g);
#pragma unroll
        for (int k = 0; k < kUnroll; k++) hits += __popcll(__ballot(r[k]));
    }
    for (int off = 32; off >= 1; off >>= 1) before += __shfl_xor(before, off, 64);
    if (lane == 0) {
        wave_before[wave] = before;
        wave_hits[wave] = hits;
    }
    __syncthreads();
    int at = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kPlanWaves; w++) {
        total += wave_before[w] + wave_hits[w];
        at += wave_before[w] + (w < wave ? wave_hits[w] : 0);
    }
    const uint64_t lower = (1ull << lane) - 1ull;
    for (int g = 0; g < per; g += kUnroll) {
        if (per > kUnroll) read(g);
#pragma unroll
        for (int k = 0; k < kUnroll; k++) {
            const uint64_t mask = __ballot(r[k]);
            if (r[k]) {
                const uint64_t slot = (uint64_t)(at + __popcll(mask & lower));
                gfd_sg_entry e;
                e.dst = gpu_dst + slot * token_size;
                e.src = cpu_base + (uint64_t)(run + (g + k) * 64 + lane) * stride;
                e.size = token_size;
                entries[slot] = e;
            }
            at += __popcll(mask);
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *count = total;
}

}  // namespace

extern "C" int gfd_plan_expert_entries(const int* routing, int num_tokens, int expert, const void* cpu_base,
                                       uint64_t stride, void* gpu_dst, uint32_t token_size, gfd_sg_entry* entries,
                                       int* count, void* stream) {
    if (!routing || !entries || !count || num_tokens < 0 || token_size == 0)
        return (int)hipErrorInvalidValue;
    const int64_t blocks = std::max<int64_t>(1, ((int64_t)num_tokens + kPlanBlock - 1) / kPlanBlock);
    const int64_t per = (blocks + kPlanGroups - 1) / kPlanGroups;
    hipLaunchKernelGGL(plan_expert_entries_kernel, dim3((unsigned)((blocks + per - 1) / per)), dim3(kPlanBlock), 0,
                       (hipStream_t)stream, routing, num_tokens, (int)(per * kPlanBlock), expert,
                       (uint64_t)(uintptr_t)cpu_base, stride, (uint64_t)(uintptr_t)gpu_dst, (uint64_t)token_size,
                       entries, count);
    return (int)hipGetLastError();
}
