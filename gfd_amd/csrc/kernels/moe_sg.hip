// MoE-routed scattered gather with a wave-specialised RMSNorm consumer (gfx950).
//
// Role in the reference: the SG warp-specialised path (include/gfd/sg_warp_spec.cuh:
// a transfer warp turns per-expert (src, dst, size) lists into copies, a compute
// warp runs a functor on each list once it has landed; examples/09_sg_warp_spec.cu
// builds the lists on the GPU).  Here the whole path stays on the GPU:
//
//   1. moe_top2_kernel   — top-2 experts per token from the logits (ties go to
//                          the lower expert id), 16 lanes per token.
//   2. moe_lists_kernel  — one workgroup per expert builds its row list in token
//                          order (stable; no atomics), plus the expert offsets.
//                          Rows are packed expert-major.
//   3. sg_gather_norm_kernel<P, C, V> — per workgroup, P producer waves read whole
//                          rows straight from pinned host memory (16-byte loads
//                          over PCIe), write them to HBM and into an LDS ring of
//                          S row slots; C consumer waves wait on the slot flags
//                          (LDS acquire + s_sleep), compute a bf16 RMSNorm of the
//                          row in fp32 and write it to HBM, then free the slot.
//                          C = 0 is the pure-transfer variant.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

#include "capi_error.h"
#include "gfd/wave_ops.h"
#include "gfd_capi.h"

// Scratch of gfd_moe_route_noalloc: the top-2 expert pairs between its two
// kernels, for up to kNoAllocMaxTokens tokens (512 KiB per GPU, held until the
// process ends).  Host code never uses this name as an address: each
// device's copy is reached through the pointer hipGetSymbolAddress returns
// for it (moe_scratch_ptr below).
constexpr int kNoAllocMaxTokens = 65536;
static __device__ __align__(256) int scratch[2 * kNoAllocMaxTokens];

namespace {

constexpr int kWave = 64;
constexpr int kSlots = 4;              // LDS ring depth per workgroup
constexpr int kMaxRowBytes = 14336;    // 7168 bf16
constexpr uint64_t kSpinLimit = 1ull << 26;  // LDS flag polls before giving up

// ---------------------------------------------------------------- routing

// A token's experts are shared by 16 lanes, four each (lane l: experts l, l +
// 16, l + 32, l + 48, -inf where there is none).
constexpr int kTokLanes = 16, kTokExperts = 64 / kTokLanes;

// Reductions over a token's lanes, one DPP row, in every lane: l with 15 - l,
// with 7 - l in each half, then l ^ 2 and l ^ 1.  Each step is one
// instruction; as LDS permutes, or carrying (value, expert) pairs through
// compares and selects, they bound a workgroup of 16 waves.
template <int kCtrl>
__device__ __forceinline__ int dpp(int v) { return __builtin_amdgcn_mov_dpp(v, kCtrl, 0xF, 0xF, true); }
__device__ __forceinline__ float row_max(float v) {
    v = fmaxf(v, __int_as_float(dpp<0x140>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(dpp<0x141>(__float_as_int(v))));
    v = fmaxf(v, __int_as_float(dpp<0x4E>(__float_as_int(v))));
    return fmaxf(v, __int_as_float(dpp<0xB1>(__float_as_int(v))));
}
__device__ __forceinline__ int row_min(int v) {
    v = min(v, dpp<0x140>(v));
    v = min(v, dpp<0x141>(v));
    v = min(v, dpp<0x4E>(v));
    return min(v, dpp<0xB1>(v));
}

// The lowest expert that holds the largest of the token's logits, in every
// lane.  A NaN ranks behind everything; `none` if all are NaN.
__device__ __forceinline__ int argmax16(const float (&x)[kTokExperts], int num_experts, int lane, int none) {
    const float top = row_max(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])));
    int i = 64;
#pragma unroll
    for (int k = kTokExperts - 1; k >= 0; k--) i = x[k] == top ? lane + k * kTokLanes : i;
    i = row_min(i);
    return i < num_experts ? i : none;
}

typedef int int2v __attribute__((ext_vector_type(2), aligned(4)));

// The lane's logits of token min(t, num_tokens - 1), one token per 16 lanes.
__device__ __forceinline__ void load_logits(float (&x)[kTokExperts], const float* __restrict__ logits, int t,
                                            int num_tokens, int num_experts, int lane) {
    const float* row = logits + (size_t)min(t, num_tokens - 1) * num_experts;
#pragma unroll
    for (int k = 0; k < kTokExperts; k++) {
        // Past the last expert: a valid load whose value is not kept.
        const int e = lane + k * kTokLanes;
        const float v = row[min(e, num_experts - 1)];
        x[k] = e < num_experts ? v : -INFINITY;
    }
}

// The token's two experts, in all of its lanes: always two, since the lists
// hold a row per choice.  The first leaves the second pass as a NaN, which no
// logit ties with (-inf may be the largest that is left); where only NaNs are
// left, the lowest other expert is taken.
__device__ __forceinline__ int2v top2_of(float (&x)[kTokExperts], int num_experts, int lane) {
    const int first = argmax16(x, num_experts, lane, 0);
#pragma unroll
    for (int k = 0; k < kTokExperts; k++)
        if (lane + k * kTokLanes == first) x[k] = __builtin_nanf("");
    return int2v{first, argmax16(x, num_experts, lane, first == 0 ? 1 : 0)};
}

// Latency bound: 4 loads, then two chains of 8 cross-lane steps.  16 tokens
// per workgroup, so that 4096 tokens reach every CU (2.4 us; 3.8 with a wave
// and 24 LDS permutes per token); 2 or 4 tokens per 16 lanes were slower from
// 10000 tokens on.
constexpr int kTop2Block = 256, kTokBlock = kTop2Block / kTokLanes;
__global__ __launch_bounds__(kTop2Block) void moe_top2_kernel(const float* __restrict__ logits, int num_tokens,
                                                              int num_experts, int* __restrict__ top2) {
    const int lane = (int)(threadIdx.x % kTokLanes);
    const int t = (int)(blockIdx.x * kTokBlock + threadIdx.x / kTokLanes);
    float x[kTokExperts];
    load_logits(x, logits, t, num_tokens, num_experts, lane);
    const int2v p = top2_of(x, num_experts, lane);
    if (lane == 0 && t < num_tokens) *reinterpret_cast<int2v*>(top2 + 2 * (size_t)t) = p;
}

// Workgroup e: offsets[e] = number of (token, choice) pairs routed to experts
// below e; row_token[offsets[e] + k] = k-th token (in token order) routed to e.
// pair(t) gives token t's two experts.  The workgroup's 16 waves own one run
// of tokens each.  Pass 1 counts the run's hits and the pairs below e, U reads
// in flight per lane; one exchange of the waves' counts gives every wave its
// first slot; pass 2 places the run's hits by ballots.  Runs of at most 64 U
// tokens (1024 U in all) stay in registers between the passes.  Bound by the
// latency of the reads: at 4096 x 64 a kernel that walked all pairs twice with
// 4 waves, one read in flight and two barriers per 256 tokens took 14.0 us,
// this one 4.4; the whole routing 16.6 -> 9.2 us a call, at 20000 x 64 66 ->
// 12.3, at 65536 x 64 204 -> 29.
constexpr int kListWaves = 16;
template <int U, typename Pair>
__device__ __forceinline__ void place_rows(Pair pair, int num_tokens, int num_experts, int* __restrict__ offsets,
                                           int* __restrict__ row_token) {
    __shared__ int wave_hits[kListWaves], wave_below[kListWaves];
    const int e = (int)blockIdx.x;
    const int lane = (int)(threadIdx.x % kWave), wave = (int)(threadIdx.x / kWave);
    // Runs are whole groups of 64 tokens.
    const int groups = (num_tokens + kWave - 1) / kWave;
    const int per = (groups + kListWaves - 1) / kListWaves;
    const int g0 = min(wave * per, groups), g1 = min(g0 + per, groups);
    int2v p[U];
    auto read = [&](int g) {
#pragma unroll
        for (int k = 0; k < U; k++) {
            const int t = (g + k) * kWave + lane;
            const int2v v = pair(min(t, num_tokens - 1));
            p[k] = g + k < g1 && t < num_tokens ? v : int2v{-1, -1};
        }
    };
    int hits = 0, below = 0;
    for (int g = g0; g < g1; g += U) {
        read(g);
#pragma unroll
        for (int k = 0; k < U; k++) {
            hits += __popcll(__ballot(p[k].x == e || p[k].y == e));
            below += __popcll(__ballot((uint32_t)p[k].x < (uint32_t)e)) +
                     __popcll(__ballot((uint32_t)p[k].y < (uint32_t)e));
        }
    }
    if (lane == 0) {
        wave_hits[wave] = hits;
        wave_below[wave] = below;
    }
    __syncthreads();
    int at = 0;
#pragma unroll
    for (int w = 0; w < kListWaves; w++) at += wave_below[w] + (w < wave ? wave_hits[w] : 0);
    if (threadIdx.x == 0) {
        offsets[e] = at;
        if (e == num_experts - 1) offsets[num_experts] = 2 * num_tokens;
    }
    const uint64_t lower = (1ull << lane) - 1ull;
    for (int g = g0; g < g1; g += U) {
        if (per > U) read(g);
#pragma unroll
        for (int k = 0; k < U; k++) {
            const bool hit = p[k].x == e || p[k].y == e;
            const uint64_t mask = __ballot(hit);
            if (hit) row_token[at + __popcll(mask & lower)] = (g + k) * kWave + lane;
            at += __popcll(mask);
        }
    }
}

__global__ __launch_bounds__(kListWaves * 64) void moe_lists_kernel(const int* __restrict__ top2, int num_tokens,
                                                                   int num_experts, int* __restrict__ offsets,
                                                                   int* __restrict__ row_token) {
    place_rows<8>([=](int t) { return *reinterpret_cast<const int2v*>(top2 + 2 * (size_t)t); }, num_tokens,
                  num_experts, offsets, row_token);
}

// Both steps in one launch for few tokens: every expert's workgroup works the
// pairs of all tokens out again, into LDS, and writes its share of top2.  The
// work repeated costs 0.6 us per 64 tokens and the launch saved 4.3 us, so up
// to 512 tokens: 60 x 4 9.6 -> 6.8 us a call, 256 x 64 9.3 -> 6.6, 512 x 64
// 9.3 -> 7.5 (1000 x 16 would be 12.2 against 9.0).
constexpr int kFusedTokens = 512;
__global__ __launch_bounds__(kListWaves * 64) void moe_route_kernel(const float* __restrict__ logits, int num_tokens,
                                                                   int num_experts, int* __restrict__ top2,
                                                                   int* __restrict__ offsets,
                                                                   int* __restrict__ row_token) {
    __shared__ int2v pairs[kFusedTokens];
    constexpr int kGroups = kListWaves * kWave / kTokLanes;  // tokens at a time
    constexpr int kAhead = 4;                                // of each group's, loaded together
    const int lane = (int)(threadIdx.x % kTokLanes), group = (int)(threadIdx.x / kTokLanes);
    for (int t0 = group; t0 < num_tokens; t0 += kAhead * kGroups) {
        float x[kAhead][kTokExperts];
#pragma unroll
        for (int a = 0; a < kAhead; a++) load_logits(x[a], logits, t0 + a * kGroups, num_tokens, num_experts, lane);
#pragma unroll
        for (int a = 0; a < kAhead; a++) {
            if (__builtin_amdgcn_readfirstlane(t0 + a * kGroups) >= num_tokens) break;  // none for the whole wave
            const int2v p = top2_of(x[a], num_experts, lane);
            if (lane == 0 && t0 + a * kGroups < num_tokens) pairs[t0 + a * kGroups] = p;
        }
    }
    __syncthreads();
    const int share = (num_tokens + (int)gridDim.x - 1) / (int)gridDim.x;
    const int s0 = (int)blockIdx.x * share, s1 = min(s0 + share, num_tokens);
    for (int t = s0 + (int)threadIdx.x; t < s1; t += kListWaves * kWave)
        *reinterpret_cast<int2v*>(top2 + 2 * (size_t)t) = pairs[t];
    place_rows<1>([&](int t) { return pairs[t]; }, num_tokens, num_experts, offsets, row_token);
}

// ------------------------------------------------------ gather + RMSNorm

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

// Round-to-nearest-even fp32 -> bf16 (finite values).
__device__ __forceinline__ uint32_t to_bf16(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ int lds_load_acquire(int* p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void lds_store_release(int* p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Wait until *flag == want; false if the spin limit ran out (the caller then
// skips its row and reports the error instead of hanging the workgroup).
__device__ __forceinline__ bool lds_wait(int* flag, int want) {
    for (uint64_t n = 0; n < kSpinLimit; n++) {
        if (lds_load_acquire(flag) == want) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}

// Workgroup b owns rows [b*R/G, (b+1)*R/G) of the expert-major row order.
// Row r copies token row_token[r] (host_base + token * token_stride,
// row_bytes = V * 1 KiB) to dst + r * row_bytes; with C > 0 it also writes
// RMSNorm(row) (bf16, weight w, epsilon eps) to out + r * row_bytes.
//
// V (16-byte vectors per lane) is a template parameter so that every lane's
// V loads are straight-line code: a guarded load sits in its own basic block,
// and the compiler then waits for all earlier loads before issuing it.  The
// vectors are native clang vectors so that they stay in registers.
template <int P, int C, int V>
__global__ __launch_bounds__(kWave*(P + C)) void sg_gather_norm_kernel(
    const uint8_t* __restrict__ host_base, uint64_t token_stride, int num_tokens, const int* __restrict__ row_token,
    int num_rows, uint8_t* __restrict__ dst, uint8_t* __restrict__ out, const uint16_t* __restrict__ weight,
    float eps, int* __restrict__ error_flag) {
    using gfd::wave::vec4u;
    constexpr uint32_t row_bytes = (uint32_t)V * kWave * 16;
    __shared__ vec4u ring[C > 0 ? kSlots : 1][V * kWave];
    __shared__ vec4u wlds[C > 0 ? V * kWave : 1];  // RMSNorm weights, staged once per workgroup
    __shared__ int slot_row[kSlots];
    const int wave = (int)(threadIdx.x / kWave);
    const int lane = (int)(threadIdx.x % kWave);
    const int r0 = (int)(((int64_t)blockIdx.x * num_rows) / gridDim.x);
    const int r1 = (int)(((int64_t)(blockIdx.x + 1) * num_rows) / gridDim.x);
    const int rows = r1 - r0;

    if (C > 0) {
        if (threadIdx.x < kSlots) slot_row[threadIdx.x] = 0;
        for (uint32_t k = threadIdx.x; k < (uint32_t)(V * kWave); k += blockDim.x)
            wlds[k] = gfd::wave::gload((uint64_t)(uintptr_t)weight + (uint64_t)k * 16);
        __syncthreads();
    }

    if (wave < P) {
        // ---------------- producer waves
        for (int i = wave; i < rows; i += P) {
            const int r = r0 + i;
            const int s = i % kSlots;
            if (C > 0 && !lds_wait(&slot_row[s], 0)) {
                if (lane == 0) atomicOr(error_flag, 1);
                return;
            }
            const int tok = row_token[r];
            if (tok < 0 || tok >= num_tokens) {  // not a valid token: report, keep the ring moving
                if (lane == 0) atomicOr(error_flag, 4);
                if (C > 0) lds_store_release(&slot_row[s], i + 1);
                continue;
            }
            const uint64_t src = (uint64_t)(uintptr_t)host_base + (uint64_t)tok * token_stride;
            const uint64_t d = (uint64_t)(uintptr_t)dst + (uint64_t)r * row_bytes;
            vec4u v[V];
#pragma unroll
            for (int k = 0; k < V; k++) v[k] = gfd::wave::gload(src + (uint64_t)(k * kWave + lane) * 16);
#pragma unroll
            for (int k = 0; k < V; k++) gfd::wave::gstore(d + (uint64_t)(k * kWave + lane) * 16, v[k]);
            if (C > 0) {
#pragma unroll
                for (int k = 0; k < V; k++) ring[s][k * kWave + lane] = v[k];
                lds_store_release(&slot_row[s], i + 1);
            }
        }
    } else if (C > 0) {
        // ---------------- consumer waves
        const int c = wave - P;
        const float inv_dim = 1.0f / (float)(row_bytes / 2);
        for (int i = c; i < rows; i += C) {
            const int r = r0 + i;
            const int s = i % kSlots;
            if (!lds_wait(&slot_row[s], i + 1)) {
                if (lane == 0) atomicOr(error_flag, 2);
                return;
            }
            vec4u x[V];
            float ss = 0.f;
#pragma unroll
            for (int k = 0; k < V; k++) {
                x[k] = ring[s][k * kWave + lane];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float a = bf16_lo(x[k][j]), b = bf16_hi(x[k][j]);
                    ss += a * a + b * b;
                }
            }
            lds_store_release(&slot_row[s], 0);  // row is in registers: free the slot
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, kWave);
            const float scale = 1.0f / sqrtf(ss * inv_dim + eps);
            const uint64_t o = (uint64_t)(uintptr_t)out + (uint64_t)r * row_bytes;
#pragma unroll
            for (int k = 0; k < V; k++) {
                const vec4u wk = wlds[k * kWave + lane];
                vec4u y;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float lo = bf16_lo(x[k][j]) * scale * bf16_lo(wk[j]);
                    const float hi = bf16_hi(x[k][j]) * scale * bf16_hi(wk[j]);
                    y[j] = to_bf16(lo) | (to_bf16(hi) << 16);
                }
                gfd::wave::gstore(o + (uint64_t)(k * kWave + lane) * 16, y);
            }
        }
    }
}

template <int V>
void launch_gather_norm(const void* host_base, uint64_t token_stride, int num_tokens, const int* row_token,
                        int num_rows, void* dst, void* out, const uint16_t* weight, float eps, int num_blocks,
                        int* error_flag, hipStream_t st) {
    if (out)
        hipLaunchKernelGGL((sg_gather_norm_kernel<4, 4, V>), dim3(num_blocks), dim3(kWave * 8), 0, st,
                           (const uint8_t*)host_base, token_stride, num_tokens, row_token, num_rows, (uint8_t*)dst,
                           (uint8_t*)out, weight, eps, error_flag);
    else
        hipLaunchKernelGGL((sg_gather_norm_kernel<4, 0, V>), dim3(num_blocks), dim3(kWave * 4), 0, st,
                           (const uint8_t*)host_base, token_stride, num_tokens, row_token, num_rows, (uint8_t*)dst,
                           (uint8_t*)nullptr, weight, eps, error_flag);
}

int g_cus = 0;
int cus() {
    if (!g_cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&g_cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || g_cus <= 0)
            g_cus = 256;
    }
    return g_cus;
}

// Device address of this device's `scratch`, looked up once per device with
// that device current; 0 or a HIP error.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int moe_scratch_ptr(int** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol;
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<int*>(g_scratch_ptr[dev]);
    return 0;
}

int launch_route(const float* logits, int num_tokens, int num_experts, int* top2, int* offsets, int* row_token,
                 hipStream_t st) {
    if (num_tokens <= kFusedTokens) {
        hipLaunchKernelGGL(moe_route_kernel, dim3(num_experts), dim3(kListWaves * kWave), 0, st, logits, num_tokens,
                           num_experts, top2, offsets, row_token);
        return (int)hipGetLastError();
    }
    hipLaunchKernelGGL(moe_top2_kernel, dim3((num_tokens + kTokBlock - 1) / kTokBlock), dim3(kTop2Block), 0, st,
                       logits, num_tokens, num_experts, top2);
    hipLaunchKernelGGL(moe_lists_kernel, dim3(num_experts), dim3(kListWaves * kWave), 0, st, top2, num_tokens,
                       num_experts, offsets, row_token);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int gfd_moe_route_noalloc(const float* logits, int num_tokens, int num_experts, int* offsets,
                                     int* row_token, void* stream) {
    if (num_tokens <= 0 || num_experts < 2 || num_experts > 64 || !logits || !offsets || !row_token) {
        gfd_internal_set_error("gfd_moe_route_noalloc: invalid argument");
        return (int)hipErrorInvalidValue;
    }
    if (num_tokens > kNoAllocMaxTokens) {
        gfd_internal_set_error("gfd_moe_route_noalloc: num_tokens exceeds the scratch maximum of 65536 tokens");
        return (int)hipErrorInvalidValue;
    }
    int* top2 = nullptr;
    const int rc = moe_scratch_ptr(&top2);
    if (rc != 0) {
        gfd_internal_set_error("gfd_moe_route_noalloc: hipGetSymbolAddress of the scratch array failed");
        return rc;
    }
    return launch_route(logits, num_tokens, num_experts, top2, offsets, row_token, (hipStream_t)stream);
}

extern "C" int gfd_moe_route(const float* logits, int num_tokens, int num_experts, int* top2, int* offsets,
                             int* row_token, void* stream) {
    if (num_tokens <= 0 || num_experts < 2 || num_experts > 64 || !logits || !top2 || !offsets || !row_token)
        return (int)hipErrorInvalidValue;
    return launch_route(logits, num_tokens, num_experts, top2, offsets, row_token, (hipStream_t)stream);
}

extern "C" int gfd_sg_gather_rmsnorm(const void* host_base, uint64_t token_stride, int num_tokens, const int* row_token,
                                     int num_rows, uint32_t row_bytes, void* dst, void* out, const uint16_t* weight,
                                     float eps, int num_blocks, int* error_flag, void* stream) {
    if (num_rows < 0 || num_tokens <= 0 || !host_base || !row_token || !dst || !error_flag || row_bytes == 0 ||
        row_bytes % (kWave * 16) != 0 || row_bytes > (uint32_t)kMaxRowBytes || (out && !weight))
        return (int)hipErrorInvalidValue;
    if (num_rows == 0) return 0;
    // Default: 64 workgroups (256 producer waves, 14 loads in flight per lane,
    // ~3.5 MiB of host reads outstanding).  Measured on MI355X for 8192 rows
    // of 14 KiB: 57.7 GB/s at 32-96 workgroups, 55 GB/s at 192-256.
    if (num_blocks <= 0) num_blocks = cus() < 64 ? cus() : 64;
    if (num_blocks > num_rows) num_blocks = num_rows;
    hipStream_t st = (hipStream_t)stream;
    switch (row_bytes / (kWave * 16)) {
#define GFD_ROW_CASE(v)                                                                                          \
    case v:                                                                                                      \
        launch_gather_norm<v>(host_base, token_stride, num_tokens, row_token, num_rows, dst, out, weight, eps, \
                              num_blocks, error_flag, st);                                                      \
        break;
        GFD_ROW_CASE(1) GFD_ROW_CASE(2) GFD_ROW_CASE(3) GFD_ROW_CASE(4) GFD_ROW_CASE(5) GFD_ROW_CASE(6)
        GFD_ROW_CASE(7) GFD_ROW_CASE(8) GFD_ROW_CASE(9) GFD_ROW_CASE(10) GFD_ROW_CASE(11) GFD_ROW_CASE(12)
        GFD_ROW_CASE(13) GFD_ROW_CASE(14)
#undef GFD_ROW_CASE
        default:
            return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}
