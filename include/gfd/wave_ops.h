#pragma once
// Wave64 building blocks shared by the gfx950 kernels (HIP sources only):
// whole-wave copies of host->HBM byte ranges, lane broadcasts, bounded LDS
// waits with s_sleep back-off, and the fences of the producer/consumer
// hand-off.
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gfd {
namespace wave {

constexpr int kWidth = 64;
// Polls of an LDS / memory flag before a wait gives up (~1-2 s with s_sleep 1).
constexpr uint64_t kSpinLimit = 1ull << 26;

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWidth - 1)); }
__device__ __forceinline__ int wave_id() { return (int)(threadIdx.x / kWidth); }

__device__ __forceinline__ uint64_t readlane64(uint64_t x, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t broadcast0(uint64_t x) { return readlane64(x, 0); }

// 16-byte vector as a native clang vector: arrays of these stay in VGPRs at
// any unroll (arrays of HIP's uint4 wrapper go to scratch from 8 on).
typedef uint32_t vec4u __attribute__((ext_vector_type(4)));
// Global-address-space views, so copies compile to global_load/global_store
// (flat instructions would also wait on the LDS counter).
typedef __attribute__((address_space(1))) vec4u gvec4u;

__device__ __forceinline__ vec4u gload(uint64_t a) { return *reinterpret_cast<const gvec4u*>(a); }
__device__ __forceinline__ void gstore(uint64_t a, vec4u v) { *reinterpret_cast<gvec4u*>(a) = v; }

// The same 16 bytes at any address: gfx9 global loads and stores take byte
// addresses, so this is one global_load/store_dwordx4 too.
typedef uint32_t vec4u_any __attribute__((ext_vector_type(4), aligned(1)));
typedef __attribute__((address_space(1))) vec4u_any gvec4u_any;

__device__ __forceinline__ vec4u gload_any(uint64_t a) { return *reinterpret_cast<const gvec4u_any*>(a); }
__device__ __forceinline__ void gstore_any(uint64_t a, vec4u v) { *reinterpret_cast<gvec4u_any*>(a) = v; }

__device__ __forceinline__ uint8_t gload_byte(uint64_t a) {
    return *reinterpret_cast<const __attribute__((address_space(1))) uint8_t*>(a);
}
__device__ __forceinline__ void gstore_byte(uint64_t a, uint8_t v) {
    *reinterpret_cast<__attribute__((address_space(1))) uint8_t*>(a) = v;
}

// How a range of n >= 16 bytes at any alignment is cut into 16-byte vectors:
// one per 16-byte block of the destination that the range touches, so all
// stores but the first and last are aligned.  Those two are moved inside the
// range (they overlap their neighbours and store the same bytes there), so
// nothing outside it is read or written and no byte loop is left.  m is the
// destination address & 15; an aligned range has m = 0 and offsets 16 v.
// A byte loop for ranges whose two sides differ mod 16 would move 64 bytes
// per wave instruction with one in flight.  Measured on MI355X, byte loop
// against this cut: submit_direct of 700 entries of 1..9000 bytes 794 us (4
// GB/s) against 78 us; 4096 tokens of 3000 bytes HBM -> host 479 against 237 us.
__host__ __device__ __forceinline__ uint64_t vec_count(uint64_t n, uint32_t m) { return (n + m + 15) >> 4; }
__host__ __device__ __forceinline__ int32_t vec_offset(int32_t v, int32_t m, int32_t n) {
    int32_t o = (v << 4) - m;
    o = o > 0 ? o : 0;
    return o < n - 16 ? o : n - 16;
}

// Copy n bytes s -> d with the whole wave, any alignment, as vec_offset()
// cuts them, U vectors in flight per lane.
template <int U = 4>
__device__ __forceinline__ void copy(uint64_t d, uint64_t s, uint64_t n) {
    const uint32_t lane = (uint32_t)lane_id();
    if (n < 16) {
        if (lane < n) gstore_byte(d + lane, gload_byte(s + lane));
        return;
    }
    const uint32_t m = (uint32_t)(d & 15);
    const uint64_t nv = vec_count(n, m);
    // Branch-free: a lane past the end works on the last vector instead
    // (loads it and stores the same bytes back).  A guarded load or store
    // sits in its own basic block, and the compiler then waits for every
    // earlier memory operation first, which leaves one in flight.
    // Each pass's lane offsets are vec_offset() relative to the pass's first
    // vector `at`, so a lane holds 32 bits per vector beside a wave-uniform
    // address (64-bit offsets spilled at U = 16 in the tile kernels).
    for (uint64_t base = 0; base < nv; base += (uint64_t)kWidth * U) {
        int64_t at = (int64_t)(base << 4) - (int64_t)m;
        at = at < (int64_t)n - 16 ? at : (int64_t)n - 16;
        const uint32_t lo = at < 0 ? (uint32_t)-at : 0u;
        const uint64_t left = (uint64_t)((int64_t)n - 16 - at);
        const uint32_t hi = left < (1u << 30) ? (uint32_t)left : (1u << 30);
        vec4u r[U];
        uint32_t rel[U];
#pragma unroll
        for (int k = 0; k < U; k++) {
            rel[k] = ((uint32_t)k * kWidth + lane) << 4;
            rel[k] = rel[k] > lo ? rel[k] : lo;
            rel[k] = rel[k] < hi ? rel[k] : hi;
            r[k] = gload_any(s + (uint64_t)at + rel[k]);
        }
#pragma unroll
        for (int k = 0; k < U; k++) gstore_any(d + (uint64_t)at + rel[k], r[k]);
    }
}

// 16-byte loads in flight per lane of a transfer wave, from the number of
// transfer waves in the grid: about 1 MiB of host reads outstanding in total
// (64 lanes x U x 16 B per wave) fills the PCIe link; far more only queues
// (measured on MI355X: 8 waves reach 48 GB/s at U = 16 but 20 GB/s at
// U = 4, while 256 waves drop from 55 to 47 GB/s at U = 16).
__device__ __forceinline__ int transfer_unroll(uint32_t transfer_waves) {
    return transfer_waves <= 64 ? 16 : (transfer_waves <= 128 ? 8 : 4);
}

template <int U>
__device__ __forceinline__ void copy(uint64_t d, uint64_t s, uint64_t n);

// copy() with U chosen at run time (16, 8 or 4).
__device__ __forceinline__ void copy_u(int u, uint64_t d, uint64_t s, uint64_t n) {
    if (u >= 16) copy<16>(d, s, n);
    else if (u >= 8) copy<8>(d, s, n);
    else copy<4>(d, s, n);
}

// Per-wave LDS scratch for copy_batch: start vector, addresses and bytes of up to 64 entries.
struct BatchLds {
    uint32_t start[kWidth];
    uint32_t size[kWidth];
    uint64_t src[kWidth];
    uint64_t dst[kWidth];
};

// ee[k] = the entry of lane's vector of pass k: the last one whose start is <=
// v (start past the batch's entries is the largest index), by a 6-step search
// without branches, one step of all U at a time so that the U LDS reads of a
// step are in flight together.  With the search inside each load's address,
// the loads went out one search apart.
template <int U>
__device__ __forceinline__ void find_entries(uint32_t base, uint32_t total, const BatchLds* lds, uint32_t (&ee)[U]) {
    const uint32_t lane = (uint32_t)lane_id();
#pragma unroll
    for (int k = 0; k < U; k++) ee[k] = 0;
#pragma unroll
    for (uint32_t step = kWidth / 2; step > 0; step >>= 1) {
        uint32_t st[U];
#pragma unroll
        for (int k = 0; k < U; k++) st[k] = lds->start[ee[k] + step];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const uint32_t v0 = base + (uint32_t)k * kWidth + lane;
            ee[k] += st[k] <= (v0 < total ? v0 : total - 1) ? step : 0;
        }
    }
}

// The flat vector stream of copy_batch: vector v of the batch belongs to entry
// e (v / vpe when every entry has vpe vectors, else the last entry whose
// start is <= v, see find_entries) at offset v - start[e].
// kAligned: every entry is 16-byte aligned on both sides and in size; else
// the entry's vectors lie as vec_offset() says (a uniform batch counts vpe
// vectors for the worst alignment; one too many repeats the last).
template <int U, bool kUniform, bool kAligned>
__device__ __forceinline__ void flat_copy(uint32_t total, uint32_t vpe, const BatchLds* lds) {
    const uint32_t lane = (uint32_t)lane_id();
    for (uint32_t base = 0; base < total; base += (uint32_t)kWidth * U) {
        vec4u r[U];
        uint64_t da[U];
        uint32_t ee[U];
        if (!kUniform) find_entries<U>(base, total, lds, ee);
#pragma unroll
        for (int k = 0; k < U; k++) {
            // Branch-free on a clamped index, as in copy().
            const uint32_t v0 = base + (uint32_t)k * kWidth + lane;
            const uint32_t v = v0 < total ? v0 : total - 1;
            const uint32_t e = kUniform ? v / vpe : ee[k];
            const uint32_t o = v - (kUniform ? e * vpe : lds->start[e]);
            const uint64_t d = lds->dst[e];
            if (kAligned) {
                r[k] = gload(lds->src[e] + ((uint64_t)o << 4));
                da[k] = d + ((uint64_t)o << 4);
            } else {
                const uint32_t off = (uint32_t)vec_offset((int32_t)o, (int32_t)(d & 15), (int32_t)lds->size[e]);
                r[k] = gload_any(lds->src[e] + off);
                da[k] = d + off;
            }
        }
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (kAligned) gstore(da[k], r[k]);
            else gstore_any(da[k], r[k]);
        }
    }
}

template <int U, bool kUniform>
__device__ __forceinline__ void flat_copy(bool aligned, uint32_t total, uint32_t vpe, const BatchLds* lds) {
    if (aligned) flat_copy<U, kUniform, true>(total, vpe, lds);
    else flat_copy<U, kUniform, false>(total, vpe, lds);
}

// Each lane copies its own entry of n < 16 bytes (0: nothing), all its loads
// in flight together.
__device__ __forceinline__ void copy_tiny(uint64_t d, uint64_t s, uint32_t n) {
    if (n == 0) return;
    uint8_t r[15];
#pragma unroll
    for (uint32_t k = 0; k < 15; k++) r[k] = gload_byte(s + (k < n ? k : n - 1));
#pragma unroll
    for (uint32_t k = 0; k < 15; k++) gstore_byte(d + (k < n ? k : n - 1), r[k]);
}

// flat_copy() staged through LDS: each lane's 16 bytes go host -> LDS with
// global_load_lds_dwordx4 (no VGPRs held while the loads are in flight), then
// LDS -> VGPR -> HBM.  `stage` is this wave's LDS area of U * 64 vectors.
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

template <int U, bool kUniform>
__device__ __forceinline__ void flat_copy_lds(uint32_t total, uint32_t vpe, const BatchLds* lds,
                                              vec4u* stage) {
    const uint32_t lane = (uint32_t)lane_id();
    for (uint32_t base = 0; base < total; base += (uint32_t)kWidth * U) {
        uint64_t da[U];
        uint32_t ee[U];
        if (!kUniform) find_entries<U>(base, total, lds, ee);
#pragma unroll
        for (int k = 0; k < U; k++) {
            const uint32_t v0 = base + (uint32_t)k * kWidth + lane;
            const uint32_t v = v0 < total ? v0 : total - 1;
            const uint32_t e = kUniform ? v / vpe : ee[k];
            const uint32_t o = v - (kUniform ? e * vpe : lds->start[e]);
            // lane l's 16 bytes land at stage[k * 64 + l]
            __builtin_amdgcn_global_load_lds((gptr_t)(uintptr_t)(lds->src[e] + ((uint64_t)o << 4)),
                                             (lptr_t)(stage + k * kWidth), 16, 0, 0);
            da[k] = lds->dst[e] + ((uint64_t)o << 4);
        }
        __builtin_amdgcn_s_waitcnt(0);  // every load has landed in LDS
#pragma unroll
        for (int k = 0; k < U; k++) gstore(da[k], stage[k * kWidth + lane]);
    }
}

// Copy a batch of nb <= 64 entries, lane j holding entry j's (dst, src, bytes),
// as one stream of 16-byte vectors across entry boundaries, whatever their
// alignment: u loads in flight per lane when all entries have the same size
// (u = 16, 8 or 4), 4 otherwise.  Entries of less than 16 bytes are copied by
// their lanes; a batch with one of 512 MiB or more goes entry by entry.
// Returns the bytes copied.
__device__ __forceinline__ uint64_t copy_batch(int u, uint64_t md, uint64_t ms, uint64_t mn, uint32_t nb,
                                               BatchLds* lds, vec4u* stage = nullptr) {
    const uint32_t lane = (uint32_t)lane_id();
    const bool mine = lane < nb;
    if (!mine) mn = 0;
    uint64_t total_bytes = mn;
#pragma unroll
    for (int o = kWidth / 2; o > 0; o >>= 1) {
        const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)total_bytes, o, kWidth);
        const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(total_bytes >> 32), o, kWidth);
        total_bytes += ((uint64_t)hi << 32) | lo;
    }
    total_bytes = broadcast0(total_bytes);
    if (__ballot(mn >= (1ull << 29)) != 0) {
        for (uint32_t j = 0; j < nb; j++) copy<4>(readlane64(md, (int)j), readlane64(ms, (int)j), readlane64(mn, (int)j));
        return total_bytes;
    }
    // 64 entries of less than 2^25 + 2 vectors each: the batch's vector index
    // fits 32 bits, and an offset in an entry 31.
    const uint32_t n = (uint32_t)mn;
    const bool aligned = __ballot(mine && ((md | ms | mn) & 15) != 0) == 0;
    const bool uniform = __ballot(mine && n != (uint32_t)__builtin_amdgcn_readfirstlane((int)n)) == 0;
    // A uniform batch that is not aligned counts its entries' vectors for
    // m = 15, so that v / vpe still finds the entry.
    uint32_t vecs = 0;
    if (n >= 16) vecs = (uint32_t)vec_count(n, aligned ? 0u : (uniform ? 15u : (uint32_t)(md & 15)));
    uint32_t incl = vecs;
#pragma unroll
    for (int o = 1; o < kWidth; o <<= 1) {
        const uint32_t t = (uint32_t)__shfl_up((int)incl, o, kWidth);
        if (lane >= (uint32_t)o) incl += t;
    }
    lds->start[lane] = mine ? incl - vecs : ~0u;
    if (mine) {
        lds->size[lane] = n;
        lds->src[lane] = ms;
        lds->dst[lane] = md;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWidth - 1);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t vpe0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)vecs);
    if (total > 0) {
        if (stage && aligned) {  // LDS-staged, `u` vectors per lane (the caller sized stage for it)
            if (!uniform) flat_copy_lds<4, false>(total, 0, lds, stage);
            else if (u >= 16) flat_copy_lds<16, true>(total, vpe0, lds, stage);
            else if (u >= 8) flat_copy_lds<8, true>(total, vpe0, lds, stage);
            else flat_copy_lds<4, true>(total, vpe0, lds, stage);
        } else if (uniform) {
            if (u >= 16) flat_copy<16, true>(aligned, total, vpe0, lds);
            else if (u >= 8) flat_copy<8, true>(aligned, total, vpe0, lds);
            else flat_copy<4, true>(aligned, total, vpe0, lds);
        } else {
            flat_copy<4, false>(aligned, total, 0, lds);
        }
    }
    if (__ballot(n > 0 && n < 16) != 0) copy_tiny(md, ms, n < 16 ? n : 0);
    __builtin_amdgcn_wave_barrier();  // lds reused by the next batch
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    return total_bytes;
}

// Make this wave's global stores visible device-wide before a flag is raised
// (producer side) / see other waves' stores after a flag is seen (consumer).
// The release writes the XCD's L2 back (buffer_wbl2), which is done when
// vmcnt is 0 again.  The compiler leaves that wait out where it sees no other
// memory operation pending (after an explicit s_waitcnt, say), so it is
// written here: 0x0F70 waits for vmcnt(0) alone.
__device__ __forceinline__ void release_agent() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __builtin_amdgcn_s_waitcnt(0x0F70);
}
__device__ __forceinline__ void acquire_agent() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }

__device__ __forceinline__ int lds_load(const int* p) {
    return __hip_atomic_load(const_cast<int*>(p), __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_store(int* p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_add(int* p, int v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Bounded waits: true once the condition holds, false after kSpinLimit polls.
__device__ __forceinline__ bool wait_lds_eq(const int* p, int want) {
    for (uint64_t n = 0; n < kSpinLimit; n++) {
        if (lds_load(p) == want) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}
__device__ __forceinline__ bool wait_lds_gt(const int* p, int than) {
    for (uint64_t n = 0; n < kSpinLimit; n++) {
        if (lds_load(p) > than) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}
__device__ __forceinline__ bool wait_lds_ne(const int* p, int old) {
    for (uint64_t n = 0; n < kSpinLimit; n++) {
        if (lds_load(p) != old) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}

__device__ __forceinline__ uint64_t load_system(const volatile uint64_t* p) {
    return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void store_system(volatile uint64_t* p, uint64_t v) {
    __hip_atomic_store(const_cast<uint64_t*>(p), v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ uint32_t load_system32(const volatile uint32_t* p) {
    return __hip_atomic_load(const_cast<uint32_t*>(p), __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Completion of a whole grid signalled to the host without a stream
// synchronisation.  Every thread of the grid calls it once after its last
// store: each wave waits until its stores have reached the L2, the first wave
// of the workgroup releases them at agent scope and counts the workgroup in
// `counter` (HBM, 0 before the launch); the last workgroup acquires them, puts
// the counter back to 0 for the next launch, and stores `value` to
// `host_word` (pinned host memory) with a system-scope release, so every byte
// the grid wrote is visible to any agent once the host reads `value` there.
// A null host_word disables it.
// An agent release writes the XCD's whole L2 back, so their number counts:
// one per workgroup instead of two per wave (the wave's and that of an
// acq_rel count) took submit_direct of 40 entries of up to 20 KB from 26.2 to
// 23.0 us, 1024 x 4 KiB into scattered pages from 90.7 to 89.3 (on 256 waves
// from 100.0 to 92.0).
struct GridDone {
    unsigned int* counter;
    uint64_t* host_word;
    uint64_t value;
};

__device__ __forceinline__ void signal_grid_done(const GridDone& g) {
    if (!g.host_word) return;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x >= kWidth) return;
    release_agent();
    if (threadIdx.x == 0) {
        const unsigned int prev = __hip_atomic_fetch_add(g.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (prev + 1 == gridDim.x) {
            __hip_atomic_store(g.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            acquire_agent();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
            __builtin_amdgcn_s_waitcnt(0x0F70);  // as in release_agent()
            __hip_atomic_store(g.host_word, g.value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

}  // namespace wave
}  // namespace gfd
