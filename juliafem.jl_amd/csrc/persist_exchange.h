// persist_exchange.h -- what the workgroups of a resident PCG exchange
// (persist.hip, persist_csr.hip): partial sums and scalars past the L2s, wave
// sums without LDS, and the sums over all workgroups.
#pragma once

#include "jfem_device.h"

namespace jfem {

// ---------------------------------------------------------------- exchange --
__device__ __forceinline__ void put_word(uint64_t *w, uint32_t epoch, uint32_t bits) {
    __hip_atomic_store(w, (uint64_t)epoch << 32 | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get_word(const uint64_t *w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the payloads of the N words w[i stride] once all of them are of this epoch;
// false after `polls` looks
template <int N>
__device__ __forceinline__ bool poll_words(const uint64_t *w, int stride, uint32_t epoch, int polls, uint32_t (&bits)[N]) {
    for (int k = 0; k < polls; ++k) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint64_t v = get_word(w + (size_t)i * stride);
            bits[i] = (uint32_t)v;
            ok = ok && (uint32_t)(v >> 32) == epoch;
        }
        if (ok) return true;
        __builtin_amdgcn_s_sleep(1);
    }
    return false;
}

// A shared node's three values, past the L2: raw buffer accesses with the sc1
// bit (cache policy bit 4).  Slots are 4 T apart.
constexpr int kSc1 = 16;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Partials {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ Partials(void *p, int slots)
        : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, slots * 4 * (int)sizeof(T), 0x00027000)) {}
    template <int NC> __device__ __forceinline__ void put(int slot, const T (&v)[NC]) const {
        const int o = slot * 4 * (int)sizeof(T);
        if constexpr (NC == 1) {
            u32x2 a;
            __builtin_memcpy(&a, v, 8);
            __builtin_amdgcn_raw_buffer_store_b64(a, rs, o, 0, kSc1);
        } else if constexpr (sizeof(T) == 8) {
            u32x4 a;
            u32x2 b;
            __builtin_memcpy(&a, v, 16);
            __builtin_memcpy(&b, v + 2, 8);
            __builtin_amdgcn_raw_buffer_store_b128(a, rs, o, 0, kSc1);
            __builtin_amdgcn_raw_buffer_store_b64(b, rs, o + 16, 0, kSc1);
        } else {
            u32x3 a;
            __builtin_memcpy(&a, v, 12);
            __builtin_amdgcn_raw_buffer_store_b96(a, rs, o, 0, kSc1);
        }
    }
    template <int NC> __device__ __forceinline__ void get(int slot, T (&v)[NC]) const {
        static_assert(NC == 3 || (NC == 1 && sizeof(T) == 8), "a node's values");
        const int o = slot * 4 * (int)sizeof(T);
        if constexpr (NC == 1) {
            const u32x2 a = __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, kSc1);
            __builtin_memcpy(v, &a, 8);
        } else if constexpr (sizeof(T) == 8) {
            const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, kSc1);
            const u32x2 b = __builtin_amdgcn_raw_buffer_load_b64(rs, o + 16, 0, kSc1);
            __builtin_memcpy(v, &a, 16);
            __builtin_memcpy(v + 2, &b, 8);
        } else {
            const u32x3 a = __builtin_amdgcn_raw_buffer_load_b96(rs, o, 0, kSc1);
            __builtin_memcpy(v, &a, 12);
        }
    }
};
__device__ __forceinline__ void put_shared(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_shared(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// this wave's stores have reached the point where all XCDs see them
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Sum over a wave, in every lane: DPP steps inside the rows of 16 lanes, then
// the four rows in order.  (The LDS-permute butterfly of wave_sum has a
// latency of some 100 cycles per step, and nothing hides it here.)
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0u, (uint32_t)b, CTRL, 0xf, 0xf, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0u, (uint32_t)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
template <int CTRL> __device__ __forceinline__ float dpp_mov(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), CTRL, 0xf, 0xf, false));
}
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kQuadXor3 = 0x1b;  // lane ^ 1, 2, 3 of a quad
constexpr int kRowMirror = 0x140, kRowHalfMirror = 0x141;
__device__ __forceinline__ double row_sum(double v) {  // sum of the lane's row of 16
    v += dpp_mov<kQuadXor1>(v);
    v += dpp_mov<kQuadXor2>(v);
    v += dpp_mov<kRowHalfMirror>(v);
    v += dpp_mov<kRowMirror>(v);
    return v;
}
__device__ __forceinline__ double lane_of(double v, int lane) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane), hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ double wave_total(double v) {
    v = row_sum(v);
    return (lane_of(v, 0) + lane_of(v, 16)) + (lane_of(v, 32) + lane_of(v, 48));
}

// All-reduce of NV doubles over the workgroups: v in: the thread's share, out:
// the grid's sums, the same bits in every thread of every workgroup; false
// when a wait gave up after `polls` looks (others may then get sums without this
// workgroup's share: the host discards the solve).  Up to 16 workgroups read each other's entries; more form
// groups of 16 (workgroup >> 4) whose first workgroup sums the group's values
// and publishes the sum once per 8 workgroups, and every workgroup reads its
// copy of the groups' sums: uncached requests to one line are served one after
// the other, so no line may have more than a few readers.  (240 workgroups
// reading one set of words, or all of them, took 4-6 us per exchange.)  A value
// is an entry of two words, and the NV entries of a workgroup lie side by side,
// one request to store and, with the neighbours', one to read (as rows of single
// words, which is four requests for two values, an iteration of 240 workgroups
// took 0.9 us longer; one hop with 16 copies of all entries, 0.4 us longer than
// that).  One wave polls: lane 16 k + m reads value k of member m, so a sum over
// members is a row sum.
// FLAT: 17 to 64 workgroups store their entries once per 8 workgroups, and each
// reads its copy of all of them, one hop.  On the CSR matrix an iteration with it and
// without takes, Hex8, 5.6 and 6.4 us with 17 workgroups, 5.7 and 6.4 with 31, 5.7 and
// 6.1 with 41, 5.9 and 6.6 with 61; Tet10 6.2 and 6.1 with 17, 6.1 and 6.8 with 23,
// 6.1 and 6.7 with 42, 6.3 and 6.4 with 64; nothing is gained with 102, and the
// element kernels, which have no registers for it, lose 2-5%.
// Calls that follow each other without a block barrier use different `sh` (a
// wave may still read it when the next one starts).
constexpr int kGroup = 16, kCopy = 8, kFlat = 64;
template <int NV> struct GridSumLds { double a[NV][16], b[NV], f[NV][2]; };
static_assert(kPersistPatches <= kGroup * kGroup && kPersistPatches / kCopy <= 32, "two levels, copies x values in a wave");

// words of n workgroups: their entries, then the copies of the groups' sums
__host__ __device__ constexpr int grid_words(int nv, int n, bool flat = false) {
    const int copies = (n + kCopy - 1) / kCopy;
    return 2 * nv * (flat && n > kGroup && n <= kFlat ? copies * n : n + (n > kGroup ? copies * kGroup : 0));
}

struct Entries {  // past the L2, as the partials
    __amdgpu_buffer_rsrc_t rs;
    int polls;
    __device__ __forceinline__ Entries(uint64_t *p, int words, int polls_)
        : rs(__builtin_amdgcn_make_buffer_rsrc(p, 0, 8 * words, 0x00027000)), polls(polls_) {}
    __device__ __forceinline__ void put(int i, uint32_t epoch, double v) const {
        const uint64_t b = (uint64_t)__double_as_longlong(v);
        const u32x4 a = {(uint32_t)b, epoch, (uint32_t)(b >> 32), epoch};
        __builtin_amdgcn_raw_buffer_store_b128(a, rs, 16 * i, 0, kSc1);
    }
    // polls until both words of entry i are of this epoch
    __device__ __forceinline__ double get(int i, uint32_t epoch, int *bad) const {
        for (int k = 0; k < polls; ++k) {
            const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * i, 0, kSc1);
            if (a.y == epoch && a.w == epoch) return __longlong_as_double((long long)((uint64_t)a.z << 32 | a.x));
            __builtin_amdgcn_s_sleep(1);
            asm volatile("" ::: "memory");  // the load is not to leave the loop
        }
        *bad = 1;
        return 0.0;
    }
};

// the sum over n <= 16 members' entries from `first` on, in every lane of row k (value k)
template <int NV>
__device__ __forceinline__ double sum_members(const Entries &en, int first, int n, uint32_t epoch, int *bad) {
    const int lane = (int)threadIdx.x & 63, k = lane >> 4, m = lane & 15;
    return row_sum(k < NV && m < n ? en.get((first + m) * NV + k, epoch, bad) : 0.0);
}

template <int NV, int NT, bool FLAT = false>
__device__ __forceinline__ bool grid_sum(double (&v)[NV], uint64_t *words, int wg, int nwg, uint32_t epoch, int polls,
                                         GridSumLds<NV> &sh, int *bad) {
    static_assert(NV <= 2 && NT / 64 <= 16, "one row of 16 lanes per value");
    constexpr int kW = NT / 64;
    const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double w = wave_total(v[k]);
        if (lane == 0) sh.a[k][wv] = w;
    }
    __syncthreads();
    if (FLAT && nwg > kGroup && nwg <= kFlat) {
        const Entries en(words, grid_words(NV, nwg, true), polls);
        if (wv == 0) {
            const int k = lane >> 4, m = lane & 15;
            const double s = row_sum(k < NV && m < kW ? sh.a[k < NV ? k : 0][m] : 0.0);
            double mine = lane_of(s, 0);
            if constexpr (NV == 2) mine = lane & 1 ? lane_of(s, 16) : mine;
            const int c = lane / NV;
            if (c < (nwg + kCopy - 1) / kCopy) en.put((c * nwg + wg) * NV + lane % NV, epoch, mine);
        }
        if (wv < NV) {
            const int i = (int)threadIdx.x;  // member i / NV, value i % NV
            const double e = i < nwg * NV ? en.get(wg / kCopy * nwg * NV + i, epoch, bad) : 0.0;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const double w = wave_total(i % NV == k ? e : 0.0);
                if (lane == 0) sh.f[k][wv] = w;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] = NV == 2 ? sh.f[k][0] + sh.f[k][NV - 1] : sh.f[k][0];
        return *bad == 0;
    }
    if (wv == 0) {
        const int k = lane >> 4, m = lane & 15;
        double s = row_sum(k < NV && m < kW ? sh.a[k < NV ? k : 0][m] : 0.0);  // row k: the block's value k
        if (nwg > 1) {
            const Entries en(words, grid_words(NV, nwg), polls);
            if (k < NV && m == 0) en.put(wg * NV + k, epoch, s);
            if (nwg > kGroup) {
                const int g = wg / kGroup, copies = (nwg + kCopy - 1) / kCopy;
                if (wg % kGroup == 0) {
                    s = sum_members<NV>(en, wg, min(kGroup, nwg - wg), epoch, bad);
                    double mine = lane_of(s, 0);
                    if constexpr (NV == 2) mine = lane & 1 ? lane_of(s, 16) : mine;
                    const int c = lane / NV;  // copy, value lane % NV
                    if (c < copies) en.put((nwg + c * kGroup + g) * NV + lane % NV, epoch, mine);
                }
                s = sum_members<NV>(en, nwg + wg / kCopy * kGroup, (nwg + kGroup - 1) / kGroup, epoch, bad);
            } else {
                s = sum_members<NV>(en, 0, nwg, epoch, bad);
            }
        }
        if (k < NV && m == 0) sh.b[k] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = sh.b[k];
    return *bad == 0;
}

}  // namespace jfem
