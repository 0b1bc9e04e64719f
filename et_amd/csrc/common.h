// Shared device/host helpers for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <atomic>
#include <stdint.h>
#include <stdio.h>

#include "../../include/et_amd.h"
#include "tile_order.h"

namespace et {

// ---- error plumbing -------------------------------------------------------
void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);

#define ET_HIP(call)                                                           \
    do {                                                                       \
        hipError_t e__ = (call);                                               \
        if (e__ != hipSuccess)                                                 \
            return ::et::hip_fail(e__, #call);                                 \
    } while (0)

#define ET_REQUIRE(cond, code, ...)                                            \
    do {                                                                       \
        if (!(cond)) {                                                         \
            ::et::set_error(__VA_ARGS__);                                      \
            return (code);                                                     \
        }                                                                      \
    } while (0)

static inline bool aligned16(const void *p) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// What kept launch_kernel from launching, for the launch_status behind it.
inline thread_local hipError_t g_not_launched = hipSuccess;

static inline int launch_status(const char *what) {
    const hipError_t kept = g_not_launched, last = hipGetLastError();
    g_not_launched = hipSuccess;
    if (kept != hipSuccess || last != hipSuccess)
        return hip_fail(kept != hipSuccess ? kept : last, what);
    return ET_OK;
}

// ---- vector types -----------------------------------------------------------
typedef _Float16 f16;
typedef f16 f16x2 __attribute__((ext_vector_type(2)));
typedef f16 f16x4 __attribute__((ext_vector_type(4)));
typedef f16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;

// D(16x16,f32) += A(16x32,f16) * B(32x16,f16).
// Register layout (wave64), g = lane/16, c = lane%16:
//   a[j] = A[c][8g+j], b[j] = B[8g+j][c], d[r] = D[4g+r][c].
// Only the pairing of a[j] with b[j] inside the same lane group matters for
// the contraction, so any consistent assignment of k to (g,j) works.
__device__ __forceinline__ f32x4 mfma16x16x32(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 16 bytes per lane straight from global memory into LDS
// (global_load_lds_dwordx4): lane L of the wave writes at lds_base + 16*L;
// lds_base must be wave-uniform, the source address is free per lane.
// Completion is tracked by vmcnt.
__device__ __forceinline__ void load_lds16(const void *gsrc, void *lds_base) {
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void *)gsrc,
        (__attribute__((address_space(3))) void *)lds_base, 16, 0, 0);
}

// The same from a wave-uniform base and a byte offset per lane, for loops that keep requests in flight while they use
// other parts of the LDS and wait for them by themselves (s_waitcnt vmcnt).  The compiler tracks requests of the builtin
// above and waits for ALL of them in front of LDS stores and barriers; this form it does not see.
__device__ __forceinline__ void load_lds16_untracked(const void *base, unsigned lane_offset, void *lds_base) {
    const unsigned dst = (unsigned)(size_t)(__attribute__((address_space(3))) char *)lds_base;
    const unsigned long long at = (unsigned long long)base;
    const unsigned long long src = (unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(at >> 32)) << 32 |
                                   (unsigned)__builtin_amdgcn_readfirstlane((unsigned)at);
    unsigned keep; // (M0 is the compiler's)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "s"(__builtin_amdgcn_readfirstlane(dst)), "v"(lane_offset), "s"(src)
                 : "memory");
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }

// Stores whose data other workgroups of the SAME launch read: an agent-scope
// store goes through the XCD's own L2 to the device's coherence point, and is
// there once vmcnt has counted it.
__device__ __forceinline__ void store_agent4(f16 *p, f16x4 v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_agent8(f16 *p, f16x8 v) {
    store_agent4(p, f16x4{v[0], v[1], v[2], v[3]});
    store_agent4(p + 4, f16x4{v[4], v[5], v[6], v[7]});
}

// ---- wave64 reductions (all lanes receive the result) -----------------------
// Data-parallel-primitive moves inside a row of 16 lanes (no LDS round trip as
// with __shfl): quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror, row_mirror.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_move<0xB1>(v);  // pairs
    v += dpp_move<0x4E>(v);  // quads
    v += dpp_move<0x141>(v); // 8 lanes
    v += dpp_move<0x140>(v); // the row of 16: every lane holds its row's sum
    // the four rows through scalar registers
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
    const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
    return (r0 + r1) + (r2 + r3);
}

// A row in 32 lanes: `lo` is what lanes 0..31 of a whole wave would hold, `hi` what lanes 32..63 would; the sum of each half
// of the wave to its lanes, in the order of wave_sum.
__device__ __forceinline__ float half_wave_sum(float lo, float hi) {
    float v[2] = {lo, hi};
#pragma unroll
    for (int i = 0; i < 2; i++) {
        v[i] += dpp_move<0xB1>(v[i]);
        v[i] += dpp_move<0x4E>(v[i]);
        v[i] += dpp_move<0x141>(v[i]);
        v[i] += dpp_move<0x140>(v[i]);
    }
    // rows of 16 lanes: (lo 0, lo 1) and (hi 0, hi 1) -> (lo 0, hi 0) and (lo 1, hi 1)
    // (the additions are written out: the compiler takes the two results of a swap that meet in one for equal)
    auto swap_add = [](unsigned x, unsigned y) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        unsigned t = r[0];
        asm("v_add_f32 %0, %0, %1" : "+v"(t) : "v"(r[1]));
        return t;
    };
    const unsigned s = swap_add(__builtin_bit_cast(unsigned, v[0]), __builtin_bit_cast(unsigned, v[1]));
    unsigned t = s;
    asm("" : "+v"(t));
    return __builtin_bit_cast(float, swap_add(s, t));
}

// GELU of four halves: x^3 in (packed) half, the sigmoid form of
// 0.5(1+tanh u) = 1/(1+exp(-2u)) in fp32, rounded to half, times x in half
// (kernels/linear.cu:36-48).
__device__ __forceinline__ f16x4 gelu4(f16x4 v) {
    const f16x4 x2 = v * v;
    const f16x4 x3 = v * x2;
    f32x4 t;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float s = __builtin_fmaf(0.044715f, (float)x3[r], (float)v[r]);
        const float e = __builtin_amdgcn_exp2f(s * (-1.5957691216057308f * 1.4426950408889634f));
        t[r] = __builtin_amdgcn_rcpf(1.0f + e);
    }
    return v * __builtin_convertvector(t, f16x4);
}

__device__ __forceinline__ float f16_bits_to_float(uint16_t b) {
    return (float)__builtin_bit_cast(f16, b);
}

// The device that a stream's work runs on, whichever is current; the null stream and the per-thread one are the current
// device's.
inline hipError_t stream_device(hipStream_t st, int *dev) {
    return !st || st == hipStreamLegacy || st == hipStreamPerThread ? hipGetDevice(dev) : hipStreamGetDevice(st, dev);
}
// `dev` is the current device while this lives
class OnDevice {
    int before = -1;

  public:
    hipError_t error;
    explicit OnDevice(int dev) : error(hipGetDevice(&before)) {
        if (error == hipSuccess && before != dev)
            error = hipSetDevice(dev);
        else
            before = -1;
    }
    ~OnDevice() {
        if (before >= 0)
            (void)hipSetDevice(before);
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;
};

// What a launcher worked out for sizes it has seen: a choice among a kernel's forms weighs up to a hundred of them, 1 us of
// the host's time at every launch, and a program calls with few sizes.  By value of the sizes alone, a table of its own
// for every thread and choice, 64 entries that displace each other.
template <class Value, int N> struct KeptChoices {
    struct Key {
        int v[N];
        bool operator==(const Key &o) const {
            for (int i = 0; i < N; i++)
                if (v[i] != o.v[i])
                    return false;
            return true;
        }
    };
    struct Entry {
        Key key;
        Value value;
        bool used;
    };
    Entry entries[64];
    Entry &at(const Key &k) {
        unsigned h = 0;
        for (int i = 0; i < N; i++)
            h = (h ^ (unsigned)k.v[i]) * 0x9E3779B1u;
        return entries[h >> 26];
    }
    template <class Work> Value get(const Key &k, Work &&work) {
        Entry &e = at(k);
        if (!e.used || !(e.key == k)) {
            e.value = work();
            e.key = k;
            e.used = true;
        }
        return e.value;
    }
};

// A launch through the kernel's function handle on the stream's device, which is looked up once per kernel instance and
// device instead of by its host address at every launch: 0.16 us less of host time a launch (13 parameters: 2.47 -> 2.31
// us, 3.59 -> 3.48 while the host is slow), where a call's smallest sizes are bound by the host.  Dynamic LDS above the
// 64 KB default has to be allowed per kernel and device, by a call to the driver: made when a launch needs more than any
// before it.  What goes wrong is left for launch_status, as with <<<>>>.
constexpr size_t DEFAULT_LDS = 64 * 1024;
struct KernelOnDevice {
    std::atomic<hipFunction_t> fn{nullptr};
    std::atomic<size_t> lds{DEFAULT_LDS}; // dynamic LDS that launches may ask for
};
// runtime.hip: makes both of the record good for such a launch
hipError_t kernel_on_device(KernelOnDevice &k, const void *kernel, int dev, size_t lds);

template <class... P, class... A>
inline hipError_t launch_function(hipFunction_t fn, void (*)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, const A &...args) {
    static_assert(sizeof...(P) == sizeof...(A), "as many arguments as the kernel has parameters");
    return [&](P... values) { // (converted to the parameters' types)
        void *params[] = {const_cast<void *>(static_cast<const void *>(&values))...};
        return hipModuleLaunchKernel(fn, grid.x, grid.y, grid.z, block.x, block.y, block.z, (unsigned)lds, st, params, nullptr);
    }(args...);
}
template <auto KERN, class... A>
inline void launch_kernel(dim3 grid, dim3 block, size_t lds, hipStream_t st, const A &...args) {
    static KernelOnDevice known[16];
    KernelOnDevice beyond; // (devices of a higher number: looked up each time)
    int dev = 0;
    hipError_t e = stream_device(st, &dev);
    if (e == hipSuccess) {
        KernelOnDevice &k = dev >= 0 && dev < 16 ? known[dev] : beyond;
        hipFunction_t fn = k.fn.load(std::memory_order_acquire);
        if (!fn || lds > k.lds.load(std::memory_order_acquire)) {
            e = kernel_on_device(k, reinterpret_cast<const void *>(KERN), dev, lds);
            fn = k.fn.load(std::memory_order_acquire);
        }
        if (e == hipSuccess)
            e = launch_function(fn, KERN, grid, block, lds, st, args...);
    }
    if (e != hipSuccess)
        g_not_launched = e;
}

} // namespace et
