// Shared device/host helpers for the gfx950 attention kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

namespace fa {

// Launches `kernel` on `stream` through hipLaunchKernel and returns the
// runtime's status for this launch alone (no hipGetLastError, so an earlier,
// unrelated error is neither reported here nor cleared; a failed launch
// stays in HIP's own last-error state as well, where a caller's
// hipGetLastError finds it). Arguments are converted to the kernel's
// parameter types first.
template <typename... Params, typename... Args>
hipError_t launch_kernel(void (*kernel)(Params...), dim3 grid, dim3 block, hipStream_t stream, Args&&... args)
{
    static_assert(sizeof...(Params) == sizeof...(Args) && sizeof...(Params) > 0, "kernel argument count");
    std::tuple<std::decay_t<Params>...> values{static_cast<std::decay_t<Params>>(std::forward<Args>(args))...};
    return std::apply(
        [&](auto&... v) {
            void* ptrs[] = {static_cast<void*>(&v)...};
            return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, 0, stream);
        },
        values);
}

// Records a non-success status of a C-ABI call in the calling thread's
// last-error slot (read by fa_get_last_error / fa_peek_at_last_error) and
// returns it unchanged. FA_ERROR_UNSUPPORTED (an unsupported head_dim, which
// the reference's launchers skip silently) is not recorded. Defined in
// fa_api.cpp.
int record_status(int status);

// bf16 is carried as raw 16-bit patterns in memory (uint16_t); conversions
// below are exact (bf16 -> f32) or IEEE round-to-nearest-even (f32 -> bf16,
// lowered to v_cvt_pk_bf16_f32 on gfx950).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_bits_to_float(uint32_t bits16)
{
    return __uint_as_float(bits16 << 16);
}

__device__ __forceinline__ float bf16_lo(uint32_t word) { return __uint_as_float(word << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t word) { return __uint_as_float(word & 0xffff0000u); }

// Two floats -> packed bf16x2 word (low half = a), RNE.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b)
{
    bf16x2 v;
    v[0] = static_cast<__bf16>(a);
    v[1] = static_cast<__bf16>(b);
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ uint16_t float_to_bf16_bits(float a)
{
    return __builtin_bit_cast(uint16_t, static_cast<__bf16>(a));
}

// wave64 reductions (butterfly over all 64 lanes)
__device__ __forceinline__ float wave_max(float x)
{
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) x = fmaxf(x, __shfl_xor(x, offset, 64));
    return x;
}

__device__ __forceinline__ float wave_sum(float x)
{
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) x += __shfl_xor(x, offset, 64);
    return x;
}

// s_waitcnt with vmcnt <= N and lgkmcnt == 0 (expcnt untouched).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
}

typedef int i32x4 __attribute__((ext_vector_type(4)));

// Buffer resource for raw (stride 0) byte-addressed loads: 48-bit base,
// num_records in bytes, and the gfx9 raw-buffer configuration word. Loads at
// offsets >= num_records return zero instead of touching memory.
constexpr uint32_t kRawBufferConfig = 0x00020000u;

// A byte address kept as two uniform 32-bit halves (scalar registers), so
// per-tile descriptor arithmetic stays on the scalar unit.
struct ScalarPtr
{
    uint32_t lo;
    uint32_t hi;
};

__device__ __forceinline__ ScalarPtr scalar_ptr(const void* p)
{
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    return ScalarPtr{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(b)))),
                     static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(b >> 32))))};
}

// Descriptor of `bytes` bytes starting `offset` bytes after `base`.
__device__ __forceinline__ i32x4 make_rsrc(ScalarPtr base, uint32_t offset, uint32_t bytes)
{
    const uint64_t b = ((static_cast<uint64_t>(base.hi) << 32) | base.lo) + offset;
    i32x4 r;
    r[0] = static_cast<int>(static_cast<uint32_t>(b));
    r[1] = static_cast<int>(static_cast<uint32_t>(b >> 32) & 0xffffu);
    r[2] = static_cast<int>(bytes);
    r[3] = static_cast<int>(kRawBufferConfig);
    return r;
}

// One 16-byte-per-lane HBM -> LDS copy: lane l's 16 bytes at byte offset
// voff of the buffer land at LDS byte address lds + 16*l
// (buffer_load_dwordx4 ... lds); offsets past the buffer's end read as zero.
// Issued through inline asm so the compiler's LDS-DMA alias tracking, which
// cannot tell the pipeline stages apart, adds no waits of its own: every
// consumer of the data waits on vmcnt explicitly before a barrier. M0 needs
// one wait state between its write and the load.
__device__ __forceinline__ void dma16(i32x4 rsrc, uint32_t voff, uint32_t lds)
{
    // rsrc must reach the asm in SGPRs: where the compiler cannot prove a
    // descriptor uniform it keeps it in VGPRs and passes that tuple to the
    // "s" operand, and the assembler rejects the copy ("invalid operand"), a
    // build error. Every descriptor here is built from uniform values; a
    // readfirstlane of each word would guard against it at two scalar moves
    // per step in the two-group loop.
    lds = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(lds)));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc), "s"(lds)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)(p)));
}

constexpr float kLog2e = 1.4426950408889634f;

// Compute units of the current device (cached per device; 256 on an
// MI355X). A failed query only affects how work is laid out.
inline int device_compute_units()
{
    constexpr int kMaxDevices = 64;
    static std::atomic<int> cache[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    int cus = cache[dev].load(std::memory_order_relaxed);
    if (cus <= 0)
    {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        cache[dev].store(cus, std::memory_order_relaxed);
    }
    return cus;
}

}  // namespace fa
