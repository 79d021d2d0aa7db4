// ksh_devutil.hpp -- small gfx950 device helpers shared by the band kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace ksh {

typedef unsigned int ksh_u32x2 __attribute__((ext_vector_type(2)));

// a wave-uniform pointer in scalar registers
template <typename T>
__device__ __forceinline__ T *uniform_ptr(T *p)
{
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(a >> 32));
    return (T *)(((unsigned long long)hi << 32) | lo);
}

// the same pointer, stated to be one to global memory (a pointer read from memory is a generic one
// to the compiler, and a flat access waits for every memory and LDS access in flight); by way of an
// integer, since a pair of pointer casts is folded away
template <typename T>
__device__ __forceinline__ T *global_ptr(T *p)
{
    return (T *)(__attribute__((address_space(1))) T *)(unsigned long long)p;
}

// broadcast of lane `src`'s value (v_readlane: the result is wave-uniform)
__device__ __forceinline__ double readlane_f64(double v, int src)
{
    int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
    int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float readlane_f32(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
__device__ __forceinline__ double bcast(double v, int src) { return readlane_f64(v, src); }
__device__ __forceinline__ float bcast(float v, int src) { return readlane_f32(v, src); }

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kQuadSwap = 0xB1, kQuadCross = 0x4E;

// (a, b) -> a of the lower 32 lanes beside b's lower, plus the same of the upper: lanes < 32 get
// a[l] + a[l + 32], lanes >= 32 get b[l - 32] + b[l]; likewise for the 16-lane rows
__device__ __forceinline__ double swap_add32(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// sums over the 64 lanes of sixteen values: lane l gets the total of value l / 4
__device__ __forceinline__ double sum_lanes(const double (&a)[16], int lane)
{
    double v[8], w[4], y[2];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = swap_add32(a[q], a[q + 8]);
#pragma unroll
    for (int q = 0; q < 4; ++q) w[q] = swap_add16(v[q], v[q + 4]);
    const bool up8 = (lane & 8) != 0, up4 = (lane & 4) != 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) y[q] = (up8 ? w[q + 2] : w[q]) + dpp_move<kRor8>(up8 ? w[q] : w[q + 2]);
    double s = (up4 ? y[1] : y[0]) + dpp_move<kHalfMirror>(up4 ? y[0] : y[1]);
    s += dpp_move<kQuadSwap>(s);
    s += dpp_move<kQuadCross>(s);
    return s;
}

// workgroup barrier that orders LDS only: global loads in flight (register prefetches private to
// their thread) are not waited for
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// value the compiler cannot see through: keeps per-lane comparisons inside a loop instead of
// hoisted (as one lane mask per comparison) out of it
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// the same for a wave-uniform value (kept in an SGPR): values derived from it are recomputed where
// they are used instead of hoisted out of a loop, each into a scalar register of its own
__device__ __forceinline__ int opaque_s(int v)
{
    asm volatile("" : "+s"(v));
    return v;
}

// Band reads and writes go through a buffer resource covering exactly the band (bytes < 2 GiB,
// checked by the launchers).  A masked-off access is sent to offset 0x80000000, beyond the
// resource: the buffer unit returns 0 for such a read and drops such a write.  Masked accesses
// thus stay straight-line code with many loads in flight, and no mask stays live across a load.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t band_rsrc(const void *base, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

constexpr unsigned kMaskedOff = 0x80000000u;

template <typename T>
__device__ __forceinline__ T load_if(bool ok, __amdgpu_buffer_rsrc_t rs, unsigned byte_off)
{
    const int off = (int)(ok ? byte_off : kMaskedOff);
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
    else
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
}

template <typename T>
__device__ __forceinline__ void store_if(bool ok, __amdgpu_buffer_rsrc_t rs, unsigned byte_off, T v)
{
    const int off = (int)(ok ? byte_off : kMaskedOff);
    if constexpr (sizeof(T) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(ksh_u32x2, v), rs, off, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, off, 0, 0);
}

// buffer access at a per-lane offset (kMaskedOff for a masked-off lane) plus a wave-uniform
// offset carried in an SGPR
template <typename T>
__device__ __forceinline__ T load_vs(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff)
{
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)voff, (int)soff, 0));
    else
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)voff, (int)soff, 0));
}

template <typename T>
__device__ __forceinline__ void store_vs(__amdgpu_buffer_rsrc_t rs, unsigned voff, unsigned soff, T v)
{
    if constexpr (sizeof(T) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(ksh_u32x2, v), rs, (int)voff, (int)soff, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, (int)voff, (int)soff, 0);
}

}  // namespace ksh
