// gpu_util.hpp -- small device helpers shared by the march kernels (GLM and CT).
#pragma once
#include "physics.hpp"

namespace glm {

constexpr int NXCD = 8;   // XCDs of an MI355X

// i mod n in [0, n) for any int i (periodic wrap of a cell or forcing index).
GLM_DEV int wrapi(int i, int n)
{
    int m = i % n;
    return m < 0 ? m + n : m;
}

// Logical tile of hardware workgroup id w when ids are dealt round-robin over NXCD XCDs: XCD x
// gets the contiguous logical range [start_x, start_x + count_x).  A bijection on [0, total).
GLM_DEV int xcd_block(int w, int total)
{
    const int q = total / NXCD, r = total % NXCD;
    const int xcd = w % NXCD, slot = w / NXCD;
    return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
}

// Indices (i, j, k) of the cells c, c + step, c + 2 step, ... of an nx x ny x . grid, carried along: the
// divisions are done once per lane, where one per cell and axis cost a reduction as much as its loads.
struct CellWalk {
    int i, j, k, di, dj, dk, nx, ny;
    GLM_DEV CellWalk(size_t c, size_t step, int nx_, int ny_) : nx(nx_), ny(ny_)
    {
        const size_t r = c / nx, rs = step / nx;
        i = (int)(c - r * nx); j = (int)(r % ny); k = (int)(r / ny);
        di = (int)(step - rs * nx); dj = (int)(rs % ny); dk = (int)(rs / ny);
    }
    GLM_DEV void next()
    {
        i += di; j += dj; k += dk;
        if (i >= nx) { i -= nx; ++j; }
        if (j >= ny) { j -= ny; ++k; }
    }
};

// Largest of the workgroup's values (the bits of non-negative doubles, NaN largest) into *out: wavefront
// shuffles, one LDS slot per wavefront, one atomic per workgroup.  Atomics on one address of the
// device run one after another, about 12 ns each across the XCDs: with one per wavefront they were
// the whole time of a CFL reduction (64^3 FP64: 4096 of them, 50 us; 180 x 130 x 99 FP32: 8192, 103 us;
// now 4.5 and 17 us).
template <int NTH>
GLM_DEV void block_max_bits(unsigned long long bits, unsigned long long* out)
{
    static_assert(NTH % 64 == 0, "whole wavefronts");
    __shared__ unsigned long long red[NTH / 64];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const unsigned long long o = __shfl_xor(bits, off, 64);
        bits = o > bits ? o : bits;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = bits;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < NTH / 64; ++w) bits = red[w] > bits ? red[w] : bits;
        // the slot only grows, so a workgroup whose value it has reached needs no atomic (64^3: 10.2 -> 4.5 us)
        if (bits > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, bits);
    }
}

// HBM access through the global address space.  Pointers read back from LDS (the cold arguments)
// have lost their address space, and generic loads are counted together with LDS operations, so
// every LDS wait in the march would also wait for the prefetch of the next planes.
template <typename T>
GLM_DEV T gload(const T* p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(1))) T*)p;
#else
    return *p;   // host pass of the kernel templates: never executed
#endif
}
// The same at a byte offset from a base that is one for the wavefront: where the offset is a 32-bit
// value of its own the instruction adds the two.
template <typename T>
GLM_DEV T gload_at(const T* base, unsigned off)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const __attribute__((address_space(1))) char* b = (const __attribute__((address_space(1))) char*)base;
    return *(const __attribute__((address_space(1))) T*)(b + off);
#else
    return *(const T*)((const char*)base + off);
#endif
}
template <typename T>
GLM_DEV void gstore_at(T* base, unsigned off, T x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __attribute__((address_space(1))) char* b = (__attribute__((address_space(1))) char*)base;
    *(__attribute__((address_space(1))) T*)(b + off) = x;
#else
    *(T*)((char*)base + off) = x;
#endif
}

template <typename T>
GLM_DEV void gstore_nt(T v, T* p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_nontemporal_store(v, (__attribute__((address_space(1))) T*)p);
#else
    *p = v;
#endif
}

template <typename T>
GLM_DEV void gstore_nt_at(T v, T* base, unsigned off)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __attribute__((address_space(1))) char* b = (__attribute__((address_space(1))) char*)base;
    __builtin_nontemporal_store(v, (__attribute__((address_space(1))) T*)(b + off));
#else
    *(T*)((char*)base + off) = v;
#endif
}
// Uses behind this point take the value as a new one: what is derived from it is not carried from
// before (an offset widened ahead of a loop, a pointer table read ahead of it).
template <typename P>
GLM_DEV void renew_s(P& p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
}
template <typename V>
GLM_DEV void renew_v(V& x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
}

// An argument block as a reference into the constant address space: a kernel reads each field with
// a scalar load where it needs it, instead of holding a copy of the whole block in registers (which
// cost the ensemble kernel 64 B per lane of spills).
template <typename S>
GLM_DEV const auto& constant_ref(const S* p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(4))) S*)p;
#else
    return *p;   // host pass of the kernel templates: never executed
#endif
}
// A kernel's own argument block read in place from the kernarg segment, where the explicit
// arguments start: for a kernel whose one argument is an S (at offset 0), each field is then a
// scalar load where it is read, as the ensemble reads its boxes' blocks, instead of coming through
// the by-value parameter (the FP64 PPM + HLLD march at 256^3: 44 -> 36 B of spills per lane, 2%
// faster).
template <typename S>
GLM_DEV const auto& kernarg_ref()
{
    return constant_ref((const S*)__builtin_amdgcn_kernarg_segment_ptr());
}

}  // namespace glm
