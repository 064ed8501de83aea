// column_hw.h -- the hardware operations of column_sweep.h on gfx950.
#pragma once

#include <hip/hip_runtime.h>

#define FF_CS_DEVICE __device__ __forceinline__
#define FF_CS_SHARED __shared__
#define FF_CS_BARRIER() __syncthreads()
#define FF_CS_LOAD32(p) __hip_atomic_load((p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define FF_CS_RAISE(p) __hip_atomic_fetch_or((p), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define FF_CS_TICKET(p) atomicAdd((p), 1u)
#define FF_CS_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
#define FF_CS_RARE(x) __builtin_expect(!!(x), 0)
#define FF_CS_ANY(x) (__ballot(x) != 0)
#define FF_CS_F2U(v) __float_as_uint(v)
#define FF_CS_U2F(u) __uint_as_float(u)
#define FF_CS_D2U(v) ((unsigned long long)__double_as_longlong(v))
#define FF_CS_U2D(u) __longlong_as_double((long long)(u))
// LDS accesses that other waves see: one instruction each, volatile, so the
// compiler keeps their program order
#define FF_CS_LDS_LOAD(p) ff::ldsLoad(p)
#define FF_CS_LDS_STORE(p, v) ff::ldsStore((p), (v))
#define FF_CS_WAVE_ORDER()  // nothing: the hardware performs a wave's LDS accesses in order
// what is loaded after it is loaded anew: buffer loads are not volatile (the
// pipelined ones are to move freely), and a poll without it could be one load
#define FF_CS_REREAD() asm volatile("" ::: "memory")
// buffers: accesses outside [0, bytes) load zeros and store nothing
#define FF_CS_BUFFER ff::ColumnBuffer
#define FF_CS_MAKE_BUFFER(p, bytes) (ff::ColumnBuffer{(void *)(p), (bytes)})
// (whole 16-byte accesses, an 8- or 4-byte one for the rest; words coherently,
// each 8-byte word in one access)
#define FF_CS_LOAD(v, b, off) ff::bufferLoad<0>((v), (b), (off))
#define FF_CS_STORE(v, b, off) ff::bufferStore<0>((v), (b), (off))
#define FF_CS_LOAD_WORDS(w, b, off) ff::bufferLoad<ff::BUFFER_COHERENT>((w), (b), (off))
#define FF_CS_STORE_WORDS(w, b, off) ff::bufferStore<ff::BUFFER_COHERENT>((w), (b), (off))
// lane j-1's (fwd) or j+1's value in each row of 16 lanes, ext at its end;
// and the value of the row of 16 lanes before (fwd) or after, ext at the end
#define FF_CS_ROW_SHIFT(fwd, v, ext) ff::rowShift<fwd>((v), (ext))
#define FF_CS_LINE_SHIFT(fwd, v, ext) ff::lineShift<fwd>((v), (ext))

namespace ff {

struct ColumnBuffer {
    void *p;
    unsigned bytes;
};

typedef unsigned ColumnU2 __attribute__((ext_vector_type(2)));
typedef unsigned ColumnU4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t bufferRsrc(const ColumnBuffer &b) {
    return __builtin_amdgcn_make_buffer_rsrc(b.p, 0, (int)b.bytes, 0x00027000);
}
// keeps the offset one register: a bounds check of a base and an immediate
// would take a negative base out of range.  (It does not make a repeated load
// of one place a new one: FF_CS_REREAD does.)
__device__ __forceinline__ int bufferOffset(unsigned off) {
    asm("" : "+v"(off));
    return (int)off;
}
constexpr int BUFFER_COHERENT = 16;  // sc1: past this die's L2

__device__ __forceinline__ double joinDouble(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)((unsigned long long)lo | ((unsigned long long)hi << 32)));
}
template <int CP, class V>
__device__ __forceinline__ void bufferLoad(V &v, const ColumnBuffer &b, unsigned off) {
    constexpr int D = sizeof(V) / 4;
    struct Dwords {
        unsigned d[D];
    } t;
#pragma unroll
    for (int q = 0; q + 4 <= D; q += 4) {
        const ColumnU4 u = __builtin_amdgcn_raw_buffer_load_b128(bufferRsrc(b), bufferOffset(off + 4 * q), 0, CP);
        t.d[q] = u.x;
        t.d[q + 1] = u.y;
        t.d[q + 2] = u.z;
        t.d[q + 3] = u.w;
    }
    constexpr int Q = D / 4 * 4;
    if constexpr (D - Q == 2) {
        const ColumnU2 u = __builtin_amdgcn_raw_buffer_load_b64(bufferRsrc(b), bufferOffset(off + 4 * Q), 0, CP);
        t.d[Q] = u.x;
        t.d[Q + 1] = u.y;
    } else if constexpr (D - Q == 1) {
        t.d[Q] = __builtin_amdgcn_raw_buffer_load_b32(bufferRsrc(b), bufferOffset(off + 4 * Q), 0, CP);
    }
    __builtin_memcpy(&v, &t, sizeof(V));
}
template <int CP, class V>
__device__ __forceinline__ void bufferStore(const V &v, const ColumnBuffer &b, unsigned off) {
    constexpr int D = sizeof(V) / 4;
    struct Dwords {
        unsigned d[D];
    } t;
    __builtin_memcpy(&t, &v, sizeof(V));
#pragma unroll
    for (int q = 0; q + 4 <= D; q += 4)
        __builtin_amdgcn_raw_buffer_store_b128(ColumnU4{t.d[q], t.d[q + 1], t.d[q + 2], t.d[q + 3]}, bufferRsrc(b),
                                               bufferOffset(off + 4 * q), 0, CP);
    constexpr int Q = D / 4 * 4;
    if constexpr (D - Q == 2)
        __builtin_amdgcn_raw_buffer_store_b64(ColumnU2{t.d[Q], t.d[Q + 1]}, bufferRsrc(b), bufferOffset(off + 4 * Q), 0,
                                              CP);
    else if constexpr (D - Q == 1)
        __builtin_amdgcn_raw_buffer_store_b32(t.d[Q], bufferRsrc(b), bufferOffset(off + 4 * Q), 0, CP);
}

// (an LDS pointer by type: the compiler leaves a volatile access through a
// generic one a flat access)
template <class U>
using LdsVolatile = volatile __attribute__((address_space(3))) U;
template <class U>
__device__ __forceinline__ U ldsLoadBits(void *p) {
    return __hip_atomic_load((LdsVolatile<U> *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class U>
__device__ __forceinline__ void ldsStoreBits(void *p, U v) {
    __hip_atomic_store((LdsVolatile<U> *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int ldsLoad(int *p) { return ldsLoadBits<int>(p); }
__device__ __forceinline__ float ldsLoad(float *p) { return __uint_as_float(ldsLoadBits<unsigned>(p)); }
__device__ __forceinline__ double ldsLoad(double *p) {
    return __longlong_as_double((long long)ldsLoadBits<unsigned long long>(p));
}
__device__ __forceinline__ void ldsStore(int *p, int v) { ldsStoreBits<int>(p, v); }
__device__ __forceinline__ void ldsStore(float *p, float v) { ldsStoreBits<unsigned>(p, __float_as_uint(v)); }
__device__ __forceinline__ void ldsStore(double *p, double v) {
    ldsStoreBits<unsigned long long>(p, (unsigned long long)__double_as_longlong(v));
}

template <bool FWD>
__device__ __forceinline__ unsigned rowShift(unsigned v, unsigned ext) {
    return __builtin_amdgcn_update_dpp(ext, v, FWD ? 0x111 : 0x101, 0xf, 0xf, false);
}
// rows R0..R3 -> {ext, R0, R1, R2} or {R1, R2, R3, ext}: swapping the rows of
// a pair gives {R0, R0, R2, R2} and {R1, R1, R3, R3}, swapping halves the row
// that crosses them
template <bool FWD>
__device__ __forceinline__ unsigned lineShift(unsigned v, unsigned ext) {
    const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    if (FWD) {
        const auto q = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
        const unsigned w = __builtin_amdgcn_update_dpp(ext, p[0], 0xE4, 0xA, 0xF, false);
        return __builtin_amdgcn_update_dpp(w, q[0], 0xE4, 0x4, 0xF, false);
    }
    const auto q = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
    const unsigned w = __builtin_amdgcn_update_dpp(ext, p[1], 0xE4, 0x5, 0xF, false);
    return __builtin_amdgcn_update_dpp(w, q[1], 0xE4, 0x2, 0xF, false);
}
template <bool FWD>
__device__ __forceinline__ float rowShift(float v, float ext) {
    return __uint_as_float(rowShift<FWD>(__float_as_uint(v), __float_as_uint(ext)));
}
template <bool FWD>
__device__ __forceinline__ double rowShift(double v, double ext) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(v), b = (unsigned long long)__double_as_longlong(ext);
    return joinDouble(rowShift<FWD>((unsigned)a, (unsigned)b), rowShift<FWD>((unsigned)(a >> 32), (unsigned)(b >> 32)));
}
template <bool FWD>
__device__ __forceinline__ float lineShift(float v, float ext) {
    return __uint_as_float(lineShift<FWD>(__float_as_uint(v), __float_as_uint(ext)));
}
template <bool FWD>
__device__ __forceinline__ double lineShift(double v, double ext) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(v), b = (unsigned long long)__double_as_longlong(ext);
    return joinDouble(lineShift<FWD>((unsigned)a, (unsigned)b), lineShift<FWD>((unsigned)(a >> 32), (unsigned)(b >> 32)));
}

}  // namespace ff
