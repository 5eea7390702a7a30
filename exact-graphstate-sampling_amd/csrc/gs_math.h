// Device helpers shared by the kernel files: storage traits, complex FP64 arithmetic, a string's own buffers, arena
// accesses.
#pragma once
#include "gs_device.h"

namespace gs {

// storage traits
template <class S>
struct Cx;

template <>
struct Cx<float2> {
    static __device__ __forceinline__ double2 widen(float2 a) { return make_double2(double(a.x), double(a.y)); }
    static __device__ __forceinline__ float2 narrow(double2 a) { return make_float2(float(a.x), float(a.y)); }
};

template <>
struct Cx<double2> {
    static __device__ __forceinline__ double2 widen(double2 a) { return a; }
    static __device__ __forceinline__ double2 narrow(double2 a) { return a; }
};

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
// a * b + c (complex, FP64)
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
    return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double norm2(double2 a) { return fma(a.x, a.x, a.y * a.y); }
// acc += |a|^2 as two fused multiply-adds
__device__ __forceinline__ void add_norm(double& acc, double2 a) { acc = fma(a.x, a.x, fma(a.y, a.y, acc)); }

// The per-string buffers of the epilogue's arguments for this block's string (blockIdx.y).
__device__ __forceinline__ Epi slot_epi(const Epi& e) {
    Epi s = e;
    const size_t y = blockIdx.y, at = y * size_t(e.ns);
    if (s.forced) s.forced += at;
    s.U += at;
    s.bits += at;
    s.cond += at;
    s.out += 4 * y;
    s.counter += y;
    return s;
}

// Arena accesses carry the non-temporal hint: every sweep streams the table once, so its lines should not displace
// anything in L2, and written lines leave few dirty lines behind.
typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float2 ld_nt(const float2* p) {
    const f2v t = __builtin_nontemporal_load(reinterpret_cast<const f2v*>(p));
    return make_float2(t.x, t.y);
}
__device__ __forceinline__ void st_nt(float2* p, float2 v) {
    const f2v t = {v.x, v.y};
    __builtin_nontemporal_store(t, reinterpret_cast<f2v*>(p));
}
__device__ __forceinline__ float4 ld_nt4(const float2* p) {
    const f4v t = __builtin_nontemporal_load(reinterpret_cast<const f4v*>(p));
    return make_float4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ void st_nt4(float2* p, float2 a, float2 b) {
    const f4v t = {a.x, a.y, b.x, b.y};
    __builtin_nontemporal_store(t, reinterpret_cast<f4v*>(p));
}
__device__ __forceinline__ double2 ld_nt(const double2* p) {
    const d2v t = __builtin_nontemporal_load(reinterpret_cast<const d2v*>(p));
    return make_double2(t.x, t.y);
}
__device__ __forceinline__ void st_nt(double2* p, double2 v) {
    const d2v t = {v.x, v.y};
    __builtin_nontemporal_store(t, reinterpret_cast<d2v*>(p));
}

// VR consecutive arena entries at an aligned index, as 16-byte vector accesses.
template <class S, int VR>
struct Run;

template <>
struct Run<float2, 1> {
    static __device__ __forceinline__ void load(const float2* m, uint64_t a, float2 (&e)[1]) { e[0] = ld_nt(m + a); }
    static __device__ __forceinline__ void store(float2* m, uint64_t a, const float2 (&e)[1]) { st_nt(m + a, e[0]); }
};
template <>
struct Run<float2, 2> {
    static __device__ __forceinline__ void load(const float2* m, uint64_t a, float2 (&e)[2]) {
        const float4 x = ld_nt4(m + a);
        e[0] = make_float2(x.x, x.y);
        e[1] = make_float2(x.z, x.w);
    }
    static __device__ __forceinline__ void store(float2* m, uint64_t a, const float2 (&e)[2]) {
        st_nt4(m + a, e[0], e[1]);
    }
};
template <>
struct Run<float2, 4> {
    static __device__ __forceinline__ void load(const float2* m, uint64_t a, float2 (&e)[4]) {
        const float4 x = ld_nt4(m + a);
        const float4 y = ld_nt4(m + a + 2);
        e[0] = make_float2(x.x, x.y);
        e[1] = make_float2(x.z, x.w);
        e[2] = make_float2(y.x, y.y);
        e[3] = make_float2(y.z, y.w);
    }
    static __device__ __forceinline__ void store(float2* m, uint64_t a, const float2 (&e)[4]) {
        st_nt4(m + a, e[0], e[1]);
        st_nt4(m + a + 2, e[2], e[3]);
    }
};
template <>
struct Run<double2, 1> {
    static __device__ __forceinline__ void load(const double2* m, uint64_t a, double2 (&e)[1]) { e[0] = ld_nt(m + a); }
    static __device__ __forceinline__ void store(double2* m, uint64_t a, const double2 (&e)[1]) { st_nt(m + a, e[0]); }
};
template <>
struct Run<double2, 2> {
    static __device__ __forceinline__ void load(const double2* m, uint64_t a, double2 (&e)[2]) {
        e[0] = ld_nt(m + a);
        e[1] = ld_nt(m + a + 1);
    }
    static __device__ __forceinline__ void store(double2* m, uint64_t a, const double2 (&e)[2]) {
        st_nt(m + a, e[0]);
        st_nt(m + a + 1, e[1]);
    }
};

// e[i] <- e[i ^ p] for p < VR (per-lane conditional swaps; an involution, used for loads and stores alike).
template <class S, int VR>
__device__ __forceinline__ void permute(S (&e)[VR], unsigned p) {
    if constexpr (VR >= 2) {
        const bool s1 = p & 1;
#pragma unroll
        for (int i = 0; i < VR; i += 2) {
            const S a = e[i], b = e[i + 1];
            e[i] = s1 ? b : a;
            e[i + 1] = s1 ? a : b;
        }
    }
    if constexpr (VR >= 4) {
        const bool s2 = p & 2;
#pragma unroll
        for (int i = 0; i < VR; i++) {
            if (i & 2) continue;
            const S a = e[i], b = e[i + 2];
            e[i] = s2 ? b : a;
            e[i + 2] = s2 ? a : b;
        }
    }
}

}  // namespace gs
