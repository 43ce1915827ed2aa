// Device code shared by the gfx950 code objects (kernels.hip, prompt.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "kargs.h"

#define WAVE 64

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// Global-memory views of device pointers. A pointer read from a table in
// device memory (expert matrices, KV slots) or selected at run time is
// generic to the compiler, and loads through it become flat loads. A flat
// load counts against the LDS/scalar wait counter as well as the vector
// one, so every LDS or scalar-load wait after it also waits for it, and the
// vector waits can no longer be partial: a kernel that overlaps its weight
// or KV stream with LDS work then runs serially. Every such pointer here
// points to global memory.
#define GLOBAL __attribute__((address_space(1)))
template <typename T> __device__ __forceinline__ T gld(const void * p) { return *(const GLOBAL T *) p; }

__device__ __forceinline__ float h2f(uint16_t h) { return (float) __builtin_bit_cast(_Float16, h); }
__device__ __forceinline__ uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, (_Float16) f); }

// 4 bits (one per column) -> 4 bytes of 0/1
__device__ __forceinline__ unsigned bits4_to_bytes(unsigned nib) { return (nib * 0x00204081u) & 0x01010101u; }

// ---------------------------------------------------------------- chunks
//
// A chunk is 16 bytes of a row's nibble plane: columns 16*(c&1)..+15 of the
// group pair (c&~1, c|1) -- byte i's low nibble belongs to the first group,
// its high nibble to the second (the FLAT layout, sml/sml-kernel.c:2140-2156).
// Lane c of a row loads chunk c, so 64 lanes read 1 KB of contiguous bytes
// per instruction; the other planes' bytes for the same weights are equally
// contiguous across lanes (a 2-bit pack serves two lanes, a 1-bit word pair
// serves a lane pair). Plane orders per width follow
// tooling/sml_quantize.py:104-106: Q2 [2], Q3 [2,1], Q4 [4], Q5 [4,1],
// Q6 [2,4] (the 2-bit plane holds bits 4-5), Q7 [4,2,1], Q8 [4,4].
template <int NB> struct Planes {
    static constexpr bool N4 = NB == 4 || NB == 5 || NB == 6 || NB == 7 || NB == 8;
    static constexpr bool N2 = NB == 2 || NB == 3 || NB == 6 || NB == 7;
    static constexpr bool N1 = NB == 3 || NB == 5 || NB == 7;
    static constexpr int P4 = NB == 6 ? 1 : 0;
    static constexpr int P2 = NB == 7 ? 1 : 0;
    static constexpr int P1 = NB == 7 ? 2 : 1;
    // bytes of each plane per row for `cols` weights
    static __device__ __forceinline__ size_t b4(int cols) { return (size_t) cols / 2; }
    static __device__ __forceinline__ size_t b2(int cols) { return (size_t) cols / 4; }
    static __device__ __forceinline__ size_t b1(int cols) { return (size_t) cols / 8; }
};

template <bool NT, typename T>
__device__ __forceinline__ T ld(const T * p) {
    const GLOBAL T * g = (const GLOBAL T *) p;
    if constexpr (NT) return __builtin_nontemporal_load(g);
    else return *g;
}

template <int NB> struct ChunkW {
    v4u n4;                       // nibble plane word (or zeros)
    v4u h4;                       // Q8 high nibbles
    v4u t2;                       // 2-bit pack half
    v2u o1;                       // 1-bit words of the group pair
};

// Chunk c of one row: pl[] are the planes' bases (uniform), ro[] the row's
// byte offset in each plane. Offsets are 32-bit so the loads address as
// uniform base + per-lane offset, which keeps one VGPR per address.
template <int NB, bool NT>
__device__ __forceinline__ void load_chunk(ChunkW<NB> & w, const uint8_t * const * pl, const uint32_t * ro, int c) {
    using P = Planes<NB>;
    if constexpr (P::N4) w.n4 = ld<NT>((const v4u *) (pl[P::P4] + (ro[P::P4] + (uint32_t) c * 16u)));
    if constexpr (NB == 8) w.h4 = ld<NT>((const v4u *) (pl[1] + (ro[1] + (uint32_t) c * 16u)));
    if constexpr (P::N2) w.t2 = ld<NT>((const v4u *) (pl[P::P2] + (ro[P::P2] + (uint32_t) (c >> 2) * 32u + (uint32_t) (c & 1) * 16u)));
    if constexpr (P::N1) w.o1 = ld<NT>((const v2u *) (pl[P::P1] + (ro[P::P1] + (uint32_t) (c >> 1) * 8u)));
}

// SiLU as the reference's x86 build computes it (sml_exp_ps + silu_mul,
// sml/sml-run.c:393-426): the argument clamped to [-88, 88], f = x*log2(e),
// r = f rounded half-even, 2^(f-r) by a degree-5 Horner chain of FMAs, and
// 1 + p*2^r folded into one FMA (how that build's compiler contracts it);
// then g / d. Contraction is off so f and f - r round as written.
__device__ __forceinline__ float silu_ref(float g) {
    #pragma clang fp contract(off)
    float x = 0.0f - g;
    x = fminf(fmaxf(x, -88.0f), 88.0f);
    const float f = x * 1.44269504088896341f;
    const float r = __builtin_rintf(f);
    const float t = f - r;
    float p = __builtin_fmaf(1.3697664e-3f, t, 8.3013611e-3f);
    p = __builtin_fmaf(p, t, 5.5826318e-2f);
    p = __builtin_fmaf(p, t, 2.4022652e-1f);
    p = __builtin_fmaf(p, t, 6.9314718e-1f);
    p = __builtin_fmaf(p, t, 1.0f);
    const float sc = __builtin_bit_cast(float, ((int) r + 127) << 23);
    return g / __builtin_fmaf(p, sc, 1.0f);
}

// ---------------------------------------------------------------- reductions, activation codes

__device__ __forceinline__ float wave_sum(float v) {
    #pragma unroll
    for (int o = 32; o; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    #pragma unroll
    for (int o = 32; o; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
// Butterflies inside a 16-lane DPP row (quad_perm xor 1, xor 2, then the
// half-row and row mirrors): every lane of the row ends with the row's result.
// A swizzle (xor 16) extends them to 32 lanes.
template <int CTRL> __device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
template <int CTRL> __device__ __forceinline__ int dpp_i(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false); }
__device__ __forceinline__ float sum16(float v) {
    v += dpp_f<0xB1>(v); v += dpp_f<0x4E>(v); v += dpp_f<0x141>(v); v += dpp_f<0x140>(v);
    return v;
}
__device__ __forceinline__ float max16(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v)); v = fmaxf(v, dpp_f<0x4E>(v)); v = fmaxf(v, dpp_f<0x141>(v)); v = fmaxf(v, dpp_f<0x140>(v));
    return v;
}
__device__ __forceinline__ int isum16(int v) {
    v += dpp_i<0xB1>(v); v += dpp_i<0x4E>(v); v += dpp_i<0x141>(v); v += dpp_i<0x140>(v);
    return v;
}
// xor 16 within 32 lanes (ds_swizzle bit mode: and 0x1F, xor 0x10)
__device__ __forceinline__ float swz16_f(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
}
__device__ __forceinline__ float sum32(float v) { v = sum16(v); return v + swz16_f(v); }
__device__ __forceinline__ float max32(float v) { v = max16(v); return fmaxf(v, swz16_f(v)); }
__device__ __forceinline__ int isum32(int v) { v = isum16(v); return v + __builtin_amdgcn_ds_swizzle(v, 0x401F); }

// Max / sum over aligned groups of 8 lanes (quad butterflies, then the half-row mirror)
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v)); v = fmaxf(v, dpp_f<0x4E>(v)); return fmaxf(v, dpp_f<0x141>(v));
}
__device__ __forceinline__ int isum8(int v) { v += dpp_i<0xB1>(v); v += dpp_i<0x4E>(v); return v + dpp_i<0x141>(v); }

// One activation code: lrintf(v * is) clamped to +-127, where an out-of-range
// or NaN product converts to INT_MIN as the reference's x86 build does
// (sml/sml-kernel.c:86-106), so it clamps to -127.
__device__ __forceinline__ int quant1(float v, float is) {
    const float r = __builtin_rintf(v * is);
    int t = (r >= -2147483648.0f && r < 2147483648.0f) ? (int) r : (int) 0x80000000u;
    return t > 127 ? 127 : t < -127 ? -127 : t;
}

// The sum of squares as the reference build computes it (sml/sml-run.c:
// 147-152, a serial loop its compiler turns into double FMAs): one lane, in
// order. Loads run ahead of the dependent chain in blocks of 16. x is in
// global memory or in LDS (generic loads: this is the rare fallback of the
// checked parallel sum below).
__device__ __noinline__ double serial_ss(const float * x, int n) {
    double ss = 0.0;
    int i = 0;
    for (; i + 16 <= n; i += 16) {
        float v[16];
        #pragma unroll
        for (int j = 0; j < 16; j++) v[j] = x[i + j];
        #pragma unroll
        for (int j = 0; j < 16; j++) ss = __builtin_fma((double) v[j], (double) v[j], ss);
    }
    for (; i < n; i++) { const float v = x[i]; ss = __builtin_fma((double) v, (double) v, ss); }
    return ss;
}

// float(ss/n) of the serial chain above, from a sum of the same squares taken
// in any order. Every square is exact in double (24-bit mantissas), all are
// nonnegative, so each order's sum lies within (n-1)*2^-53*(1+2^-30) of the
// exact sum, relatively: the serial and the given sum differ by less than
// d = 4*(n+4)*2^-53*s, with a margin for the rounding of d itself. Division
// by n and the float conversion are monotone, so when s-d and s+d give the
// same float that float is the serial chain's; it fails for about one input
// in 10^4 (a rounding boundary inside the window) and for inf/NaN sums, and
// the caller then runs the chain.
__device__ __forceinline__ bool ss_mean_alike(double s, int n, float & out) {
    const double d = s * ((double) (4 * (n + 4)) * 0x1p-53);
    const float lo = (float) ((s - d) / (double) n), hi = (float) ((s + d) / (double) n);
    out = lo;
    return lo == hi;
}

// Four values' squares added to a double sum, in sml_normq2's order (its
// callers share it so that their sums agree bit for bit).
__device__ __forceinline__ double ss_add4(double ss, float4 v) {
    return ss + ((double) v.x * v.x + (double) v.y * v.y + (double) v.z * v.z + (double) v.w * v.w);
}
