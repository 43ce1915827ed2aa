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
