// gfx950 (MI355X) kernels of prompt reading on the matrix cores: the batched
// products whose every output keeps a GEMV's float order. A code object of
// its own (prompt.hsaco), kernels named sml_pp_*.
#include "dev.h"

// The codes of chunk c as bytes: ca for group c&~1, cb for group c|1, each
// over the chunk's 16 columns (0 .. 2^NB - 1).
template <int NB>
__device__ __forceinline__ void chunk_codes(const ChunkW<NB> & w, int c, v4u & ca, v4u & cb) {
    using P = Planes<NB>;
    ca = v4u{0u, 0u, 0u, 0u};
    cb = ca;
    int sh = 0;
    if constexpr (P::N4) { ca = w.n4 & 0x0F0F0F0Fu; cb = (w.n4 >> 4u) & 0x0F0F0F0Fu; sh = 4; }
    if constexpr (NB == 8) { ca |= (w.h4 & 0x0F0F0F0Fu) << 4u; cb |= w.h4 & 0xF0F0F0F0u; }
    if constexpr (P::N2) {
        const unsigned k = 2u * (unsigned) (c & 2);          // bit-plane of group c&~1 within its pack
        const v4u ea = (w.t2 >> k) & 0x03030303u, eb = (w.t2 >> (k + 2u)) & 0x03030303u;
        ca |= ea << (unsigned) sh;
        cb |= eb << (unsigned) sh;
        sh += 2;
    }
    if constexpr (P::N1) {
        const unsigned wa = w.o1.x >> (16 * (c & 1)), wb = w.o1.y >> (16 * (c & 1));
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            ca[i] |= bits4_to_bytes((wa >> (4 * i)) & 15u) << sh;
            cb[i] |= bits4_to_bytes((wb >> (4 * i)) & 15u) << sh;
        }
    }
}

// ---------------------------------------------------------------- batched GEMM in a GEMV's order
//
// Y[p][r] = W.a[p] for the positions p of a prompt chunk, every output bit
// for bit that position's GEMV: the group dots are integers, so the matrix
// cores may form them in any order, and the float epilogue then runs in the
// GEMV's. Per-32 activations (s_g, sum_g per group). Per (row, position) and
// group, with wsc = sd*sq_g and wmn = md*(mq_g - 127):
//     v = fma(wsc, s_g*dot_g, v);  v = fma(wmn, s_g*sum_g, v)
//  - REF false: gemv_body's order. Lane l of that kernel owns the groups
//    l, l + 64, ... of a row, in order, and the 64 lanes' sums meet in a
//    balanced binary tree. Here the groups go by quad: quad q of 0..15
//    covers lanes 4q..4q+3, its 4 chains run over the groups 64k + 4q + i
//    (k = 0, 1, ...), their sums meet as (v0+v1) + (v2+v3), and the 16 quads'
//    sums go through the tree's upper levels as a binary counter does (at
//    most 4 pending sums). Columns: a multiple of 128.
//  - REF true: the reference's order (gemv_body EX): chain j of 8 runs over
//    the groups j, j + 8, ... of the row; then ((v0+v4)+(v1+v5)) +
//    ((v2+v6)+(v3+v7)). Columns: a multiple of 256.
//
// Bound: VALU issue. A group of an output costs one conversion, one multiply
// and two fused multiply-adds for 32 multiply-adds of the dot, which take a
// sixteenth of a v_mfma_i32_16x16x32_i8. So the tile is chosen to keep
// everything else off the VALU: codes are unpacked to bytes, the fields
// converted and s_g*sum_g formed once per tile while it is staged in LDS, not
// once per wave or lane.
//
// Workgroup: 8 waves, 64 weight rows (SwiGLU: 32 rows of gate and the same 32
// of up) x 64 positions, a wave 32 x 16 as two MFMA tiles, two workgroups a
// CU. A stage holds 8 groups (REF: a superblock; else a quad at k and the
// same quad at k + 1) of the tile in LDS, 43 KB; the next stage's global
// loads are in flight while one computes. (4 waves of 32 x 32: 4% faster at 512
// positions of the SwiGLU, 30-60% slower where a launch has fewer workgroups
// than the chip takes, each stage's latency then being a wave's own.) In LDS
// a group's codes lie as [16-column half][row][16 bytes], so the stores are
// whole 16-byte words and the 32 lanes of two k-slices read 512 contiguous
// bytes. The MFMA's A holds positions and B weight rows: lane l owns weight
// row l%16 of a tile and its positions 4(l/16)..+3.
//
// Measured, 512 positions in one launch against the VALU GEMM in slices of 32
// (us): 2 x 14336 x 4096 SwiGLU 2944 -> 394, 4096 x 14336 1465 -> 208,
// 6144 x 4096 ~900 -> 104, 4096 x 4096 678 -> 67 (258 TOP/s; the VALU issues
// 80% of the time, 17 of its 25 instructions per tile and group the epilogue
// and the MFMA); REF against the earlier 16-row x 64-position form at 64
// positions: SwiGLU 148 -> 58, 4096 x 4096 36.8 -> 35.7.
#define PX_POS 64
#define PX_ROWS 64
#define PX_HALF (64 * 16 + 16)                       // bytes of half a group's codes (16 columns) in LDS
#define PX_SLOT (2 * PX_HALF)                        // bytes of a group's codes in LDS
#define PX_FROW 80                                   // bytes of a row's 8 (wsc, wmn) pairs
#define PX_SROW 68                                   // floats of a group's positions
#define PX_A (8 * PX_SLOT)
#define PX_F (2 * PX_A)
#define PX_S (PX_F + PX_ROWS * PX_FROW)
#define PX_LDS (PX_S + 2 * 8 * PX_SROW * 4)          // then, Q8: 8 x PX_SROW ints

template <int V> struct Int { static constexpr int value = V; };

template <int NB, bool SW, bool REF>
__device__ void px_body(const sml_kgemm & a) {
    #pragma clang fp contract(off)
    typedef long v1l;
    constexpr int NA = REF ? 8 : 4;                  // chains of a stage's groups
    extern __shared__ __align__(16) uint8_t lds[];
    const int n = a.cols, ng = n / 32, ns = (ng + 7) / 8, m_all = a.m_all, rows = a.rows;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, i16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 1, wp = wave >> 1;
    // consecutive tiles share their weight rows and sit on one XCD (workgroup
    // i runs on XCD i mod 8), so the position tiles find them in its L2
    constexpr int RT = SW ? PX_ROWS / 2 : PX_ROWS;
    const int nrt = (rows + RT - 1) / RT, npt = (m_all + PX_POS - 1) / PX_POS, total = nrt * npt;
    const int id = blockIdx.x, xcd = id & 7, slot = id >> 3, q8 = total >> 3, rem = total & 7;
    const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + slot;
    const int rt = lid / npt, r0 = rt * RT, p0 = (lid - rt * npt) * PX_POS;

    // staging of the weight rows: thread t takes chunk t%8 of the stage's two
    // quads (4 chunks of 16 bytes each) of row t/8
    const sml_kmat & mk0 = a.m0[0];
    const sml_kmat & mk1 = a.m0[SW ? 1 : 0];
    using P = Planes<NB>;
    const int j8 = tid & 7, wrow = tid >> 3;
    const bool up = SW && wrow >= 32;
    const uint32_t r = (uint32_t) min(r0 + (SW ? wrow & 31 : wrow), rows - 1);
    const uint8_t * pl[3];
    uint32_t ro[3] = {0, 0, 0};
    #pragma unroll
    for (int k = 0; k < 3; k++) pl[k] = up ? mk1.plane[k] : mk0.plane[k];
    if constexpr (P::N4) ro[P::P4] = r * (uint32_t) P::b4(n);
    if constexpr (NB == 8) ro[1] = r * (uint32_t) P::b4(n);
    if constexpr (P::N2) ro[P::P2] = r * (uint32_t) P::b2(n);
    if constexpr (P::N1) ro[P::P1] = r * (uint32_t) P::b1(n);
    // the fields: a thread takes the group pair t%4 of weight row t/4 (the
    // first 256 threads) or of position t/4 (the others)
    const int fp = tid & 3, fr = (tid & 255) >> 2;
    const bool frows = tid < 256;
    const sml_kmat & mf = SW && fr >= 32 ? mk1 : mk0;
    const uint32_t frow = (uint32_t) min(r0 + (SW ? fr & 31 : fr), rows - 1);
    const uint8_t * fqb = mf.sqmq + (size_t) frow * ng * 2;
    const uint8_t * fdb = (const uint8_t *) mf.sdmd + (size_t) frow * ns * 4;
    const size_t fpos = (size_t) min(p0 + fr, m_all - 1) * ng;
    // the activation codes: thread t takes 16-byte word t%16 of positions t/16 and t/16 + 32
    const int ja = tid & 15;
    uint32_t aoff[2];
    #pragma unroll
    for (int i = 0; i < 2; i++) aoff[i] = (uint32_t) min(p0 + (tid >> 4) + 32 * i, m_all - 1) * (uint32_t) n;

    // stage (q, k): REF superblock k; else quad q's groups 64k + 4q.. in slots
    // 0-3 and 64(k+1) + 4q.. in slots 4-7 (k + 1 past the row: the first again)
    ChunkW<NB> cw;
    v4u aw[2];
    uint32_t fqv, fdv;
    float2 sv;
    int2 uv;
    auto first_group = [&](int q, int k, int half) -> int {
        if constexpr (REF) return 8 * k + 4 * half;
        const int g = 64 * (k + half) + 4 * q;
        return g < ng ? g : 64 * k + 4 * q;
    };
    auto fetch = [&](int q, int k) {
        const int gw = first_group(q, k, j8 >> 2), ga = first_group(q, k, ja >> 3), gf = first_group(q, k, fp >> 1) + 2 * (fp & 1);
        load_chunk<NB, false>(cw, pl, ro, gw + (j8 & 3));
        #pragma unroll
        for (int i = 0; i < 2; i++) aw[i] = gld<v4u>(a.q + (aoff[i] + 32u * (uint32_t) ga + 16u * (uint32_t) (ja & 7)));
        if (frows) {
            fqv = gld<uint32_t>(fqb + 2 * gf);
            fdv = gld<uint32_t>(fdb + 4 * (gf >> 3));
        } else {
            sv = gld<float2>(a.scale + fpos + gf);
            uv = gld<int2>(a.sums + fpos + gf);
        }
    };
    float * const lss = (float *) (lds + PX_S);                  // [8][PX_SROW] s
    float * const lsu = lss + 8 * PX_SROW;                       // [8][PX_SROW] s * sum
    int * const lsi = (int *) (lsu + 8 * PX_SROW);               // Q8: [8][PX_SROW] 128 * sum
    auto stage = [&]() {
        v4u ca, cb;
        chunk_codes<NB>(cw, j8, ca, cb);
        // Q8: codes less 128 (an int8); the dot gets 128 * sum back as the MFMA's C
        if constexpr (NB == 8) { ca ^= 0x80808080u; cb ^= 0x80808080u; }
        uint8_t * d = lds + (j8 & 6) * PX_SLOT + (j8 & 1) * PX_HALF + wrow * 16;
        *(v4u *) d = ca;
        *(v4u *) (d + PX_SLOT) = cb;
        #pragma unroll
        for (int i = 0; i < 2; i++) *(v4u *) (lds + PX_A + ja * PX_HALF + ((tid >> 4) + 32 * i) * 16) = aw[i];
        if (frows) {
            const float sd = h2f((uint16_t) (fdv & 0xFFFFu)), md = h2f((uint16_t) (fdv >> 16));
            *(float4 *) (lds + PX_F + fr * PX_FROW + fp * 16) =
                make_float4(sd * (float) (fqv & 0xFFu), md * ((float) ((fqv >> 8) & 0xFFu) - 127.0f),
                            sd * (float) ((fqv >> 16) & 0xFFu), md * ((float) (fqv >> 24) - 127.0f));
        } else {
            lss[2 * fp * PX_SROW + fr] = sv.x;
            lss[(2 * fp + 1) * PX_SROW + fr] = sv.y;
            lsu[2 * fp * PX_SROW + fr] = sv.x * (float) uv.x;
            lsu[(2 * fp + 1) * PX_SROW + fr] = sv.y * (float) uv.y;
            if constexpr (NB == 8) {
                lsi[2 * fp * PX_SROW + fr] = 128 * uv.x;
                lsi[(2 * fp + 1) * PX_SROW + fr] = 128 * uv.y;
            }
        }
    };

    // the wave's LDS rows: weight tile t, position tile u
    int lrow[2];
    #pragma unroll
    for (int t = 0; t < 2; t++) lrow[t] = (SW ? 32 * t + 16 * wr : 32 * wr + 16 * t) + i16;
    float acc[NA][2][4];                             // [chain][weight tile][position]
    #pragma unroll
    for (int j = 0; j < NA; j++)
        #pragma unroll
        for (int t = 0; t < 2; t++)
            #pragma unroll
            for (int r = 0; r < 4; r++) acc[j][t][r] = 0.0f;
    auto compute = [&](auto half) {                  // slots 4 half .. 4 half + 3
        #pragma unroll
        for (int gg = 0; gg < 4; gg++) {
            constexpr int H = decltype(half)::value;
            const int g = 4 * H + gg, j = REF ? g : gg;
            const uint8_t * sl = lds + g * PX_SLOT + (kq >> 1) * PX_HALF + (kq & 1) * 8;
            const v1l av = *(const v1l *) (sl + PX_A + (16 * wp + i16) * 16);
            const float4 s4 = *(const float4 *) (lss + g * PX_SROW + 16 * wp + 4 * kq);
            const float4 u4 = *(const float4 *) (lsu + g * PX_SROW + 16 * wp + 4 * kq);
            const v4i c0 = NB == 8 ? *(const v4i *) (lsi + g * PX_SROW + 16 * wp + 4 * kq) : v4i{0, 0, 0, 0};
            const float sp[4] = {s4.x, s4.y, s4.z, s4.w}, up[4] = {u4.x, u4.y, u4.z, u4.w};
            #pragma unroll
            for (int t = 0; t < 2; t++) {
                const v1l bv = *(const v1l *) (sl + lrow[t] * 16);
                const float2 wf = *(const float2 *) (lds + PX_F + lrow[t] * PX_FROW + g * 8);
                const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, c0, 0, 0, 0);
                #pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float v = __builtin_fmaf(wf.x, sp[r] * (float) d[r], acc[j][t][r]);
                    acc[j][t][r] = __builtin_fmaf(wf.y, up[r], v);
                }
            }
            // order the groups (an empty statement on the sums so far): left
            // free, every group's products are formed before the first is
            // consumed, and the registers of all are live at once
            #pragma unroll
            for (int t = 0; t < 2; t++)
                asm volatile("" : "+v"(acc[j][t][0]), "+v"(acc[j][t][1]), "+v"(acc[j][t][2]), "+v"(acc[j][t][3]));
        }
    };

    float out[2][4];
    fetch(0, 0);
    stage();
    __syncthreads();
    if constexpr (REF) {
        const int nsb = ng / 8;
        for (int b = 0; b < nsb; b++) {
            const bool more = b + 1 < nsb;
            if (more) fetch(0, b + 1);
            compute(Int<0>());
            compute(Int<1>());
            __syncthreads();
            if (more) stage();
            __syncthreads();
        }
        #pragma unroll
        for (int t = 0; t < 2; t++)
            #pragma unroll
            for (int r = 0; r < 4; r++) {
                auto v = [&](int j) { return acc[j % NA][t][r]; };
                out[t][r] = ((v(0) + v(4)) + (v(1) + v(5))) + ((v(2) + v(6)) + (v(3) + v(7)));
            }
    } else {
        float st[4][2][4];                           // the tree's pending sums, by level
        for (int q = 0; q < 16; q++) {
            for (int k = 0; 64 * k + 4 * q < ng; k += 2) {
                int nq = q, nk = k + 2;
                if (64 * nk + 4 * nq >= ng) { nq++; nk = 0; }
                const bool more = nq < 16 && 4 * nq < ng;
                if (more) fetch(nq, nk);
                compute(Int<0>());
                if (64 * (k + 1) + 4 * q < ng) compute(Int<1>());
                __syncthreads();
                if (more) stage();
                __syncthreads();
            }
            #pragma unroll
            for (int t = 0; t < 2; t++)
                #pragma unroll
                for (int r = 0; r < 4; r++) {
                    out[t][r] = (acc[0][t][r] + acc[1][t][r]) + (acc[2][t][r] + acc[3][t][r]);
                    #pragma unroll
                    for (int j = 0; j < 4; j++) acc[j][t][r] = 0.0f;
                }
            // up the tree: a level's second sum joins the first and moves on
            #pragma unroll
            for (int lv = 0; lv < 4; lv++) {
                const bool second = (q >> lv) & 1;
                #pragma unroll
                for (int t = 0; t < 2; t++)
                    #pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (second) out[t][r] = st[lv][t][r] + out[t][r];
                        else st[lv][t][r] = out[t][r];
                    }
                if (!second) break;
            }
        }
    }

    #pragma unroll
    for (int r = 0; r < 4; r++) {
        const int pos = p0 + 16 * wp + 4 * kq + r;
        if (pos >= m_all) continue;
        float * y = a.y + (size_t) pos * rows;
        if constexpr (SW) {
            const int row = r0 + 16 * wr + i16;
            if (row < rows) y[row] = silu_ref(out[0][r]) * out[1][r];            // sml/sml-run.c:416-426
        } else {
            #pragma unroll
            for (int t = 0; t < 2; t++) {
                const int row = r0 + 32 * wr + 16 * t + i16;
                if (row >= rows) continue;
                float v = out[t][r];
                if (a.bias) v += a.bias[row];
                if (a.resid) v = a.resid[(size_t) pos * rows + row] + v;
                y[row] = v;
            }
        }
    }
}

// four waves a SIMD (two workgroups a CU): at most 128 registers
#define PX_KERNELS(NAME, NB, REF)                                                                                    \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME##NB(const sml_kgemm a) { px_body<NB, false, REF>(a); }   \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME##NB##_s(const sml_kgemm a) { px_body<NB, true, REF>(a); }
PX_KERNELS(sml_pp_gemm_q, 2, false) PX_KERNELS(sml_pp_gemm_q, 3, false) PX_KERNELS(sml_pp_gemm_q, 4, false)
PX_KERNELS(sml_pp_gemm_q, 5, false) PX_KERNELS(sml_pp_gemm_q, 6, false) PX_KERNELS(sml_pp_gemm_q, 7, false)
PX_KERNELS(sml_pp_gemm_q, 8, false) PX_KERNELS(sml_pp_xgemm_q, 4, true) PX_KERNELS(sml_pp_xgemm_q, 8, true)
