// gfx950 (MI355X) kernels of prompt reading on the matrix cores: the batched
// products whose every output keeps a GEMV's float order. A code object of
// its own (prompt.hsaco), kernels named sml_pp_*.
#include "dev.h"

// four words of an array that is aligned as its elements only
struct __attribute__((packed, aligned(4))) int4_a4 { int x, y, z, w; };
struct __attribute__((packed, aligned(4))) float4_a4 { float x, y, z, w; };

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

template <int NB, bool SW, bool REF, bool FEW = false>
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
        if (FEW && p0 + 16 * wp >= m_all) return;    // no position: the wave only stages
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

// Four waves a SIMD (two workgroups a CU): at most 128 registers, and no
// instance but sml_pp_xgemm_q4 fits: a lane's sums and chains, the pending tree
// sums (32) and the next stage's loads spill 2 to 21 registers (Q4 4 and 6 of
// the SwiGLU, Q7 and Q8 15 and 21) to scratch.
#define PX_KERNELS(NAME, NB, REF)                                                                                    \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME##NB(const sml_kgemm a) { px_body<NB, false, REF>(a); }   \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME##NB##_s(const sml_kgemm a) { px_body<NB, true, REF>(a); }
PX_KERNELS(sml_pp_gemm_q, 2, false) PX_KERNELS(sml_pp_gemm_q, 3, false) PX_KERNELS(sml_pp_gemm_q, 4, false)
PX_KERNELS(sml_pp_gemm_q, 5, false) PX_KERNELS(sml_pp_gemm_q, 6, false) PX_KERNELS(sml_pp_gemm_q, 7, false)
PX_KERNELS(sml_pp_gemm_q, 8, false) PX_KERNELS(sml_pp_xgemm_q, 4, true) PX_KERNELS(sml_pp_xgemm_q, 8, true)
// The reference order in launches of at most a workgroup a CU, where a stage's
// own latency is the time: registers for all of it (131 to 142, nothing
// spilled), and waves without a position leave their SIMD to the others. Two
// Qwen2.5-1.5B-shaped layers, exact mode, whole prompt of 2 / 32 / 64 ids (us):
// Q8 423 / 451 / 480 -> 332 / 366 / 429, Q4 347 / 374 / 403 -> 315 / 345 / 387;
// where a CU takes more workgroups the second one hides as much (Llama-3-8B
// shape, Q4, 512 ids: 2907, 3048 so).
#define PX_FEW(NB)                                                                                                           \
    extern "C" __global__ __launch_bounds__(512, 2) void sml_pp_xgemm_q##NB##_f(const sml_kgemm a) { px_body<NB, false, true, true>(a); } \
    extern "C" __global__ __launch_bounds__(512, 2) void sml_pp_xgemm_q##NB##_s_f(const sml_kgemm a) { px_body<NB, true, true, true>(a); }
PX_FEW(4) PX_FEW(8)

// ---------------------------------------------------------------- prompt GEMM in the superblock regime
//
// Y[p][r] = W.a[p] for a chunk of prompt positions p (hundreds) and every row
// r of a Q4 or Q6 matrix, in the reference's prompt regime (sml_quantize_act_sb
// and flat4_sb_body, sml/sml-kernel.c:115-185,1142-1190): per superblock b of
// 256 columns the integer sums
//     isum = sum_g sq_g * dot_g,    imin = sum_g (mq_g - 127) * sum(q_g),
// then y = fma(isum, sd_b * s_b, y); y = fma(imin, md_b * s_b, y) in fp32 (s_b:
// the position's activation scale of superblock b).
//
// Both sums run on the matrix cores whole, so the VALU touches an output once
// per superblock and not once per group:
//  - isum: v = sq_g * code < 2^14 is split into signed bytes, v = 256 hi + lo
//    (lo = v's low byte as an int8, hi = (v + 128) >> 8), and the superblock's
//    dots with hi and with lo are 4 chained v_mfma_i32_16x16x64_i8 each (|isum|
//    < 2^31). Twice the matrix operations of one dot per group, at the full
//    rate of the K = 64 form (the K = 32 form runs at half of it), and no
//    multiply-add per group on the VALU.
//  - imin: one v_mfma_f32_16x16x16_f16 over the 8 groups' sums, each as its
//    low 6 bits and the rest (both exact in fp16), against mq_g - 127 twice;
//    every product and partial sum is an integer below 2^24, so it is exact.
//
// Workgroup: 4 waves on the same 16 P positions, each on 16 weight rows of its
// own (SwiGLU: two on gate, two on the same rows of up). A wave reads its
// rows' planes straight into registers (16 rows x 64 bytes a load) and forms
// hi and lo there once per superblock, for all P position tiles: lane l holds
// row l%16 and, of 64 columns s, the 16 bytes that are its slice kq = l/16 of
// nibble word kq + 4 (s/2): group 4 (s/2) + 2 (kq/2) + s%2, columns 16
// (kq%2)..+15. The activation rows go to LDS as they are, copied by the memory
// unit itself (no registers), double-buffered a superblock ahead; word w of
// position p lies at w ^ (p % 16), so the 16 rows a wave reads at once fall
// into different banks. The MFMA's A holds positions and B weight rows: a lane
// owns weight row l%16 of a tile and positions 4 kq..+3.
//
// Bound: VALU issue, half of it used (a tile and superblock costs 24
// instructions of epilogue, 9 MFMAs and 200 / P of splitting the weights);
// the rest is waits of the two to four waves a SIMD holds. Against a dot per
// group with the multiply by sq_g and a second product for the min term on
// every group (512 positions, us): SwiGLU 2 x 14336 x 4096 364 -> 226, 4096 x
// 14336 194 -> 142, Q6 225 -> 167; the same sums, the same bits. Two blocks of
// rows a wave: 223 and 259. 8 waves a workgroup, three buffers and the weights
// two superblocks ahead: 258 and 157.
//
// Tiles are numbered so that consecutive ones share their weight rows and sit
// on one XCD (workgroup i runs on XCD i mod 8).
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
#define PS_STAGE(P) ((P) * 16 * (256 + 32 + 4))        // codes, group sums in fp16, scale of 16 P positions: two in LDS

// 16 bytes a lane from base + off straight into LDS, the wave's 64 lanes side
// by side from dst (a wave-uniform address) on. Written out because the
// compiler, which cannot tell the buffers apart, otherwise waits for every copy
// in flight before the next LDS read; the caller waits (vmcnt) and then meets
// the other waves before any of the bytes is read. (Loads that the compiler
// counts itself only ever wait longer for the copies it does not.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"             // m0 among the clobbers: it is what the statement sets
__device__ __forceinline__ void copy_lds16(const void * base, uint32_t off, const void * dst) {
    const uint32_t at = (uint32_t) (uintptr_t) (const __attribute__((address_space(3))) void *) dst;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(__builtin_amdgcn_readfirstlane(at)), "v"(off), "s"(base) : "m0", "memory");
}
#pragma clang diagnostic pop

template <int NB, bool SW, int P>
__device__ void ps_body(const sml_kgemm & a) {
    constexpr int NP = 16 * P;
    extern __shared__ __align__(16) uint8_t lds[];
    const int n = a.cols, ng = n / 32, nsb = n / 256, m_all = a.m_all, rows = a.rows;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, i16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int NW = 4;                               // waves
    constexpr int RT = SW ? 8 * NW : 16 * NW;
    const int nrt = (rows + RT - 1) / RT, npt = (m_all + NP - 1) / NP, total = nrt * npt;
    const int id = blockIdx.x, xcd = id & 7, slot = id >> 3, q8 = total >> 3, rem = total & 7;
    const int lid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + slot;
    const int rt = lid / npt, r0 = rt * RT, p0 = (lid - rt * npt) * NP;

    // this wave's 16 weight rows (SwiGLU: waves 0 and 1 of gate, 2 and 3 the same of up)
    constexpr int NIB = NB == 6 ? 1 : 0;
    const bool up = SW && wave >= NW / 2;
    const int grow = r0 + 16 * (SW ? wave & (NW / 2 - 1) : wave) + i16;
    const sml_kmat & m = up ? a.m0[SW ? 1 : 0] : a.m0[0];
    const size_t wr = (size_t) min(grow, rows - 1);
    const uint8_t * wn = m.plane[NIB] + wr * (size_t) (n / 2) + 16 * kq;
    const uint8_t * wh = m.plane[0] + wr * (size_t) (n / 4) + 16 * (kq & 1);
    const uint8_t * fqb = m.sqmq + wr * (size_t) ng * 2;
    const uint8_t * fdb = (const uint8_t *) m.sdmd + wr * (size_t) nsb * 4;
    struct {
        v4u w[2], h[2];             // the row's nibble words kq, kq + 4; Q6: its halves of the two 2-bit packs
        uint32_t sq[2];             // (sq, mq) of groups 2 (kq/2), +1 and 4 + 2 (kq/2), +1
        v2u mq;                     // (sq, mq) of groups 4 (kq%2)..+3
        uint32_t fd;                // (sd, md)
    } raw;
    auto fetch_w = [&](int b) {
        #pragma unroll
        for (int p = 0; p < 2; p++) {
            raw.w[p] = gld<v4u>(wn + (size_t) b * 128 + 64 * p);
            if constexpr (NB == 6) raw.h[p] = gld<v4u>(wh + (size_t) b * 64 + 32 * p);
            raw.sq[p] = gld<uint32_t>(fqb + (size_t) b * 16 + 8 * p + 4 * (kq >> 1));
        }
        raw.mq = gld<v2u>(fqb + (size_t) b * 16 + 8 * (kq & 1));
        raw.fd = gld<uint32_t>(fdb + (size_t) b * 4);
    };
    // the positions: wave w copies rows 4 (8 i + w)..+3 of the tile, a lane 16
    // bytes; positions past the end read the last one
    constexpr int NC = 4 * P / NW;
    uint32_t aoff[NC];
    #pragma unroll
    for (int i = 0; i < NC; i++) {
        const int pr = 4 * (NW * i + wave) + (lane >> 4);
        aoff[i] = (uint32_t) min(p0 + pr, m_all - 1) * (uint32_t) n + 16u * (uint32_t) ((lane & 15) ^ (pr & 15));
    }
    auto fetch_a = [&](int b) {
        uint8_t * base = lds + (size_t) (b & 1) * PS_STAGE(P) + wave * 1024;
        #pragma unroll
        for (int i = 0; i < NC; i++) copy_lds16(a.q, aoff[i] + 256u * (uint32_t) b, base + i * (NW * 1024));
    };
    // the positions' group sums and scales: thread t takes 4 groups (t%2) of
    // position t/2
    const int sp = tid >> 1, sh = tid & 1;
    const bool sums = tid < 2 * NP;
    const size_t soff = (size_t) min(p0 + (sums ? sp : 0), m_all - 1) * ng + 4 * sh;
    int4 su = make_int4(0, 0, 0, 0);
    float ss = 0.0f;
    auto fetch_s = [&](int b) {
        if (sums) { su = gld<int4>(a.sums + soff + 8 * b); ss = gld<float>(a.scale + soff + 8 * b); }
    };
    auto stage_s = [&](int b) {
        if (!sums) return;
        uint8_t * base = lds + (size_t) (b & 1) * PS_STAGE(P) + NP * 256;
        const int sv[4] = {su.x, su.y, su.z, su.w};
        v4h lo, hi;
        #pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = (_Float16) (float) (sv[i] & 63);
            hi[i] = (_Float16) (float) (sv[i] & ~63);
        }
        *(v4h *) (base + sp * 32 + 8 * sh) = lo;
        *(v4h *) (base + sp * 32 + 16 + 8 * sh) = hi;
        if (sh == 0) *(float *) (base + NP * 32 + sp * 4) = ss;
    };
    int ao[4];                                          // the lane's words of 64 columns s in its position's row
    #pragma unroll
    for (int s = 0; s < 4; s++) ao[s] = i16 * 256 + 16 * ((8 * (s >> 1) + 4 * (kq >> 1) + 2 * (s & 1) + (kq & 1)) ^ i16);

    float acc[P][4];
    #pragma unroll
    for (int u = 0; u < P; u++)
        #pragma unroll
        for (int r = 0; r < 4; r++) acc[u][r] = 0.0f;

    auto step = [&](int b) {
        // hi and lo of the wave's rows
        v4i hi[4], lo[4];
        v4h bm;
        #pragma unroll
        for (int s = 0; s < 4; s++) {
            typedef unsigned short v2s __attribute__((ext_vector_type(2)));
            const unsigned sq = (raw.sq[s >> 1] >> (16 * (s & 1))) & 0xFFu;
            const v2s m2 = __builtin_bit_cast(v2s, sq | sq << 16), k2 = {0x80, 0x80};
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                const unsigned w = raw.w[s >> 1][e] >> (4 * (s & 1));
                unsigned c0 = w & 0x000F000Fu, c1 = (w >> 8) & 0x000F000Fu;      // columns 0, 2 and 1, 3
                if constexpr (NB == 6) {
                    const unsigned h = raw.h[s >> 1][e] >> (4 * (kq >> 1) + 2 * (s & 1));
                    c0 |= (h & 0x00030003u) << 4;
                    c1 |= ((h >> 8) & 0x00030003u) << 4;
                }
                const unsigned u0 = __builtin_bit_cast(unsigned, (v2s) (__builtin_bit_cast(v2s, c0) * m2 + k2));
                const unsigned u1 = __builtin_bit_cast(unsigned, (v2s) (__builtin_bit_cast(v2s, c1) * m2 + k2));
                hi[s][e] = (int) __builtin_amdgcn_perm(u1, u0, 0x07030501u);
                lo[s][e] = (int) (__builtin_amdgcn_perm(u1, u0, 0x06020400u) ^ 0x80808080u);
            }
        }
        #pragma unroll
        for (int i = 0; i < 4; i++)
            bm[i] = (_Float16) (float) ((int) ((raw.mq[i >> 1] >> (16 * (i & 1) + 8)) & 0xFFu) - 127);
        const float dsc = h2f((uint16_t) (raw.fd & 0xFFFFu)), mdsc = h2f((uint16_t) (raw.fd >> 16));
        const bool more = b + 1 < nsb;
        if (more) {
            fetch_a(b + 1);
            fetch_s(b + 1);
            fetch_w(b + 1);
        }
        const uint8_t * base = lds + (size_t) (b & 1) * PS_STAGE(P);
        // two position tiles at a time, the hi and the lo sums apart: four
        // independent chains of MFMAs (a chain's next product waits for its
        // last); the next pair's operands are read during this one's epilogue
        v4i av[2][4];
        v4h as[2];
        float4 s4[2];
        auto operands = [&](int u0) {
            #pragma unroll
            for (int k = 0; k < 2; k++) {
                const int u = u0 + k;
                #pragma unroll
                for (int s = 0; s < 4; s++) av[k][s] = *(const v4i *) (base + u * 4096 + ao[s]);
                as[k] = *(const v4h *) (base + NP * 256 + (16 * u + i16) * 32 + 8 * kq);
                s4[k] = *(const float4 *) (base + NP * 288 + (16 * u + 4 * kq) * 4);
            }
        };
        operands(0);
        #pragma unroll
        for (int u0 = 0; u0 < P; u0 += 2) {
            const float sv[2][4] = {{s4[0].x, s4[0].y, s4[0].z, s4[0].w}, {s4[1].x, s4[1].y, s4[1].z, s4[1].w}};
            v4i h[2], l[2];
            v4f im[2];
            #pragma unroll
            for (int s = 0; s < 4; s++)
                #pragma unroll
                for (int k = 0; k < 2; k++) {
                    h[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[k][s], hi[s], s ? h[k] : v4i{0, 0, 0, 0}, 0, 0, 0);
                    l[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[k][s], lo[s], s ? l[k] : v4i{0, 0, 0, 0}, 0, 0, 0);
                }
            #pragma unroll
            for (int k = 0; k < 2; k++)
                im[k] = __builtin_amdgcn_mfma_f32_16x16x16f16(as[k], bm, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            if (u0 + 2 < P) operands(u0 + 2);
            #pragma unroll
            for (int k = 0; k < 2; k++) {
                float (&o)[4] = acc[u0 + k];
                #pragma unroll
                for (int r = 0; r < 4; r++) {
                    o[r] += (float) ((h[k][r] << 8) + l[k][r]) * (dsc * sv[k][r]);
                    o[r] += im[k][r] * (mdsc * sv[k][r]);
                }
                // (an empty statement on the sums so far: left free, the
                // products of every tile are held in registers at once)
                asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
            }
        }
        if (more) stage_s(b + 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the next superblock's rows are in LDS
        __syncthreads();
    };
    fetch_a(0);
    fetch_s(0);
    fetch_w(0);
    stage_s(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int b = 0; b < nsb; b++) step(b);

    if constexpr (SW) {
        // the up waves hand their sums to the gate waves through LDS
        float4 * x = (float4 *) lds + (wave & (NW / 2 - 1)) * P * 64 + lane;
        if (up) {
            #pragma unroll
            for (int u = 0; u < P; u++) x[u * 64] = make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
        }
        __syncthreads();
        if (up) return;
        #pragma unroll
        for (int u = 0; u < P; u++) {
            const float4 v = x[u * 64];
            acc[u][0] = silu_ref(acc[u][0]) * v.x;                                   // sml/sml-run.c:416-426
            acc[u][1] = silu_ref(acc[u][1]) * v.y;
            acc[u][2] = silu_ref(acc[u][2]) * v.z;
            acc[u][3] = silu_ref(acc[u][3]) * v.w;
        }
    }
    if (grow >= rows) return;
    #pragma unroll
    for (int u = 0; u < P; u++)
        #pragma unroll
        for (int r = 0; r < 4; r++) {
            const int pos = p0 + 16 * u + 4 * kq + r;
            if (pos >= m_all) continue;
            float v = acc[u][r];
            if (!SW && a.bias) v += a.bias[grow];
            if (!SW && a.resid) v = a.resid[(size_t) pos * rows + grow] + v;
            a.y[(size_t) pos * rows + grow] = v;
        }
}

#define PS_KERNEL(NB, P)                                                                                              \
    extern "C" __global__ __launch_bounds__(256, 2) void sml_pp_sgemm_q##NB##_p##P(const sml_kgemm a) { ps_body<NB, false, P>(a); } \
    extern "C" __global__ __launch_bounds__(256, 2) void sml_pp_sgemm_q##NB##_s_p##P(const sml_kgemm a) { ps_body<NB, true, P>(a); }
PS_KERNEL(4, 2) PS_KERNEL(4, 4) PS_KERNEL(4, 6) PS_KERNEL(4, 8)
PS_KERNEL(6, 2) PS_KERNEL(6, 4) PS_KERNEL(6, 6) PS_KERNEL(6, 8)

// ---------------------------------------------------------------- prompt attention on MFMA (flash form)
//
// For prompt reading at level 2 (and the attention entry point): the entries
// of a launch are consecutive positions of one sequence whose K and V rows
// sml_ropekv has already rotated and written to the cache (fp16). The
// (entry, query head) pairs of a kv head are its rows, whatever the heads a
// kv head serves: a workgroup takes 128 of them, 16 a wave, and walks the KV
// positions of its split in blocks of 64 with an online softmax, on
// v_mfma_f32_16x16x32_f16 (lane l: A row / B column l%16, k = 8(l/16)..+7; D
// rows 4(l/16)..+3 of column l%16):
//  - S^T = K Q^T: A = the block's K rows, B = the wave's rotated q (as rope8
//    rotates it) as two fp16 parts, q_hi = fp16(q) and q_lo = fp16(q - q_hi),
//    so the scores carry q to ~2^-22; a lane then holds row l%16 at KV
//    positions 4(l/16)..+3 of each 16-position tile;
//  - the softmax in base 2 and fp32, masked past each entry's position, its
//    first block as one over that block alone (a prompt of up to 64 positions
//    sums in the order of the plain online form);
//  - O += P V: A = P straight from the S^T layout (the MFMA's k slots
//    8(l/16)..+7 hold KV rows 4(l/16)..+3 of two 16-position tiles), as fp16
//    high and low parts like q (P rounded once to fp16, against a sum of the
//    unrounded P, moved a MoE prompt enough to flip a routed expert), B = V
//    by transposing LDS reads (ds_read_b64_tr_b16: 16 lanes read 4 rows of
//    16 dims and take a dim's 4 rows each), the same slot order.
// K and V go from memory to LDS without registers, a block ahead, 16-byte
// words swizzled by row so that both kinds of read touch every bank once; 4
// waves per SIMD (two workgroups per CU). What bounds it: matrix and vector
// instructions of the same waves (64 MFMA of 16 clocks and ~220 others a
// block), about half of the time each. 509 rows at 1531, 32 heads over 8:
// 42 us, 124 with a wave per head, V transposed by 2-byte LDS writes (8 to
// a bank) and 2 waves per SIMD; 16 rows to a wave 42 against 45 for 32 (half
// the LDS reads, half the waves).
// One split: the output is written directly; several: partials of sml_attn's
// layout, merged by sml_pp_merge. fp32 accumulation in its own order: graded
// as level-2 prompt reading is.
typedef short v4s __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
#define PF_KB 64                                        // KV positions a block
#define PF_STAGE (2 * PF_KB * 256)                      // its K rows, then its V rows

__device__ void pf_body(const sml_kattn & a) {
    constexpr int W = 8, HD = 128, RW = 16;                            // rows (query, head) of a wave
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, i16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = blockIdx.x, rep = a.n_head / a.n_kv, nrow = a.nseq * rep;
    const int rb = (int) (gridDim.y - 1 - blockIdx.y) * W * RW, rw = rb + wave * RW;
    const int kvd = a.n_kv * HD, half = HD / 2;
    auto entry = [&](int row) { return min(row, nrow - 1) / rep; };
    auto at = [&](int b) { return a.pos ? a.pos[b] : a.pos0 + b; };
    // this split's KV range, cut at the workgroup's last position, and the wave's end in it
    const int t_lo = blockIdx.z * a.fchunk, t_end = min(t_lo + a.fchunk, at(entry(rb + W * RW - 1)) + 1);
    const int w_end = rw < nrow ? min(t_end, at(entry(rw + RW - 1)) + 1) : 0;
    const size_t sl_off = a.kc_slots ? a.layer_off : 0;
    const uint16_t * kc = (a.kc_slots ? a.kc_slots[a.slot[entry(rb)]] : a.kcache) + sl_off + (size_t) kh * HD;
    const uint16_t * vc = (a.vc_slots ? a.vc_slots[a.slot[entry(rb)]] : a.vcache) + sl_off + (size_t) kh * HD;

    // the rotated q of row i16, dims 32c + 8g + e, as fp16 B operands (hi, lo)
    const float sl = a.inv * 1.44269504088896341f;
    v8h qb[4], ql[4];
    int posq;
    {
        const int row = min(rw + i16, nrow - 1), b = row / rep, h = kh * rep + (row - b * rep);
        posq = at(b);
        const float * qp = a.q + (size_t) b * a.qkv_stride + (size_t) h * HD + 8 * g;
        float x[4][8];
        #pragma unroll
        for (int c = 0; c < 4; c++)
            #pragma unroll
            for (int e = 0; e < 8; e += 4) *(float4 *) &x[c][e] = *(const float4 *) (qp + 32 * c + e);
        #pragma unroll
        for (int c = 0; c < 2; c++) {
            float cs[8], sn[8];
            #pragma unroll
            for (int e = 0; e < 8; e += 4) {
                *(float4 *) &cs[e] = *(const float4 *) (a.cos_t + (size_t) posq * half + 32 * c + 8 * g + e);
                *(float4 *) &sn[e] = *(const float4 *) (a.sin_t + (size_t) posq * half + 32 * c + 8 * g + e);
            }
            #pragma unroll
            for (int e = 0; e < 8; e++) {
                const float lo = x[c][e], hi = x[c + 2][e];
                x[c][e] = __builtin_fmaf(lo, cs[e], -(hi * sn[e]));              // sml/sml-run.c:363-368, fused as its build does
                x[c + 2][e] = __builtin_fmaf(lo, sn[e], hi * cs[e]);
            }
        }
        #pragma unroll
        for (int c = 0; c < 4; c++)
            #pragma unroll
            for (int e = 0; e < 8; e++) {
                qb[c][e] = (_Float16) x[c][e];
                ql[c][e] = (_Float16) (x[c][e] - (float) qb[c][e]);
            }
    }
    float m_run = -INFINITY;                            // of row i16 (the same in its 4 lanes)
    float l_run = 0.0f;                                 // the lane's positions' share of its sum
    v4f o[8];
    #pragma unroll
    for (int dt = 0; dt < 8; dt++) o[dt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // a block's rows into LDS: 16-byte word w of row r at place w ^ 2(r & 7);
    // rows past the range repeat its first
    auto fetch = [&](int buf, int t0) {
        uint8_t * st = lds + buf * PF_STAGE;
        const uint16_t * kb = kc + (size_t) t0 * kvd, * vb = vc + (size_t) t0 * kvd;
        #pragma unroll
        for (int i = 0; i < 16 / W; i++) {
            const int r = 4 * (W * i + wave) + g;
            const uint32_t off = (uint32_t) (t0 + r < t_end ? r : 0) * (uint32_t) (kvd * 2) + 16u * (uint32_t) (i16 ^ (2 * (r & 7)));
            copy_lds16(kb, off, st + 4 * (W * i + wave) * 256);
            copy_lds16(vb, off, st + PF_KB * 256 + 4 * (W * i + wave) * 256);
        }
    };
    const int krow = i16 * 256, kx = 2 * (i16 & 7);     // K row i16 of a tile
    const int vrow = 4 * g + (i16 >> 2), vx = vrow & 7; // the V row this lane reads for its 16 lanes
    const int vat = PF_KB * 256 + vrow * 256 + 8 * (i16 & 3);

    auto compute = [&](int buf, int t0) {
        const uint8_t * st = lds + buf * PF_STAGE;
        // S^T: 4 tiles of 16 positions x 16 rows
        v4f s[4];
        #pragma unroll
        for (int j = 0; j < 4; j++) {
            s[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            #pragma unroll
            for (int c = 0; c < 4; c++) {
                const v8h ka = *(const v8h *) (st + 16 * j * 256 + krow + 16 * ((4 * c + g) ^ kx));
                s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[c], s[j], 0, 0, 0);
                s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, ql[c], s[j], 0, 0, 0);
            }
        }
        v8h pa[2], pl[2];
        // mask (the blocks that reach past a row's position) and the block's max for the lane's row
        const int lim = min(posq, t_end - 1) - t0 - 4 * g;
        float mx = -INFINITY;
        #pragma unroll
        for (int j = 0; j < 4; j++)
            #pragma unroll
            for (int r = 0; r < 4; r++) {
                s[j][r] = 16 * j + r <= lim ? s[j][r] * sl : -INFINITY;
                mx = fmaxf(mx, s[j][r]);
            }
        // the base of the weights is the first max and moves only when a
        // later one passes it by 15 (weights up to 2^15, within fp16's
        // range): most blocks need no reduction over the row's lanes
        if (__any(mx > m_run + 15.0f)) {
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = mx > m_run + 15.0f ? mx : m_run;
            // rescale O (its rows are 4g..4g+3)
            const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
            l_run *= alpha;
            float al[4];
            #pragma unroll
            for (int r = 0; r < 4; r++) al[r] = __shfl(alpha, 4 * g + r);
            #pragma unroll
            for (int dt = 0; dt < 8; dt++)
                #pragma unroll
                for (int r = 0; r < 4; r++) o[dt][r] *= al[r];
            m_run = m_new;
        }
        const float mu = m_run == -INFINITY ? 0.0f : m_run;   // no position yet: keep zeros
        float ls = 0.0f;
        #pragma unroll
        for (int j = 0; j < 4; j++)
            #pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const float p0 = __builtin_amdgcn_exp2f(s[j][r] - mu), p1 = __builtin_amdgcn_exp2f(s[j][r + 1] - mu);
                ls += p0;
                ls += p1;
                const v2h ph = {(_Float16) p0, (_Float16) p1};
                float r0, r1;                             // p - hi, exact
                asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(ph), "v"(p0));
                asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(ph), "v"(p1));
                const v2h pr = {(_Float16) r0, (_Float16) r1};
                pa[j >> 1][4 * (j & 1) + r] = ph[0];
                pa[j >> 1][4 * (j & 1) + r + 1] = ph[1];
                pl[j >> 1][4 * (j & 1) + r] = pr[0];
                pl[j >> 1][4 * (j & 1) + r + 1] = pr[1];
            }
        l_run += ls;
        // O += P V: per 32 positions k, slots 8g..8g+3 are rows 4g..4g+3 of
        // tile 2k, 8g+4..8g+7 those of tile 2k+1
        #pragma unroll
        for (int dt = 0; dt < 8; dt++) {
            const uint8_t * vr = st + vat + ((dt ^ vx) << 5);
            #pragma unroll
            for (int k = 0; k < 2; k++) {
                typedef __attribute__((address_space(3))) v4s lv4s;
                const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lv4s *) (vr + 32 * k * 256));
                const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lv4s *) (vr + (32 * k + 16) * 256));
                const v8h w = __builtin_bit_cast(v8h, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[k], w, o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl[k], w, o[dt], 0, 0, 0);
            }
        }
    };

    if (t_lo < t_end) {
        fetch(0, t_lo);
        int buf = 0;
        for (int t0 = t_lo; t0 < t_end; t0 += PF_KB, buf ^= 1) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this block's rows are in LDS
            __syncthreads();
            if (t0 + PF_KB < t_end) fetch(buf ^ 1, t0 + PF_KB);  // past the barrier: nobody reads the last block
            if (t0 < w_end) compute(buf, t0);
        }
    }

    // the lane's rows: 4g..4g+3 of each tile, dims 16dt + i16
    const bool one = gridDim.z == 1;
    l_run += __shfl_xor(l_run, 16);
    l_run += __shfl_xor(l_run, 32);
    #pragma unroll
    for (int r = 0; r < 4; r++) {
        const float lq = __shfl(l_run, 4 * g + r), mq = __shfl(m_run, 4 * g + r);
        const int row = rw + 4 * g + r;
        if (row >= nrow) continue;
        const int b = row / rep, h = kh * rep + (row - b * rep);
        if (one) {
            float * out = a.out + (size_t) b * a.n_head * HD + (size_t) h * HD;
            #pragma unroll
            for (int dt = 0; dt < 8; dt++) out[16 * dt + i16] = o[dt][r] / lq;
        } else {
            float * blk = a.part + (size_t) b * a.n_head * a.nsplit * (HD + 2);
            float * po = blk + ((size_t) h * a.nsplit + blockIdx.z) * HD;
            float2 * pml = (float2 *) (blk + (size_t) a.n_head * a.nsplit * HD) + (size_t) h * a.nsplit + blockIdx.z;
            #pragma unroll
            for (int dt = 0; dt < 8; dt++) po[16 * dt + i16] = o[dt][r];
            if (i16 == 0) *pml = make_float2(mq, lq);
        }
    }
}

extern "C" __global__ __launch_bounds__(512, 4) void sml_pp_flash(const sml_kattn a) { pf_body(a); }

// The splits of sml_pp_flash merged: 32 lanes a (row, head), four dims a lane,
// the splits in order. A launch per head and row as the decode merge makes
// is bound by its workgroups' start and one serial chain of loads: 509 rows
// of 32 heads, 4 splits, 15.6 us there and 7.3 here.
extern "C" __global__ __launch_bounds__(256) void sml_pp_merge(const sml_kattn a) {
    const int idx = blockIdx.x * 8 + (threadIdx.x >> 5), l = threadIdx.x & 31, ns = a.nsplit;
    if (idx >= a.nseq * a.n_head) return;
    const int b = idx / a.n_head, h = idx - b * a.n_head;
    const float * blk = a.part + (size_t) b * a.n_head * ns * 130;
    const float4_a4 * po = (const float4_a4 *) (blk + (size_t) h * ns * 128) + l;   // 8-byte aligned: odd splits of odd heads
    const float2 * pml = (const float2 *) (blk + (size_t) a.n_head * ns * 128) + (size_t) h * ns;
    float M = -INFINITY;
    for (int s = l; s < ns; s += 32) M = fmaxf(M, pml[s].x);
    M = max32(M);                                             // finite: a row's first split is active
    float L = 0.0f;
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    #pragma unroll 4
    for (int s = 0; s < ns; s++) {
        const float2 ml = pml[s];
        const float4_a4 v = po[s * 32];
        const float e = __builtin_amdgcn_exp2f(ml.x - M);     // 0 for splits past the position
        L += e * ml.y;
        o.x += e * v.x; o.y += e * v.y; o.z += e * v.z; o.w += e * v.w;
    }
    *((float4_a4 *) (a.out + (size_t) idx * 128) + l) = {o.x / L, o.y / L, o.z / L, o.w / L};
}

// ---------------------------------------------------------------- normalization + quantization of many rows
//
// sml_normq2's codes, scales and sums bit for bit (its sum of squares order,
// its formulas), a workgroup a row. There each of a row's n/256 workgroups
// reads the whole row for the norm, and every value comes by its own gather
// from memory; here the row is read once, normalized into LDS, and each
// output gathers from there four columns a lane (a group of 32 is 8 lanes, a
// superblock one wave).
// 512 x 4096 with its norm: 9.1 us, 18.6 there (mean over a layer's four).
extern "C" __global__ __launch_bounds__(256) void sml_pp_normq(const sml_knormq2 a) {
    extern __shared__ __align__(16) float y[];                // [n]
    __shared__ double red[4];
    const int n = a.n, tid = threadIdx.x;
    const size_t bo = (size_t) blockIdx.x * n, bg = (size_t) blockIdx.x * (n / 32);
    const float * x = a.x + bo;
    if (a.norm_w) {
        double ss = 0.0;
        #pragma unroll 4
        for (int i = tid * 4; i < n; i += 1024) {
            const float4 v = *(const float4 *) (x + i);
            *(float4 *) (y + i) = v;
            ss = ss_add4(ss, v);
        }
        #pragma unroll
        for (int o = 32; o; o >>= 1) ss += __shfl_xor(ss, o);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        const double tot = red[0] + red[1] + red[2] + red[3];
        float msq = (float) (tot / (double) n);
        if (a.exact && !ss_mean_alike(tot, n, msq)) {
            // the serial chain (the same decision in every thread)
            __syncthreads();
            if (tid == 0) red[0] = serial_ss(x, n);
            __syncthreads();
            msq = (float) (red[0] / (double) n);
        }
        const float sc = 1.0f / sqrtf(msq + a.eps);
        #pragma unroll 4
        for (int i = tid * 4; i < n; i += 1024) {             // the thread's own words
            float4 v = *(const float4 *) (y + i);
            const float4_a4 w = *(const float4_a4 *) (a.norm_w + i);
            v.x = v.x * sc * w.x; v.y = v.y * sc * w.y; v.z = v.z * sc * w.z; v.w = v.w * sc * w.w;
            *(float4 *) (y + i) = v;
        }
    } else {
        #pragma unroll 4
        for (int i = tid * 4; i < n; i += 1024) *(float4 *) (y + i) = *(const float4 *) (x + i);
    }
    __syncthreads();
    for (int o = 0; o < a.nout; o++) {
        const int32_t * perm = a.perm[o];
        #pragma unroll 4
        for (int j0 = 0; j0 < n; j0 += 1024) {
            const int j = j0 + 4 * tid;
            const bool ok = j < n;                            // whole groups of 32
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (ok) {
                if (perm) {
                    const int4_a4 p = *(const int4_a4 *) (perm + j);
                    v[0] = y[p.x]; v[1] = y[p.y]; v[2] = y[p.z]; v[3] = y[p.w];
                } else {
                    *(float4 *) v = *(const float4 *) (y + j);
                }
            }
            const float m4 = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
            const float amax = a.per256 ? wave_max(m4) : max8(m4);
            const float s = amax / 127.0f;
            const float is = s > 0.0f ? 1.0f / s : 0.0f;
            uint32_t w = 0;
            int t4 = 0;
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = quant1(v[e], is);
                t4 += t;
                w |= (uint32_t) (t & 0xFF) << (8 * e);
            }
            const int sum = isum8(t4);
            if (!ok) continue;
            *(uint32_t *) (a.q[o] + bo + j) = w;
            if ((tid & 7) == 0) { a.scale[o][bg + (j >> 5)] = s; a.sums[o][bg + (j >> 5)] = sum; }
        }
    }
}

// ---------------------------------------------------------------- prompt attention in decoding's float order
//
// For prompts read at level 1, whose attention equals decoding's bit for bit.
// Decoding spreads a position's 128 dims over 16 lanes and a split's positions
// over 8 waves of 4 such rows; the values it computes are, per (entry, query
// head, split): a score as 16 chains of 8 FMAs and their balanced tree; per
// wave w (positions 4w..4w+3 of every 32) the max, the weights in base 2 and
// their sum, each row's chain over the 32s and the tree over the 4 rows, for
// the weights and for P V; then a chain over the waves. Here a wave takes a
// whole entry and computes just these: the scores with a lane per position
// (the chains and the tree in registers: no cross-lane adds), the 8 softmaxes
// at once, 8 lanes each, P V with two dims a lane and the weights from LDS by
// broadcast. K and V are staged once per 16 entries, straight to LDS (K's
// 16-byte words swizzled by position); q comes rotated (sml_pp_ropeq, in
// place) by scalar loads, and the FMAs take fp16 K and V as they are
// (v_fma_mix). No barrier past the staging.
// Bound by VALU issue (256 FMAs a position and head, 1.4 instructions each):
// 512 rows at 509, 32 heads over 8: 226 us + 5.5, 620 with a 16-lane row per
// position (cross-lane sums, q rotated by every row, two barriers an entry).
extern "C" __global__ __launch_bounds__(256) void sml_pp_ropeq(const sml_kattn a) {
    const int t = blockIdx.x * 256 + threadIdx.x;             // 4 dims of a row's first halves
    const int per = a.n_head * 16, b = t / per;
    if (b >= a.nseq) return;
    const int h = (t - b * per) >> 4, d = 4 * (t & 15), pos = a.pos[b];
    float * q = (float *) a.q + (size_t) b * a.qkv_stride + (size_t) h * 128 + d;
    const float4 lo = *(const float4 *) q, hi = *(const float4 *) (q + 64);
    const float4 c = *(const float4 *) (a.cos_t + (size_t) pos * 64 + d), s = *(const float4 *) (a.sin_t + (size_t) pos * 64 + d);
    *(float4 *) q = make_float4(__builtin_fmaf(lo.x, c.x, -(hi.x * s.x)), __builtin_fmaf(lo.y, c.y, -(hi.y * s.y)),
                                __builtin_fmaf(lo.z, c.z, -(hi.z * s.z)), __builtin_fmaf(lo.w, c.w, -(hi.w * s.w)));
    *(float4 *) (q + 64) = make_float4(__builtin_fmaf(lo.x, s.x, hi.x * c.x), __builtin_fmaf(lo.y, s.y, hi.y * c.y),
                                       __builtin_fmaf(lo.z, s.z, hi.z * c.z), __builtin_fmaf(lo.w, s.w, hi.w * c.w));
}

__device__ __forceinline__ float lane_val(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

template <int REP, int NL>
__device__ void pa_body(const sml_kattn & a) {
    constexpr int HD = 128, CH = 64 * NL, W = 8;
    constexpr int NG = (REP + 3) / 4, RG = (REP + NG - 1) / NG;     // heads in groups of up to 4
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t * lk = lds, * lv = lds + CH * 256;
    float * lp = (float *) (lds + 2 * CH * 256) + wave * RG * CH;
    const int kh = blockIdx.y, split = blockIdx.x, kvd = a.n_kv * HD, ns = a.nsplit;
    const int b0 = blockIdx.z * a.tpw, b1 = min(b0 + a.tpw, a.nseq);
    const int t0 = split * CH, tl = min(a.pos[b1 - 1] + 1, t0 + CH);
    const float sl = a.inv * 1.44269504088896341f;
    if (t0 < tl) {
        const size_t at = (size_t) t0 * kvd + (size_t) kh * HD;
        const uint16_t * kc = (a.kc_slots ? a.kc_slots[a.slot[b0]] + a.layer_off : a.kcache) + at;
        const uint16_t * vc = (a.vc_slots ? a.vc_slots[a.slot[b0]] + a.layer_off : a.vcache) + at;
        #pragma unroll
        for (int i = 0; i < CH / (4 * W); i++) {
            const int r0 = 4 * (W * i + wave), r = r0 + (lane >> 4), w = lane & 15;
            const uint32_t row = (uint32_t) (t0 + r < tl ? r : 0) * (uint32_t) (kvd * 2);
            copy_lds16(kc, row + 16u * (uint32_t) (w ^ (r & 15)), lk + r0 * 256);
            copy_lds16(vc, row + 16u * (uint32_t) w, lv + r0 * 256);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    for (int b = b0 + wave; b < b1; b += W) {
        const int T = a.pos[b] + 1;
        float * blk = a.part + (size_t) b * a.n_head * ns * (HD + 2);
        float2 * pml = (float2 *) (blk + (size_t) a.n_head * ns * HD) + (size_t) kh * REP * ns + split;
        float * po = blk + ((size_t) kh * REP * ns + split) * HD + 2 * lane;
        if (t0 >= T) {
            if (lane < REP) pml[(size_t) lane * ns] = make_float2(-INFINITY, 0.0f);
            continue;
        }
        const int n = min(T - t0, CH);
        for (int g = 0; g < NG; g++) {
            const __attribute__((address_space(4))) float * q[RG];
            #pragma unroll
            for (int j = 0; j < RG; j++)
                q[j] = (const __attribute__((address_space(4))) float *) (a.q + (size_t) b * a.qkv_stride +
                                                                          (size_t) (kh * REP + min(g * RG + j, REP - 1)) * HD);
            // scores of positions lane, lane + 64: 16 chains of 8 and their tree
            float sc[RG][NL], st[3][RG][NL];
            #pragma unroll
            for (int l = 0; l < 16; l++) {
                v8h k[NL];
                #pragma unroll
                for (int u = 0; u < NL; u++) k[u] = *(const v8h *) (lk + (lane + 64 * u) * 256 + 16 * (l ^ (lane & 15)));
                #pragma unroll
                for (int j = 0; j < RG; j++)
                    #pragma unroll
                    for (int u = 0; u < NL; u++) {
                        float p = 0.0f;
                        #pragma unroll
                        for (int e = 0; e < 8; e++) p = __builtin_fmaf(q[j][8 * l + e], (float) k[u][e], p);
                        if (l & 1) p = st[0][j][u] + p;
                        if ((l & 3) == 3) p = st[1][j][u] + p;
                        if ((l & 7) == 7) p = st[2][j][u] + p;
                        if (l == 15) p = sc[j][u] + p;
                        if (!(l & 1)) st[0][j][u] = p;
                        else if ((l & 3) == 1) st[1][j][u] = p;
                        else if ((l & 7) == 3) st[2][j][u] = p;
                        else sc[j][u] = p;
                    }
            }
            // the softmax of each of decoding's 8 waves (wave w: positions 4w..4w+3
            // of every 32), 8 lanes each here
            float e[RG], lw[RG], L[RG], M[RG];
            #pragma unroll
            for (int j = 0; j < RG; j++) {
                float m = -INFINITY;
                #pragma unroll
                for (int u = 0; u < NL; u++) {
                    sc[j][u] = lane + 64 * u < n ? sc[j][u] * sl : -INFINITY;
                    m = fmaxf(m, sc[j][u]);
                }
                m = fmaxf(m, dpp_f<0xB1>(m));
                m = fmaxf(m, dpp_f<0x4E>(m));
                m = fmaxf(m, __shfl_xor(m, 32));
                const float mj = m == -INFINITY ? 0.0f : m;
                float ls = 0.0f;
                #pragma unroll
                for (int u = 0; u < NL; u++) {
                    const float p = __builtin_amdgcn_exp2f(sc[j][u] - mj), x = __shfl_xor(p, 32);
                    lp[j * CH + 64 * u + lane] = p;
                    ls += lane < 32 ? p : x;
                    ls += lane < 32 ? x : p;
                }
                ls = ls + dpp_f<0xB1>(ls);
                lw[j] = ls + dpp_f<0x4E>(ls);
                float x = fmaxf(m, dpp_f<0x141>(m));
                x = fmaxf(x, dpp_f<0x140>(x));
                M[j] = fmaxf(x, swz16_f(x));                  // finite: wave 0 holds t0
                e[j] = __builtin_amdgcn_exp2f(m - M[j]);
                L[j] = 0.0f;
            }
            // P V for dims 2 lane, 2 lane + 1: each wave's four chains over the
            // 32s, their sum, then the waves by their weights
            float o[RG][2];
            #pragma unroll
            for (int j = 0; j < RG; j++) o[j][0] = o[j][1] = 0.0f;
            #pragma unroll 1
            for (int w = 0; w < W; w++) {
                float acc[RG][4][2];
                #pragma unroll
                for (int j = 0; j < RG; j++)
                    #pragma unroll
                    for (int r = 0; r < 4; r++) acc[j][r][0] = acc[j][r][1] = 0.0f;
                #pragma unroll
                for (int i = 0; i < 2 * NL; i++) {
                    v2h v[4];
                    #pragma unroll
                    for (int r = 0; r < 4; r++) v[r] = *(const v2h *) (lv + (32 * i + 4 * w + r) * 256 + 4 * lane);
                    #pragma unroll
                    for (int j = 0; j < RG; j++) {
                        const float4 p = *(const float4 *) (lp + j * CH + 32 * i + 4 * w);
                        const float pr[4] = {p.x, p.y, p.z, p.w};
                        #pragma unroll
                        for (int r = 0; r < 4; r++) {
                            acc[j][r][0] = __builtin_fmaf(pr[r], (float) v[r][0], acc[j][r][0]);
                            acc[j][r][1] = __builtin_fmaf(pr[r], (float) v[r][1], acc[j][r][1]);
                        }
                    }
                }
                #pragma unroll
                for (int j = 0; j < RG; j++) {
                    const float ew = lane_val(e[j], 4 * w);
                    L[j] = __builtin_fmaf(ew, lane_val(lw[j], 4 * w), L[j]);
                    #pragma unroll
                    for (int d = 0; d < 2; d++)
                        o[j][d] = __builtin_fmaf(ew, (acc[j][0][d] + acc[j][1][d]) + (acc[j][2][d] + acc[j][3][d]), o[j][d]);
                }
            }
            #pragma unroll
            for (int j = 0; j < RG; j++) {
                const int h = g * RG + j;
                if (h >= REP) continue;
                *(float2 *) (po + (size_t) h * ns * HD) = make_float2(o[j][0], o[j][1]);
                if (lane == 0) pml[(size_t) h * ns] = make_float2(M[j], L[j]);
            }
        }
    }
}
#define PA_KERNEL(R)                                                                                                          \
    extern "C" __global__ __launch_bounds__(512, 4) void sml_pp_attn_r##R(const sml_kattn a) { pa_body<R, 2>(a); }            \
    extern "C" __global__ __launch_bounds__(512, 4) void sml_pp_attn_s64_r##R(const sml_kattn a) { pa_body<R, 1>(a); }
PA_KERNEL(1) PA_KERNEL(2) PA_KERNEL(3) PA_KERNEL(4) PA_KERNEL(5) PA_KERNEL(6) PA_KERNEL(7) PA_KERNEL(8)
