/* H-TILE linear for every shape the aligned kernels do not take (gfx950): any M, N, K,
 * block size and pointer alignment, f32 or BF16 out.
 *
 * A row of the pin starts at element n K, which need not be a multiple of the block size, of
 * a byte's two nibbles or of a load's width, so a lane's weights are read from their own
 * (unaligned) byte address and shifted by a nibble where n K is odd, and each group of 32
 * weights carries the two block scales it can touch and where the second begins.
 *
 * Split: one workgroup per 16 NB rows of W and 16 MB rows of x; its 8 waves take contiguous
 * parts of K (128-wide chunks) and meet in LDS, in wave order, so a matrix of a few thousand
 * rows fills the CUs without a K split across workgroups, and no workspace is needed. As in
 * k_htile_rl, lane (m16, g) of a wave holds elements [32 g, +32) of a chunk of W row m16 and
 * of x row m16: word s of each is MFMA step s's operand (the K order inside a chunk is the
 * same for both). x comes straight from the caches: it is small beside the planes here.
 *
 * Arithmetic: the f32 weight w = CELLS * absmax as three exact BF16 planes (hi, mid, lo;
 * GlintTileProducer::finish_split's rule), each multiplied with x in the MFMA, f32 sums. The
 * products are exact, so y differs from the scalar sum of w x only by the order of its f32
 * additions, for BF16 out as for f32 out (a subnormal x is aligned by the matrix core as if it were
 * 2^-126: the sums are then exact to 2^-23 of sum |w| 2^-126). Where a scale is nonzero and below
 * 2^-90 (lo may then have bits BF16 cannot hold) or an output comes out infinite or NaN (an
 * infinite or NaN scale or x, where inf * 0 of a plane is not the product's value, or an
 * overflow), the workgroup forms its outputs again with one f32 FMA per weight in k order
 * (htile_any_again).
 *
 * Bound: the dequantization (about 9 VALU instructions and one LDS read per weight, once per
 * 16 MB rows of x) and the latency of a wave's 4 or 5 dependent chunks; the planes' bytes
 * would take 3 us at 17 x 3001 x 4104. Measured (f32 out unless noted, M x N x K, blocks of
 * 64, rotated pins) against a kernel of scalar f32 FMAs on 64 x 32 LDS tiles:
 *   1 x 3001 x 4104 bf16 643 -> 12.5 us, 17 x 3001 x 4104 693 -> 15.6, 1 x 4999 x 3001 534 -> 18.1,
 *   33 x 3001 x 4104 (blocks of 32) 788 -> 21.3, 64 x 3000 x 4104 (blocks of 16) 802 -> 38.8,
 *   130 x 5000 x 5000 1069 -> 64, 512 x 14336 x 4104 bf16 2160 -> 408, 5 x 256 x 256 35 -> 4.0.
 * Relative error against 64 bits 1.4e-7 to 2.7e-7, where the scalar sums had 1.1e-6. */
#ifndef GLINT_HTILE_ANY_H_
#define GLINT_HTILE_ANY_H_

#include "glint_common.h"
#include "tile_mfma.h"

#define ANY_KW 8 /* waves per workgroup = parts of K */
#define ANY_SCALE_LO 0x12800000u /* f32 bits of 2^-90 */

typedef glint_u32x4 glint_u32x4_b1 __attribute__((aligned(1)));
typedef glint_u32x4 glint_u32x4_b2 __attribute__((aligned(2)));

__device__ __forceinline__ uint32_t glint_nibble(const uint8_t *pk, int64_t i) {
    return (pk[i >> 1] >> ((uint32_t)(i & 1) * 4)) & 15u;
}

/* A workgroup's outputs v[j] (threadIdx.x + j T of the 16 NB x 16 MB tile) once more, by one f32
 * FMA per weight in k order, w = CELLS * absmax: 128 elements of K at a time, the tile's weights
 * and x as f32 through LDS (rows of 132 words: 16 rows' 16-byte reads lie in different banks), the
 * next 128 loaded meanwhile. A thread brings 8 elements of a row of W and of 16 MB / 32 rows of x,
 * read element by element where the row ends. Every thread of the workgroup calls it.
 * Bound: the f32 FMAs and their LDS reads (3 or 4 of 16 bytes for 4 NB NA FMAs). One NaN in x, all
 * scales 1e-35, against one thread per output walking K in global memory, and a kernel of scalar
 * f32 FMAs on 64 x 32 LDS tiles: 17 x 3001 x 4104 98, 98 us (1349, 1352; 630, 633),
 * 130 x 5000 x 5000 BF16 208, 410 (10420, 20700; 1070, 1070), 512 x 14336 x 4104 BF16 650, 2300
 * (16650, 113000; 2240, 2260). */
template <int MB, int NB>
__device__ __forceinline__ void htile_any_again(float *lds, const uint8_t *hole, const uint8_t *plug,
                                                const float *absmax, const uint16_t *x, int m0, int n0, int M, int N,
                                                int K, int bs,
                                                float (&v)[(NB * MB * 256 + 64 * ANY_KW - 1) / (64 * ANY_KW)]) {
    constexpr int T = 64 * ANY_KW, KC = 128, ROW = KC + 4, XJ = (16 * MB + 31) / 32, NA = MB > 1 ? MB / 2 : 1;
    static_assert(T == 512 && (MB == 1 || MB % 2 == 0), "the outputs of a thread are NB x NA of the tile's 16 x 16");
    static_assert((16 * NB + 16 * MB) * ROW + 256 <= GLINT_LDS_CELLS64_WORDS, "the tiles fit the table's LDS");
    float *ws = lds, *xs = ws + 16 * NB * ROW, *cells = xs + 16 * MB * ROW;
    const int tid = (int)threadIdx.x, row = tid >> 4, k8 = 8 * (tid & 15);
    const bool wact = row < 16 * NB;
    int64_t e = (int64_t)min(n0 + row, N - 1) * K + k8, q = e / bs; /* the thread's next weight, its block */
    uint32_t r = (uint32_t)(e - q * bs);                            /* and its place there */
    const int dq = KC / bs;
    const uint32_t dr = (uint32_t)(KC % bs);
    uint32_t h = 0, p = 0;
    float a[8];
    glint_u32x4 xw[XJ];
    auto load = [&](int k0) {
        const int kin = min(max(K - k0 - k8, 0), 8);
        const int nb = wact && kin > 0 ? (int)(((e + kin - 1) >> 1) - (e >> 1)) + 1 : 0; /* bytes: at most 5 */
        uint64_t hb = 0, pb = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i)
            if (i < nb) {
                hb |= (uint64_t)hole[(e >> 1) + i] << (8 * i);
                pb |= (uint64_t)plug[(e >> 1) + i] << (8 * i);
            }
        h = (uint32_t)(hb >> (4 * (e & 1)));
        p = (uint32_t)(pb >> (4 * (e & 1)));
        int64_t qi = q;
        uint32_t ri = r;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            a[i] = wact && i < kin ? absmax[qi] : 0.0f;
            if (++ri == (uint32_t)bs) {
                ri = 0;
                ++qi;
            }
        }
        e += KC;
        q += dq;
        r += dr;
        if (r >= (uint32_t)bs) {
            r -= (uint32_t)bs;
            ++q;
        }
#pragma unroll
        for (int j = 0; j < XJ; ++j) {
            const uint16_t *xp = x + (int64_t)min(m0 + row + 32 * j, M - 1) * K + k0 + k8;
            xw[j] = glint_u32x4{0u, 0u, 0u, 0u};
            if (row + 32 * j < 16 * MB && kin == 8)
                xw[j] = *(const glint_u32x4_b2 *)xp;
            else if (row + 32 * j < 16 * MB)
                for (int i = 0; i < kin; ++i)
                    xw[j][i >> 1] |= (uint32_t)xp[i] << (16 * (i & 1));
        }
    };
    auto put = [&](int k0) {
        const int kin = min(max(K - k0 - k8, 0), 8);
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) /* past K zeros, also under an infinite x: they change no sum */
            w[i] = i < kin ? cells[((h >> (4 * i)) & 15u) << 4 | ((p >> (4 * i)) & 15u)] * a[i] : 0.0f;
        if (wact) {
            *(glint_f32x4 *)(ws + row * ROW + k8) = glint_f32x4{w[0], w[1], w[2], w[3]};
            *(glint_f32x4 *)(ws + row * ROW + k8 + 4) = glint_f32x4{w[4], w[5], w[6], w[7]};
        }
#pragma unroll
        for (int j = 0; j < XJ; ++j)
            if (row + 32 * j < 16 * MB)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    *(glint_f32x4 *)(xs + (row + 32 * j) * ROW + k8 + 4 * i) =
                        glint_f32x4{glint_bf16lo(xw[j][2 * i]), glint_bf16hi(xw[j][2 * i]),
                                    glint_bf16lo(xw[j][2 * i + 1]), glint_bf16hi(xw[j][2 * i + 1])};
    };
    /* output j = jb NA + ja: W row 16 jb + tid % 16 and x row 16 (tid / 256 + 2 ja) + .. of the tile */
    const float *wr = ws + (tid & 15) * ROW, *xr = xs + (16 * (tid >> 8) + 4 * ((tid & 63) >> 4) + ((tid >> 6) & 3)) * ROW;
    const bool out = MB > 1 || tid < 256;
#pragma unroll
    for (int j = 0; j < NB * NA; ++j)
        v[j] = 0.0f;
    load(0);
    __syncthreads(); /* the outputs of the first way have been read */
    if (tid < 256)
        cells[tid] = (&kCells[0][0])[tid];
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += KC) {
        put(k0);
        __syncthreads();
        if (k0 + KC < K)
            load(k0 + KC);
        if (out)
#pragma unroll 4
            for (int k = 0; k < min(KC, K - k0); k += 4) {
                glint_f32x4 wv[NB], xv[NA];
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    wv[j] = *(const glint_f32x4 *)(wr + 16 * j * ROW + k);
#pragma unroll
                for (int j = 0; j < NA; ++j)
                    xv[j] = *(const glint_f32x4 *)(xr + 32 * j * ROW + k);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int j = 0; j < NB * NA; ++j)
                        v[j] = fmaf(wv[j / NA][c], xv[j % NA][c], v[j]);
            }
        __syncthreads();
    }
}

/* ODD: K is odd, so odd rows start in the middle of a byte. SB: bs < 32, more than two
 * blocks may meet in 32 elements: every weight's scale is its own load. */
template <int MB, int NB, bool ODD, bool SB, class Out>
__global__ __launch_bounds__(64 * ANY_KW) void k_htile_any(const uint8_t *__restrict__ hole,
                                                           const uint8_t *__restrict__ plug,
                                                           const float *__restrict__ absmax,
                                                           const uint16_t *__restrict__ x,
                                                           typename Out::T *__restrict__ y, int M, int N, int K,
                                                           int bs, int strip0) {
    constexpr int T = 64 * ANY_KW;
    constexpr int NA = MB * NB >= 4 ? 1 : 3; /* accumulators per output tile: one per plane where tiles are few */
    constexpr int OUTS = NB * MB * 256;
    static_assert(ANY_KW * OUTS <= GLINT_LDS_CELLS64_WORDS, "partials fit the table's LDS");
    __shared__ __attribute__((aligned(16))) float ltab[GLINT_LDS_CELLS64_WORDS];
    __shared__ int s_again;
    const int lane = threadIdx.x & 63, m16 = lane & 15, g = lane >> 4;
    const int kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane4 = (uint32_t)(lane & 31) * 4u; /* the half-filled table: copy lane % 32 */
    const int n0 = (strip0 + (int)blockIdx.x) * 16 * NB, m0 = blockIdx.y * 16 * MB;
    /* this wave's whole chunks of 128; the last wave also takes the partial chunk */
    const int nfull = K >> 7, cpw = (nfull + ANY_KW - 1) / ANY_KW;
    const int cbeg = min(kw * cpw, nfull), cend = min(cbeg + cpw, nfull);

    GlintCellFillHN<2048 / T> fill;
    glint_cells_fillh_sload(fill);

    /* rows past N or M repeat the last one (their outputs are not stored) */
    const uint16_t *xp[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
        xp[b] = x + (int64_t)min(m0 + 16 * b + m16, M - 1) * K + 32 * g;
    struct Strip {
        int64_t e;      /* first element of the lane's group in the next chunk to load */
        int64_t q;      /* its block */
        int r;          /* its place in that block */
    };
    Strip sp[NB];
    const int dq = 128 / bs, dr = 128 % bs;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        sp[b].e = (int64_t)min(n0 + 16 * b + m16, N - 1) * K + 32 * g + (int64_t)cbeg * 128;
        sp[b].q = sp[b].e / bs;
        sp[b].r = (int)(sp[b].e - sp[b].q * bs);
    }
    const uint32_t nsh[2] = {0u, 4u};
    uint32_t sh[NB]; /* ODD: the row's nibble shift */
#pragma unroll
    for (int b = 0; b < NB; ++b)
        sh[b] = ODD ? nsh[sp[b].e & 1] : 0u;

    struct WChunk {
        glint_u32x4 h, p;
        uint32_t h4, p4; /* ODD: the 17th byte */
        float a0, a1;    /* scales before and from element jb on */
        int jb;
        int64_t q;       /* SB: block of element 0 */
        int r;
    };
    struct Stage {
        WChunk w[NB];
        glint_u32x4 x[NB == 1 ? MB : 1][4];
    };
    glint_u32x4 x1[NB == 1 ? 1 : MB][4]; /* two strips: x of the chunk at work, not loaded ahead (registers) */
    uint32_t amin = 0xFFFFFFFFu; /* smallest |scale| bits - 1 met (0 wraps to the top) */
    auto wload = [&](WChunk &c, Strip &s) {
        const uint8_t *hb = hole + (s.e >> 1), *pb = plug + (s.e >> 1);
        c.h = *(const glint_u32x4_b1 *)hb;
        c.p = *(const glint_u32x4_b1 *)pb;
        if constexpr (ODD) { /* read at an even row too: element 31's byte again there */
            const int last = 15 + (int)(s.e & 1);
            c.h4 = hb[last];
            c.p4 = pb[last];
        }
        if constexpr (SB) {
            c.q = s.q;
            c.r = s.r;
        } else {
            c.jb = bs - s.r;
            c.a0 = absmax[s.q];
            c.a1 = absmax[s.q + (c.jb < 32 ? 1 : 0)];
        }
        s.e += 128;
        s.q += dq;
        s.r += dr;
        if (s.r >= bs) {
            s.r -= bs;
            ++s.q;
        }
    };
    auto xload = [&](glint_u32x4 (&xs)[MB][4], int c) {
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                xs[b][s] = *(const glint_u32x4_b2 *)(xp[b] + (int64_t)c * 128 + 8 * s);
    };
    auto xreg = [&](Stage &st) -> glint_u32x4 (&)[MB][4] {
        if constexpr (NB == 1)
            return st.x;
        else
            return x1;
    };
    auto load = [&](Stage &st, int c) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
            wload(st.w[b], sp[b]);
        if constexpr (NB == 1)
            xload(st.x, c);
    };

    glint_f32x4 acc[NB][MB][NA];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
            for (int i = 0; i < NA; ++i)
                acc[b][a][i] = glint_f32x4{0.f, 0.f, 0.f, 0.f};

    /* 8 weights by their codes and scales, split into three planes */
    auto split = [&](uint32_t H, uint32_t P, const float (&sc)[8], glint_bf16x8 (&bp)[3]) {
        const uint32_t E = glint_codes_even(H, P), O = glint_codes_odd(H, P);
        float v[8];
        v[0] = glint_lds_f32(ltab, glint_cell_addr<0>(E, lane4));
        v[1] = glint_lds_f32(ltab, glint_cell_addr<0>(O, lane4));
        v[2] = glint_lds_f32(ltab, glint_cell_addr<1>(E, lane4));
        v[3] = glint_lds_f32(ltab, glint_cell_addr<1>(O, lane4));
        v[4] = glint_lds_f32(ltab, glint_cell_addr<2>(E, lane4));
        v[5] = glint_lds_f32(ltab, glint_cell_addr<2>(O, lane4));
        v[6] = glint_lds_f32(ltab, glint_cell_addr<3>(E, lane4));
        v[7] = glint_lds_f32(ltab, glint_cell_addr<3>(O, lane4));
        uint32_t hi[8], mid[8], lo[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float w = v[i] * sc[i];
            const float r1 = w - __uint_as_float(__float_as_uint(w) & 0xFFFF0000u);
            hi[i] = __float_as_uint(w);
            mid[i] = __float_as_uint(r1);
            lo[i] = __float_as_uint(r1 - __uint_as_float(mid[i] & 0xFFFF0000u));
        }
        uint32_t pk[3][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) { /* the perm keeps each word's upper half: the truncation */
            pk[0][j] = __builtin_amdgcn_perm(hi[2 * j + 1], hi[2 * j], 0x07060302u);
            pk[1][j] = __builtin_amdgcn_perm(mid[2 * j + 1], mid[2 * j], 0x07060302u);
            pk[2][j] = __builtin_amdgcn_perm(lo[2 * j + 1], lo[2 * j], 0x07060302u);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            bp[i] = __builtin_bit_cast(glint_bf16x8, glint_u32x4{pk[i][0], pk[i][1], pk[i][2], pk[i][3]});
    };
    /* a chunk; kin: elements of the lane's group inside the row (32, fewer in the last chunk) */
    auto compute = [&](Stage &st, int kin, bool tail) {
        const auto &xs = xreg(st);
        bool two = false;
        if constexpr (!SB) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                two |= st.w[b].jb < 32;
                amin = min(amin, min((__float_as_uint(st.w[b].a0) & 0x7FFFFFFFu) - 1u,
                                     (__float_as_uint(st.w[b].a1) & 0x7FFFFFFFu) - 1u));
            }
            two = __any(two);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const WChunk &c = st.w[b];
                uint32_t H = c.h[s], P = c.p[s];
                if constexpr (ODD) {
                    const uint32_t hn = s < 3 ? c.h[s < 3 ? s + 1 : 3] : c.h4, pn = s < 3 ? c.p[s < 3 ? s + 1 : 3] : c.p4;
                    H = __builtin_amdgcn_alignbit(hn, H, sh[b]);
                    P = __builtin_amdgcn_alignbit(pn, P, sh[b]);
                }
                float sc[8];
                if constexpr (SB) {
                    int64_t q = c.q + (c.r + 8 * s) / bs;
                    int r = (c.r + 8 * s) % bs;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const bool in = !tail || 8 * s + i < kin;
                        sc[i] = in ? absmax[q] : 0.0f;
                        amin = min(amin, (__float_as_uint(sc[i]) & 0x7FFFFFFFu) - 1u);
                        if (++r == bs) {
                            r = 0;
                            ++q;
                        }
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        sc[i] = c.a0;
                    if (two || tail)
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            sc[i] = 8 * s + i < c.jb ? c.a0 : c.a1;
                            if (tail && 8 * s + i >= kin)
                                sc[i] = 0.0f;
                        }
                }
                glint_bf16x8 bp[3];
                split(H, P, sc, bp);
#pragma unroll
                for (int pl = 2; pl >= 0; --pl)
#pragma unroll
                    for (int a = 0; a < MB; ++a)
                        acc[b][a][NA == 3 ? pl : 0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(glint_bf16x8, xs[a][s]), bp[pl], acc[b][a][NA == 3 ? pl : 0], 0, 0, 0);
            }
        }
    };

    /* one chunk in flight beside the one computed */
    Stage st0, st1;
    if (cbeg < cend)
        load(st0, cbeg);
    glint_cells_fillh_sstore(ltab, fill);
    if (threadIdx.x == 0)
        s_again = 0;
    __syncthreads();
    int c = cbeg;
    auto whole = [&](Stage &st, int c) {
        if constexpr (NB > 1)
            xload(x1, c);
        compute(st, 32, false);
    };
    for (; c + 2 < cend; c += 2) {
        load(st1, c + 1);
        whole(st0, c);
        load(st0, c + 2);
        whole(st1, c + 1);
    }
    if (c + 1 < cend) {
        load(st1, c + 1);
        whole(st0, c);
        whole(st1, c + 1);
    } else if (c < cend) {
        whole(st0, c);
    }

    /* the partial chunk, read element by element: nothing past a row's end is read */
    if (kw == ANY_KW - 1 && (K & 127)) {
        const int kin = min(max(K - nfull * 128 - 32 * g, 0), 32);
        Stage &t = st0;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            WChunk &w = t.w[b];
            const int64_t e = (int64_t)min(n0 + 16 * b + m16, N - 1) * K + (int64_t)nfull * 128 + 32 * g;
            const int nb = kin > 0 ? (int)(((e + kin - 1) >> 1) - (e >> 1)) + 1 : 0; /* bytes: at most 17 */
            const uint8_t *hb = hole + (e >> 1), *pb = plug + (e >> 1);
            uint32_t hw[5], pw[5];
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                hw[i] = pw[i] = 0u;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * i + j < nb) {
                        hw[i] |= (uint32_t)hb[4 * i + j] << (8 * j);
                        pw[i] |= (uint32_t)pb[4 * i + j] << (8 * j);
                    }
            }
            w.h = glint_u32x4{hw[0], hw[1], hw[2], hw[3]};
            w.p = glint_u32x4{pw[0], pw[1], pw[2], pw[3]};
            w.h4 = hw[4];
            w.p4 = pw[4];
            w.q = kin > 0 ? e / bs : 0;
            w.r = kin > 0 ? (int)(e - w.q * bs) : 0;
            w.jb = bs - w.r;
            if constexpr (!SB) {
                w.a0 = kin > 0 ? absmax[w.q] : 0.0f;
                w.a1 = w.jb < kin ? absmax[w.q + 1] : 0.0f;
            }
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                uint32_t xw[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint16_t *p = xp[b] + (int64_t)nfull * 128 + 8 * s + 2 * i;
                    xw[i] = 8 * s + 2 * i < kin ? p[0] : 0u;
                    if (8 * s + 2 * i + 1 < kin)
                        xw[i] |= (uint32_t)p[1] << 16;
                }
                xreg(t)[b][s] = glint_u32x4{xw[0], xw[1], xw[2], xw[3]};
            }
        compute(t, kin, true);
    }

    /* the waves' sums, added in wave order; the table is no longer read */
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v = acc[b][a][0][i];
                if constexpr (NA == 3)
                    v += acc[b][a][1][i] + acc[b][a][2][i];
                ltab[kw * OUTS + ((b * MB + a) * 4 + i) * 64 + lane] = v;
            }
    if (amin < ANY_SCALE_LO - 1u)
        s_again = 1;
    __syncthreads();
    float v[(OUTS + T - 1) / T];
    bool again = false;
#pragma unroll
    for (int j = 0; j < (OUTS + T - 1) / T; ++j) {
        const int o = (int)threadIdx.x + j * T;
        if (OUTS % T != 0 && o >= OUTS)
            break;
        v[j] = ltab[o];
#pragma unroll
        for (int k = 1; k < ANY_KW; ++k)
            v[j] += ltab[k * OUTS + o];
        again |= !(__builtin_fabsf(v[j]) < __builtin_inff());
    }
    if (again)
        s_again = 1;
    __syncthreads();
    if (s_again)
        htile_any_again<MB, NB>(ltab, hole, plug, absmax, x, m0, n0, M, N, K, bs, v);
#pragma unroll
    for (int j = 0; j < (OUTS + T - 1) / T; ++j) {
        const int o = (int)threadIdx.x + j * T;
        if (OUTS % T != 0 && o >= OUTS)
            break;
        const int l = o & 63, i = (o >> 6) & 3, a = (o >> 8) % MB, b = (o >> 8) / MB;
        const int m = m0 + 16 * a + 4 * (l >> 4) + i, n = n0 + 16 * b + (l & 15);
        if (m < M && n < N)
            Out::store(y, (int64_t)m * N + n, v[j]);
    }
}

/* 16, 32 or 64 rows of x per workgroup by M. Above 64 rows two strips of W per wave where the
 * workgroups still cover the CUs: the reads of x per weight halve (130 x 5000 x 5000 80 -> 64
 * us, 2048 x 4096 x 4104 531 -> 441; x is then not loaded a chunk ahead, which would spill). */
template <class Out, int MB, int NB, bool SB>
static int htile_any_launch_nb(const uint8_t *hole, const uint8_t *plug, const float *absmax, const void *x, void *y,
                               int M, int N, int K, int bs, hipStream_t st) {
    auto kern = (K & 1) ? k_htile_any<MB, NB, true, SB, Out> : k_htile_any<MB, NB, false, SB, Out>;
    const int64_t strips = ((int64_t)N + 16 * NB - 1) / (16 * NB), most = 1 << 21; /* a grid has < 2^32 threads */
    const unsigned gy = (unsigned)(((int64_t)M + 16 * MB - 1) / (16 * MB));
    for (int64_t s0 = 0; s0 < strips; s0 += most)
        kern<<<dim3((unsigned)std::min(most, strips - s0), gy), 64 * ANY_KW, 0, st>>>(
            hole, plug, absmax, (const uint16_t *)x, (typename Out::T *)y, M, N, K, bs, (int)s0);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}
template <class Out>
static int htile_any_launch(const uint8_t *hole, const uint8_t *plug, const float *absmax, const void *x, void *y,
                            int M, int N, int K, int bs, hipStream_t st) {
    if (bs < 32)
        return M <= 16 ? htile_any_launch_nb<Out, 1, 1, true>(hole, plug, absmax, x, y, M, N, K, bs, st)
                       : htile_any_launch_nb<Out, 4, 1, true>(hole, plug, absmax, x, y, M, N, K, bs, st);
    if (M <= 16)
        return htile_any_launch_nb<Out, 1, 1, false>(hole, plug, absmax, x, y, M, N, K, bs, st);
    if (M <= 32)
        return htile_any_launch_nb<Out, 2, 1, false>(hole, plug, absmax, x, y, M, N, K, bs, st);
    if (M > 64 && (int64_t)((N + 31) / 32) * ((M + 63) / 64) >= glint_cu_count())
        return htile_any_launch_nb<Out, 4, 2, false>(hole, plug, absmax, x, y, M, N, K, bs, st);
    return htile_any_launch_nb<Out, 4, 1, false>(hole, plug, absmax, x, y, M, N, K, bs, st);
}

#endif
