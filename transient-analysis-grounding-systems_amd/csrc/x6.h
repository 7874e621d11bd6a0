// Complex64 products on the bf16 MFMA cores of gfx950.
#pragma once

#include "tags_common.h"

namespace tags {

// ---------------------------------------------------------------------------
// complex64 on the bf16 MFMA cores (variants 22..32). Every fp32 operand value
// x is split into three bf16 parts x = x1 + x2 + x3, each the round-to-nearest
// bf16 of what the earlier parts leave: x1 holds the leading 8 significant
// bits, x2 the next 8, x3 the last 8, so that the parts sum to x exactly (for
// |x| well inside the normal range; the differences are exact in fp32). A real
// product x y is formed from the six part products x1y1, x1y2, x2y1, x1y3,
// x2y2, x3y1, accumulated in fp32; the three left out (x2y3, x3y2, x3y3) add up
// to less than 2^-24 |x||y|, the size of one fp32 rounding of the term.
// Complex products take four real ones (re re - im im, re im + im re): 24 bf16
// MFMAs where the three-multiply fp32 form issues 3 fp32 ones, and bf16 runs at
// 16x the fp32 MFMA rate on gfx950, so a complex product takes 24 / 16 = 1.5
// fp32-MFMA issue slots instead of 3.
//
// The operands are first packed (k_pack_x6) into MFMA fragment order: for a
// block of 32 rows of A (32 columns of B) and a slab of 16 k, part p (the
// three parts of the real values, then of the imaginary ones) is 64 lanes x 8
// bf16 = 1 KiB, lane l holding row (column) l % 32 at k = 8 (l / 32) .. + 7,
// zero past the matrix. A wave loads each fragment with one 16-byte load per
// lane straight into MFMA operand registers, the next slab's while the
// current one's MFMAs run; blocks past the product's edge repeat the last
// block and their results are dropped at the store.
// v_mfma_f32_32x32x16_bf16: lane l supplies A[l % 32][8 (l / 32) + e] and
// B[8 (l / 32) + e][l % 32], e = 0..7 (A and B packed alike, so the k order
// inside a slab is the same on both sides, which is all the sum needs); result
// value v of lane l is D[(v % 4) + 8 (v / 4) + 4 (l / 32)][l % 32], as for the
// 32 x 32 f32 blocks above.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int X6_KMAX = 256;  // largest K (the LU's widest step)
constexpr int X6_FRAG = 64;   // 16-byte words per fragment
constexpr int X6_PARTS = 6;

// round to nearest even bf16 (finite x), as the upper 16 bits of an fp32
__device__ inline unsigned bf16_rn(float x)
{
    unsigned u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ inline void x6_split(float x, unsigned& h1, unsigned& h2, unsigned& h3)
{
    h1 = bf16_rn(x);
    const float r1 = x - __uint_as_float(h1 << 16);
    h2 = bf16_rn(r1);
    const float r2 = r1 - __uint_as_float(h2 << 16);
    h3 = bf16_rn(r2);
}

// 16-byte word of the first part of row i, columns k .. k + 7 (k a multiple of 8)
// in a pack of ks slabs per block; part p is X6_FRAG p words further
__device__ inline long x6_word(int i, int k, int ks)
{
    return ((long)(i >> 5) * ks + (k >> 4)) * (X6_PARTS * X6_FRAG) + ((k >> 3) & 1) * 32 + (i & 31);
}
// the parts of eight consecutive columns of a row to o, o + X6_FRAG, ..
__device__ inline void x6_pack8(const c32 (&x)[8], u32x4* o)
{
    unsigned w[X6_PARTS][4];
#pragma unroll
    for (int e = 0; e < 8; e += 2)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            unsigned a1, a2, a3, b1, b2, b3;
            x6_split(c ? x[e].y : x[e].x, a1, a2, a3);
            x6_split(c ? x[e + 1].y : x[e + 1].x, b1, b2, b3);
            w[3 * c + 0][e / 2] = a1 | (b1 << 16);
            w[3 * c + 1][e / 2] = a2 | (b2 << 16);
            w[3 * c + 2][e / 2] = a3 | (b3 << 16);
        }
#pragma unroll
    for (int p = 0; p < X6_PARTS; p++) {
        u32x4 q;
        q.x = w[p][0];
        q.y = w[p][1];
        q.z = w[p][2];
        q.w = w[p][3];
        o[p * X6_FRAG] = q;
    }
}

struct X6Args {
    int M, N, K;
    int ks;           // slabs per block in the packs (at least those of K)
    const u32x4* pa;  // packed A rows
    const u32x4* pb;  // packed B columns
    long spk;         // item stride of the packs (16-byte words)
    c32* C;
    long ldc;
    const int* crow;
    long sc, scr;
    int mode;  // 0: C = A B; 1: C -= A B
};

__device__ __forceinline__ bf16x8 as_bf16(u32x4 u) { return __builtin_bit_cast(bf16x8, u); }
__device__ __forceinline__ f32x16 mfma_x6(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(a), as_bf16(b), c, 0, 0, 0);
}

// C = v (mode 0) or C -= v (mode 1) for one complex64 entry
template <bool NTC>
__device__ __forceinline__ void x6_store(c32* p, float re, float im, int mode)
{
    float* f = (float*)p;
    if constexpr (NTC) {
        if (mode == 0) {
            __builtin_nontemporal_store(re, f);
            __builtin_nontemporal_store(im, f + 1);
        } else {
            const float cr = __builtin_nontemporal_load(f), ci = __builtin_nontemporal_load(f + 1);
            __builtin_nontemporal_store(cr - re, f);
            __builtin_nontemporal_store(ci - im, f + 1);
        }
    } else {
        if (mode == 0) {
            *p = c32{re, im};
        } else {
            const c32 c = *p;
            *p = c32{c.x - re, c.y - im};
        }
    }
}

// The same product with the work-group's fragments of each slab staged once
// in LDS (double-buffered): every thread copies its share of the slab's
// fragments (global -> registers -> LDS, 16 bytes at a time, a wave's words
// contiguous) for the next slab while the MFMAs of the current one run, and
// each wave reads its own fragments from LDS, one barrier per slab. The
// work-group fetches a fragment once instead of once per wave that uses it.
// The tile at row tile tm and column tile tn; the operands' and C's pointers are
// the item's.
template <int WGM, int WGN, int TM, int TN, bool NTC, int DEPTH>
__device__ __forceinline__ void x6l_tile(const X6Args& g, int tm, int tn)
{
    constexpr int NT = 64 * WGM * WGN;
    constexpr int BM = 32 * TM * WGM, BN = 32 * TN * WGN;
    constexpr int FA = BM / 32 * X6_PARTS, FB = BN / 32 * X6_PARTS;  // fragments per slab
    constexpr int NF = FA + FB;
    constexpr int NW = NF * X6_FRAG / NT;  // 16-byte words a thread stages
    static_assert(NW * NT == NF * X6_FRAG, "slab words per thread");
    static_assert(NT % 64 == 0 && (NT / 64) * NW == NF, "fragments per wave");
    __shared__ u32x4 lds[2][NF * X6_FRAG];

    const u32x4* pa = g.pa;
    const u32x4* pb = g.pb;
    c32* C = g.C;
    const int* crow = g.crow;
    const int M = g.M, N = g.N, KS = (g.K + 15) / 16, KP = g.ks;
    // the wave index is uniform: kept in scalar registers, so that the
    // fragment addresses are a scalar base plus the lane's offset
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int nbm = (M + 31) / 32, nbn = (N + 31) / 32;
    // staging: word q of this thread is word `lane` of fragment wave + (NT/64) q
    // of the slab (A fragments first: block, part; then B's)
    const u32x4* src[NW];
#pragma unroll
    for (int q = 0; q < NW; q++) {
        const int fi = wave + (NT / 64) * q;
        if (fi < FA) {
            const int b = min(tm * (BM / 32) + fi / X6_PARTS, nbm - 1);
            src[q] = pa + (long)b * KP * (X6_PARTS * X6_FRAG) + (fi % X6_PARTS) * X6_FRAG + lane;
        } else {
            const int f2 = fi - FA;
            const int b = min(tn * (BN / 32) + f2 / X6_PARTS, nbn - 1);
            src[q] = pb + (long)b * KP * (X6_PARTS * X6_FRAG) + (f2 % X6_PARTS) * X6_FRAG + lane;
        }
    }
    // two register sets: with DEPTH 2 a slab's words are fetched two slabs
    // before they are stored to LDS, so that a fetch from beyond L2 is covered
    u32x4 stage[2][NW];
    auto gload = [&](int set, int ks) {
        const long o = (long)ks * (X6_PARTS * X6_FRAG);
#pragma unroll
        for (int q = 0; q < NW; q++) stage[set][q] = src[q][o];
    };
    auto sstore = [&](int set, int buf) {
#pragma unroll
        for (int q = 0; q < NW; q++)
            lds[buf][(wave + (NT / 64) * q) * X6_FRAG + lane] = stage[set][q];
    };

    f32x16 re[TM][TN], im[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                re[i][j][v] = 0.f;
                im[i][j][v] = 0.f;
            }
        }
    auto mma = [&](int buf) {
        const u32x4* la = lds[buf] + (wm * TM * X6_PARTS) * X6_FRAG + lane;
        const u32x4* lb = lds[buf] + (FA + wn * TN * X6_PARTS) * X6_FRAG + lane;
        u32x4 a[TM][X6_PARTS], b[TN][X6_PARTS], nbi[TN][3];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int p = 0; p < X6_PARTS; p++) a[i][p] = la[(i * X6_PARTS + p) * X6_FRAG];
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int p = 0; p < X6_PARTS; p++) b[j][p] = lb[(j * X6_PARTS + p) * X6_FRAG];
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int t = 0; t < 3; t++) nbi[j][t] = b[j][3 + t] ^ 0x80008000u;
        constexpr int PS[6] = {2, 1, 0, 1, 0, 0}, PT[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const int s = PS[q], t = PT[q];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    re[i][j] = mfma_x6(a[i][s], b[j][t], re[i][j]);
                    im[i][j] = mfma_x6(a[i][s], b[j][3 + t], im[i][j]);
                }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    re[i][j] = mfma_x6(a[i][3 + s], nbi[j][t], re[i][j]);
                    im[i][j] = mfma_x6(a[i][3 + s], b[j][t], im[i][j]);
                }
        }
    };
    // the same products one column block at a time, a scheduling barrier
    // between blocks, so that only one block's B fragments are live (fewer
    // registers, room for the second staging set)
    auto mma_cols = [&](int buf) {
        const u32x4* la = lds[buf] + (wm * TM * X6_PARTS) * X6_FRAG + lane;
        const u32x4* lb = lds[buf] + (FA + wn * TN * X6_PARTS) * X6_FRAG + lane;
        u32x4 a[TM][X6_PARTS];
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int p = 0; p < X6_PARTS; p++) a[i][p] = la[(i * X6_PARTS + p) * X6_FRAG];
#pragma unroll
        for (int j = 0; j < TN; j++) {
            u32x4 b[X6_PARTS], nbi[3];
#pragma unroll
            for (int p = 0; p < X6_PARTS; p++) b[p] = lb[(j * X6_PARTS + p) * X6_FRAG];
#pragma unroll
            for (int t = 0; t < 3; t++) nbi[t] = b[3 + t] ^ 0x80008000u;
            constexpr int PS[6] = {2, 1, 0, 1, 0, 0}, PT[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
            for (int q = 0; q < 6; q++) {
                const int s = PS[q], t = PT[q];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    re[i][j] = mfma_x6(a[i][s], b[t], re[i][j]);
                    im[i][j] = mfma_x6(a[i][s], b[3 + t], im[i][j]);
                    re[i][j] = mfma_x6(a[i][3 + s], nbi[t], re[i][j]);
                    im[i][j] = mfma_x6(a[i][3 + s], b[t], im[i][j]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if constexpr (DEPTH == 1) {
        gload(0, 0);
        sstore(0, 0);
        __syncthreads();
        for (int ks = 0; ks < KS; ks++) {
            const bool more = ks + 1 < KS;
            if (more) gload(0, ks + 1);
            mma(ks & 1);
            if (more) sstore(0, (ks + 1) & 1);
            __syncthreads();
        }
    } else {
        // slab s is fetched into set s % 2 at slab s - 2 and stored to LDS
        // buffer s % 2 at the end of slab s - 1
        gload(0, 0);
        sstore(0, 0);
        if (KS > 1) gload(1, 1);
        if (KS > 2) gload(0, 2);
        __syncthreads();
        for (int ks = 0; ks < KS; ks += 2) {
            // even slab ks in LDS buffer 0; ks + 1 in set 1, ks + 2 in set 0
            mma_cols(0);
            if (ks + 1 < KS) sstore(1, 1);
            if (ks + 3 < KS) gload(1, ks + 3);
            __syncthreads();
            if (ks + 1 >= KS) break;
            mma_cols(1);
            if (ks + 2 < KS) sstore(0, 0);
            if (ks + 4 < KS) gload(0, ks + 4);
            __syncthreads();
        }
    }

    const int m0 = tm * BM + wm * TM * 32, n0 = tn * BN + wn * TN * 32;
    const int kl = lane >> 5, ml = lane & 31;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = m0 + i * 32 + (v & 3) + 8 * (v >> 2) + 4 * kl;
            if (row >= M) continue;
            c32* cr = C + (long)(crow ? crow[row] : row) * g.ldc;
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int col = n0 + j * 32 + ml;
                if (col >= N) continue;
                x6_store<NTC>(cr + col, re[i][j][v], im[i][j][v], g.mode);
            }
        }
}

}  // namespace tags
