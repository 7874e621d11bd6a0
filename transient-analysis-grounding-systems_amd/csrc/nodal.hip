// Nodal solve of the HEM immittance system from explicit symmetric inverses,
// batched over the frequency samples of a group.
//
//   [ -Z_L   0    A ] [i_L]   [r_L]
//   [   0  -Z_T   B ] [i_T] = [r_T]     A, B: incidence, two entries per row
//   [ A^T   B^T   0 ] [ u ]   [r_U]
//
// is solved by Y_L = Z_L^-1, Y_T = Z_T^-1, S = A^T Y_L A + B^T Y_T B and
//   S u = r_U + A^T Y_L r_L + B^T Y_T r_T,  i_L = Y_L (A u - r_L),  i_T alike,
// refined on W with double-double residuals. Z_L, Z_T and S are complex
// symmetric with a definite real or imaginary part, so no row exchanges are
// needed; a sample whose refinement does not meet the acceptance rule is left
// to the caller's pivoted factorisation.
//
// Why explicit inverses: the blocked symmetric sweep below takes 4 dim^3 real
// operations for an inverse (half of a general one's), all of them in one
// shape of matrix product that does not shrink from step to step; the
// incidence products with Y are gathers of four entries; and every solve of
// the refinement is a matrix-vector product at memory speed, where triangular
// solves are a chain of dependent blocks. For a 60 x 60 m grid (m = 7,440,
// n = 6,541) that is 4.4e12 operations per sample, against 8.7e12 for the
// block elimination with the node columns carried along and 1.84e13 for the
// pivoted elimination.
//
// The node system. At low frequency |Y_L| >> |Y_T|, and the constant vector,
// which A annihilates, has in S a quadratic form far below the rounding of
// S's entries. So S_p = S + tau 1 1^T is inverted instead (tau: the mean
// diagonal / n, so that the constant vector's eigenvalue is of the diagonal's
// size), and the constant part alpha of u = alpha 1 + w follows from sums that
// A does not enter: with c = S 1 = B^T (Y_T 1) and s = 1^T S 1 = sum(Y_T 1)
// (A 1 = 0, B 1 = 1), h = S_p^-1 c, y = S_p^-1 f and F = 1^T f,
//   alpha = (F - c^T y) / (s - c^T h),  w = y - alpha h.
// A u = A w is then formed without alpha. In complex64 a refinement step then
// contracts the error by 1e-2 .. 1e-4 at every frequency from 100 Hz to 10 MHz
// (m = 30 .. 1320), where the plain S stalled below 20 kHz.
//
// Separate conductors. With several parts of the node graph every part's constant
// vector 1_j is such a vector (with the shift of 1 1^T alone two rods contracted by
// 0.1 a step at 60 Hz, a conductor beside a rod not at all). The shift and alpha
// then belong to the first part, and every other part's root node r_j takes
// the part's constant as its unknown: u = w + beta_j on part j, w = 0 at r_j, so
// that row and column r_j of the system become
//   1_j^T S e_u = (B^T Y_T 1_j)_u,  1_j^T S 1_k = sum over j of Y_T 1_k,
// again without A, and entry r_j of a right-hand side becomes the sum of r_U and
// Y_T r_T over the part. On the CPU in complex64: 1e-6 .. 1e-4 a step for two to
// eight parts from 60 Hz to 1 MHz.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "dd.h"
#include "mfma.h"
#include "nodal.h"

namespace tags {

// Work-group index over `total` pieces of work such that each XCD (blockIdx.x
// mod 8) takes a contiguous range, so that the pieces of one item meet in one
// L2; -1 past the end. The grid is 8 * ceil(total / 8).
__device__ inline long xcd_flat(long total)
{
    const long per = (total + 7) / 8;
    const long f = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    return f < total ? f : -1;
}
static unsigned xcd_grid(long total) { return (unsigned)(8 * ((total + 7) / 8)); }

// One family of symmetric matrices being inverted: `items` matrices of order
// dim in ld x ld storage (ld = dim rounded up to 64, zero beyond dim), of
// which the 64 x 64 tiles on and below the diagonal are kept.
template <typename T>
struct NdPhase {
    cx<T>* A;
    long sA;
    int ld, dim, items;
    cx<T>*tp, *op;  // T and O of the current step in MFMA fragment order
    long sp;
    cx<T>* P;       // inverses of the step's diagonal blocks, in fragment order
};

// Fragment order of a ld x NB panel: a wave's MFMA operand (16 rows, 4 k) is
// 64 consecutive complex values; complex64 keeps two k groups side by side,
// so that every lane loads 16 bytes.
template <typename T, int NB>
__device__ inline long nd_pk(int i, int k)
{
    if constexpr (sizeof(T) == 8)
        return ((long)(i >> 4) * (NB / 4) + (k >> 2)) * 64 + (k & 3) * 16 + (i & 15);
    else
        return (((long)(i >> 4) * (NB / 8) + (k >> 3)) * 64 + (k & 3) * 16 + (i & 15)) * 2 +
               ((k >> 2) & 1);
}

// Complex MFMA accumulators: complex128 by four real products (re, im),
// complex64 by three (re re, im im, (re + im)(re + im); Gauss), as the LU's
// products of each type.
template <typename T>
struct NdAcc;
template <>
struct NdAcc<double> {
    typename Mfma<double>::v4 re, im;
    __device__ void zero() { re = im = typename Mfma<double>::v4{0, 0, 0, 0}; }
    __device__ void mac(c64 x, c64 y)
    {
        re = Mfma<double>::run(x.x, y.x, re);
        im = Mfma<double>::run(x.x, y.y, im);
        re = Mfma<double>::run(-x.y, y.y, re);
        im = Mfma<double>::run(x.y, y.x, im);
    }
    __device__ c64 get(int v) const { return c64{re[v], im[v]}; }
};
template <>
struct NdAcc<float> {
    typename Mfma<float>::v4 rr, ii, ss;
    __device__ void zero() { rr = ii = ss = typename Mfma<float>::v4{0, 0, 0, 0}; }
    __device__ void mac(c32 x, c32 y)
    {
        rr = Mfma<float>::run(x.x, y.x, rr);
        ii = Mfma<float>::run(x.y, y.y, ii);
        ss = Mfma<float>::run(x.x + x.y, y.x + y.y, ss);
    }
    __device__ c32 get(int v) const { return c32{rr[v] - ii[v], ss[v] - rr[v] - ii[v]}; }
};

// The value is needed here: keeps the loads of the next k group ahead of this
// one's products (the compiler otherwise moves them to their use, one iteration
// later, and every wave waits out each load).
template <typename T, int N>
__device__ __forceinline__ void nd_pin(cx<T> (&e)[N])
{
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("" : "+v"(e[i].x), "+v"(e[i].y));
}

// acc (tiles of a wave) += T_i O_j^T over the k groups [g0, g1) of 16-row
// strips: operands in fragment order straight from memory, the loads of the next
// D - 1 groups in flight during one group's MFMAs. Two hide the latency where
// several waves share a SIMD; the diagonal block's product has one wave on each.
template <typename T, int NB, int TI, int TJ, int D = 2>
__device__ __forceinline__ void nd_mma(const cx<T>* tp, const cx<T>* op, int i0, int j0, int g0,
                                       int g1, NdAcc<T> (&acc)[TI][TJ])
{
    constexpr int KG = sizeof(T) == 8 ? 4 : 8;  // k per 16-byte lane load
    constexpr int KU = KG / 4;
    constexpr long FS = (long)(NB / KG) * 64;  // loads of one 16-row strip
    struct alignas(16) Frag {
        cx<T> e[KU];
    };
    const int lane = threadIdx.x & 63;
    const Frag* ta = (const Frag*)tp + (i0 / 16) * FS + lane;
    const Frag* ob = (const Frag*)op + (j0 / 16) * FS + lane;
    if (g0 >= g1) return;
    Frag a[D][TI], b[D][TJ];
    auto load = [&](int d, int g) {
        const long o = (long)min(g, g1 - 1) * 64;
#pragma unroll
        for (int i = 0; i < TI; i++) a[d][i] = ta[i * FS + o];
#pragma unroll
        for (int j = 0; j < TJ; j++) b[d][j] = ob[j * FS + o];
        // otherwise the compiler moves the loads to their use, past the products
        // they are to run beside
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int d = 0; d < D; d++) load(d, g0 + d);
    auto mac = [&](int d) {
#pragma unroll
        for (int u = 0; u < KU; u++)
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++) acc[i][j].mac(a[d][i].e[u], b[d][j].e[u]);
        __builtin_amdgcn_sched_barrier(0);
    };
    int g = g0;
    for (; g + D <= g1; g += D)
#pragma unroll
        for (int d = 0; d < D; d++) {
            mac(d);
            load(d, g + d + D);
        }
#pragma unroll
    for (int d = 0; d + 1 < D; d++)
        if (g + d < g1) mac(d);
}
template <typename T>
constexpr int nd_groups(int k)  // k groups of nd_mma in k columns
{
    return sizeof(T) == 8 ? k / 4 : k / 8;
}

// ---------------------------------------------------------------------------
// The symmetric sweep of a block K of columns:
//   P = A_KK^-1, T = A_*K P, A_ij -= T_i A_jK^T, A_*K = T, A_KK = -P;
// after all blocks A holds -A^-1. Every matrix in between is symmetric, rows
// before and after K are treated alike, and only tiles on and below the
// diagonal are touched.
//
// A step takes NB / 64 blocks K_0, K_1, .. of 64 columns from c0 on. Per block
// t, k_nd_diag forms P_t and k_nd_panel O_t = A_*K_t as the earlier blocks of
// the step leave it and T_t = O_t P_t, both without touching A:
//   O_t(i) = A_iK_t - sum_{s < t} T_s(i) O_s(K_t)^T,
// and for a row block K_s of the step itself, s < t (already swept),
//   O_t(K_s) = T_s(K_t)^T - sum_{s < u < t} T_u(K_s) O_u(K_t)^T.
// Then one k_nd_update reads and writes every tile once with all NB columns:
//   A_ij -= sum_u T_u(i) O_u(j)^T,
// and a tile of row block K_s and / or column block K_r, q = max(s, r), gets
//   (-P_q if s = r, else T_q of the other side) - sum_{u > q} T_u(i) O_u(j)^T.
// ---------------------------------------------------------------------------

// LDS of nd_sweep64
template <typename T>
struct NdSweep {
    cx<T> O[2][64][17];  // block column of 16, of this step and of the next
    cx<T> W[64][17];     // each wave's rows of it times the inverse
    cx<T> P[2][16][17];  // minus the inverse of its diagonal block
    cx<T> row[2][16];    // two pivot rows of the diagonal block ..
    cx<T> piv[3];        // .. and their 2 x 2 block
};

// orders LDS accesses of a wave's lanes
__device__ __forceinline__ void nd_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// out = -M^-1 over the first kv rows and columns of a symmetric 16 x 16 matrix
// (which is taken as the identity past kv), by one wave: lanes hold four columns
// of a row. Two pivots at a time, with the inverse I of their 2 x 2 block in
// closed form: the pivot rows (they are the pivot columns too) go through LDS
// with minus the identity in place of the block, which is kept apart; then
// a -= (o I) o^T over both rows serves every entry, once the pivot rows and
// columns themselves are cleared.
template <typename T>
__device__ __forceinline__ void nd_sweep16(const cx<T> (*M)[17], cx<T> (*out)[17], NdSweep<T>& sh,
                                           int kv, int lane)
{
    const int r = lane >> 2, c0 = 4 * (lane & 3);
    const cx<T> zero{0, 0};
    cx<T> a[4];
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = r == c0 + j && r >= kv ? cx<T>{1, 0} : M[r][c0 + j];
    auto put = [&](int n) {
        if (r == n || r == n + 1) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int c = c0 + j;
                cx<T> x = a[j];
                if (c == n || c == n + 1) {
                    if (c >= r) sh.piv[r - n + c - n] = x;
                    x = cx<T>{c == r ? (T)-1 : (T)0, 0};
                }
                sh.row[r - n][c] = x;
                a[j] = zero;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = csel(c0 + j == n || c0 + j == n + 1, zero, a[j]);
        nd_wave_sync();
    };
    put(0);
    for (int k = 0; k < kv; k += 2) {
        const cx<T> p = sh.piv[0], q = sh.piv[1], s = sh.piv[2];
        const cx<T> u = sh.row[0][r], v = sh.row[1][r];
        cx<T> o0[4], o1[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            o0[j] = sh.row[0][c0 + j];
            o1[j] = sh.row[1][c0 + j];
        }
        const cx<T> d = crecip_fast(cfnma(cmul(p, s), q, q));
        const cx<T> i00 = cmul(s, d), i11 = cmul(p, d), t = cmul(q, d);
        const cx<T> l0 = cfnma(cmul(u, i00), v, t), l1 = cfnma(cmul(v, i11), u, t);
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = cfnma(cfnma(a[j], l0, o0[j]), l1, o1[j]);
        nd_wave_sync();
        if (k + 2 < kv) put(k + 2);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) out[r][c0 + j] = a[j];
    nd_wave_sync();
}

// The sweep of a 64 x 64 matrix by four waves, which hold 16 rows each in the
// layout of MFMA results (a[j][v]: column 16 j + lane % 16): a = -a^-1 over its
// first kv rows and columns, 16 at a time. One wave inverts the diagonal block;
// then with O the block column as it was and P that inverse, wave w forms
// W = O_w P and its tiles A_wj -= W O_j^T (in the block's own rows, from zero
// and with W = -P), and the block column becomes W (-P). The tiles of the next
// block column come first, so that its inverse runs beside the other waves'
// remaining products. Per 16 columns one barrier, eight dependent steps of two
// pivots and 16 MFMA products a wave: 64 columns take 25 us in complex128 and 19
// us in complex64, against 28 and 26 us with every entry swept by two pivots at a
// time on the vector units (about 380 instructions per step and thread) and 40 us
// by one. The dependent steps bound it. All threads of the work-group call this;
// those of `idle` only meet the barriers.
template <typename T>
__device__ __forceinline__ void nd_sweep64(cx<T> (&a)[4][4], NdSweep<T>& sh, int kv, int w,
                                           int lane, bool idle = false)
{
    const int lr = lane & 15, lk = lane >> 4, nb = (kv + 15) / 16;
    if (!idle) {
#pragma unroll
        for (int v = 0; v < 4; v++) sh.O[0][16 * w + Mfma<T>::row(lane, v)][lr] = a[0][v];
        nd_wave_sync();
        if (w == 0) nd_sweep16(&sh.O[0][0], sh.P[0], sh, min(16, kv), lane);
    }
    __syncthreads();
    auto step = [&](auto bc) {
        constexpr int b = decltype(bc)::value, h = b & 1;
        if (b >= nb) return;
        if (!idle) {
            cx<T> l[4];
            if (w != b) {
                NdAcc<T> acc;
                acc.zero();
#pragma unroll
                for (int g = 0; g < 4; g++)
                    acc.mac(sh.O[h][16 * w + lr][4 * g + lk], sh.P[h][4 * g + lk][lr]);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const cx<T> x = acc.get(v);
                    a[b][v] = cx<T>{-x.x, -x.y};
                    sh.W[16 * w + Mfma<T>::row(lane, v)][lr] = a[b][v];
                }
                nd_wave_sync();
#pragma unroll
                for (int g = 0; g < 4; g++) l[g] = sh.W[16 * w + lr][4 * g + lk];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        a[j][v] = j == b ? sh.P[h][Mfma<T>::row(lane, v)][lr] : cx<T>{0, 0};
#pragma unroll
                for (int g = 0; g < 4; g++) l[g] = sh.P[h][lr][4 * g + lk];
            }
            auto tile = [&](int j) {
                NdAcc<T> acc;
                acc.zero();
#pragma unroll
                for (int g = 0; g < 4; g++) acc.mac(l[g], sh.O[h][16 * j + lr][4 * g + lk]);
#pragma unroll
                for (int v = 0; v < 4; v++) a[j][v] = csub(a[j][v], acc.get(v));
            };
            if (b < 3 && b + 1 < nb) {
                constexpr int x = b < 3 ? b + 1 : b;
                tile(x);
#pragma unroll
                for (int v = 0; v < 4; v++)
                    sh.O[h ^ 1][16 * w + Mfma<T>::row(lane, v)][lr] = a[x][v];
                nd_wave_sync();
                if (w == x)
                    nd_sweep16(&sh.O[h ^ 1][16 * x], sh.P[h ^ 1], sh, min(16, kv - 16 * x), lane);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j != b && j != b + 1 && j < nb) tile(j);
        }
        __syncthreads();
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
}

// P_t, one work-group per item. A matrix of one block (whole) is finished here:
// both triangles of A get -P.
template <typename T, int NB>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 1) void k_nd_diag(NdPhase<T> p, int c0, int t,
                                                  int whole)
{
    const long item = blockIdx.x;
    const cx<T>* A = p.A + item * p.sA;
    cx<T>* P = p.P + (item * (NB / 64) + t) * 4096;
    const int cK = c0 + 64 * t, kv = min(64, p.dim - cK);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15;
    __shared__ NdSweep<T> sh;
    cx<T> a[4][4];
    // (entry r, c of the tile: row 16 wave + .., column 16 j + ..)
    auto each = [&](auto&& f) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                f(16 * wave + Mfma<T>::row(lane, v), 16 * j + lr, a[j][v], j, v);
    };
    each([&](int r, int c, cx<T>& x, int, int) {
        x = r < kv && c < kv ? A[(long)(cK + max(r, c)) * p.ld + cK + min(r, c)] : cx<T>{0, 0};
    });
    if constexpr (NB > 64) {
        if (t > 0) {
            // less the step's earlier blocks
            NdAcc<T> acc[1][4];
#pragma unroll
            for (int j = 0; j < 4; j++) acc[0][j].zero();
            nd_mma<T, NB, 1, 4, sizeof(T) == 4 ? 3 : 4>(p.tp + item * p.sp, p.op + item * p.sp, cK + 16 * wave, cK, 0,
                                   nd_groups<T>(64 * t), acc);
            each([&](int r, int c, cx<T>& x, int j, int v) {
                if (r < kv && c < kv) x = csub(x, acc[0][j].get(v));
            });
        }
    }
    nd_sweep64(a, sh, kv, wave, lane);
    cx<T>* own = p.A + item * p.sA;
    each([&](int r, int c, cx<T>& x, int, int) {
        const bool in = r < kv && c < kv;
        if (whole)
            own[(long)r * p.ld + c] = in ? x : cx<T>{0, 0};
        else
            P[nd_pk<T, 64>(c, r)] = in ? cx<T>{-x.x, -x.y} : cx<T>{0, 0};
    });
}

// O_t and T_t of 64 rows: four waves of 16 rows and 64 columns, which need no
// barrier: O_t and T_t pass through LDS from the MFMA result layout to the
// operand layout within a wave, so that both are stored a 16-byte fragment per
// lane. Bound by the MFMAs (200 matrices of order 400: 36 us a panel, 55 with
// 8-byte stores and the rows before the step read across the tiles' rows).
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_nd_panel(NdPhase<T> p, int c0, int t)
{
    constexpr int KG = sizeof(T) == 8 ? 4 : 8, KU = KG / 4;  // as in nd_mma
    constexpr long FS = (long)(NB / KG) * 64;
    constexpr int GP = 64 / KG;  // k groups of one block
    struct alignas(16) Frag {
        cx<T> e[KU];
    };
    const int nt = p.ld / 64;
    const long flat = xcd_flat((long)p.items * nt);
    if (flat < 0) return;
    const int item = (int)(flat / nt), rb = (int)(flat % nt);
    const int s = rb * 64 - c0, cK = c0 + 64 * t;
    const int own = s >= 0 && s < NB ? s / 64 : -1;  // block of the step these rows are in
    if (own == t) return;
    const bool swept = own >= 0 && own < t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int i0 = rb * 64 + wave * 16;
    if (i0 >= p.dim) return;
    const int kv = min(64, p.dim - cK);
    const cx<T>* A = p.A + (long)item * p.sA;
    cx<T>* tp = p.tp + (long)item * p.sp;
    cx<T>* op = p.op + (long)item * p.sp;
    const Frag* P = (const Frag*)(p.P + ((long)item * (NB / 64) + t) * 4096) + lane;
    __shared__ cx<T> tile[4][16][65];  // each wave's own
    cx<T>(*my)[65] = tile[wave];
    cx<T> o[4][4];
    // O_t(i): rows before the step are read from the transposed tiles, with the
    // product transposed alike, so that the lanes of a load are neighbours
    auto block = [&](auto& acc, auto at, bool tr) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = Mfma<T>::row(lane, v);
                const int i = tr ? lr : r, k = 16 * c + (tr ? r : lr);
                my[i][k] = k < kv ? csub(o[c][v], at(acc, c).get(v)) : cx<T>{0, 0};
            }
    };
    if (s < 0) {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int k = 16 * c + Mfma<T>::row(lane, v);
                o[c][v] = k < kv ? A[(long)(cK + k) * p.ld + i0 + lr] : cx<T>{0, 0};
            }
        NdAcc<T> acc[4][1];
#pragma unroll
        for (int c = 0; c < 4; c++) acc[c][0].zero();
        if (NB > 64 && t > 0)
            nd_mma<T, NB, 4, 1>(op, tp, cK, i0, 0, nd_groups<T>(64 * t), acc);
        block(acc, [](auto& a, int c) { return a[c][0]; }, true);
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + Mfma<T>::row(lane, v), k = 16 * c + lr;
                o[c][v] = k >= kv ? cx<T>{0, 0}
                          : swept ? tp[nd_pk<T, NB>(cK + k, i - c0)]
                                  : A[(long)i * p.ld + cK + k];
            }
        NdAcc<T> acc[1][4];
#pragma unroll
        for (int c = 0; c < 4; c++) acc[0][c].zero();
        if (NB > 64 && t > 0)
            nd_mma<T, NB, 1, 4>(tp, op, i0, cK, nd_groups<T>(swept ? 64 * (own + 1) : 0),
                                nd_groups<T>(64 * t), acc);
        block(acc, [](auto& a, int c) { return a[0][c]; }, false);
    }
    // T_t(i) = O_t(i) P_t; both stored a fragment at a time
    Frag* oo = (Frag*)op + (i0 / 16) * FS + (long)t * GP * 64 + lane;
    Frag* to = (Frag*)tp + (i0 / 16) * FS + (long)t * GP * 64 + lane;
    Frag b[4], bn[4];
#pragma unroll
    for (int c = 0; c < 4; c++) b[c] = P[c * GP * 64];
    NdAcc<T> acc[4];
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c].zero();
    nd_wave_sync();
    for (int g = 0; g < GP; g++) {
        const int gn = min(g + 1, GP - 1);
#pragma unroll
        for (int c = 0; c < 4; c++) bn[c] = P[(c * GP + gn) * 64];
        Frag a;
#pragma unroll
        for (int u = 0; u < KU; u++) a.e[u] = my[lr][KG * g + 4 * u + lk];
        oo[g * 64] = a;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < KU; u++)
#pragma unroll
            for (int c = 0; c < 4; c++) acc[c].mac(a.e[u], b[c].e[u]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            nd_pin(bn[c].e);
            b[c] = bn[c];
        }
    }
    nd_wave_sync();
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int v = 0; v < 4; v++) my[Mfma<T>::row(lane, v)][16 * c + lr] = acc[c].get(v);
    nd_wave_sync();
#pragma unroll
    for (int g = 0; g < GP; g++) {
        Frag a;
#pragma unroll
        for (int u = 0; u < KU; u++) a.e[u] = my[lr][KG * g + 4 * u + lk];
        to[g * 64] = a;
    }
}

// row and column tile of index t of a triangle's tiles (row >= column)
__device__ inline void tri_tile(int t, int& ti, int& tj)
{
    ti = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while ((ti + 1) * (ti + 2) / 2 <= t) ti++;
    while (ti * (ti + 1) / 2 > t) ti--;
    tj = t - ti * (ti + 1) / 2;
}

// 64 x 64 tiles of the update: four waves of 32 x 32, operands in fragment
// order straight from L2 (a wave needs 4 bytes per cycle of them beside its
// MFMAs, so LDS staging would only add barriers). At order 7440 and 256 columns
// 114 TFLOP/s of fp32 products (154 reached by large matrix products); waves of
// 32 x 64 and 64 x 64, of which fewer fit, take 1.3 and 1.9 times as long, tiles
// in 8 x 8 groups for L2 as long, and the bf16 cores (six products of split
// parts for each of four real ones) twice as long.
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_nd_update(NdPhase<T> p, int c0)
{
    const int nt = p.ld / 64, k0 = c0 / 64, nq = min(NB / 64, nt - k0);
    const int ntri = nt * (nt + 1) / 2;
    const long flat = xcd_flat((long)p.items * ntri);
    if (flat < 0) return;
    const int item = (int)(flat / ntri);
    int ti, tj;
    tri_tile((int)(flat % ntri), ti, tj);
    const int si = ti >= k0 && ti < k0 + nq ? ti - k0 : -1;
    const int sj = tj >= k0 && tj < k0 + nq ? tj - k0 : -1;
    const int q = max(si, sj);
    cx<T>* A = p.A + (long)item * p.sA;
    const cx<T>* tp = p.tp + (long)item * p.sp;
    const cx<T>* op = p.op + (long)item * p.sp;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i0 = ti * 64 + (wave >> 1) * 32, j0 = tj * 64 + (wave & 1) * 32;
    if (i0 >= p.dim || j0 >= p.dim || j0 > i0 + 31) return;
    NdAcc<T> acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j].zero();
    const int kt = (min(NB, p.dim - c0) + 7) & ~7;
    nd_mma<T, NB, 2, 2>(tp, op, i0, j0, nd_groups<T>(64 * (q + 1)), nd_groups<T>(kt), acc);
    const cx<T>* P = q < 0 ? nullptr : p.P + ((long)item * (NB / 64) + q) * 4096;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = i0 + 16 * i + Mfma<T>::row(lane, v);
            if (r >= p.dim) continue;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int c = j0 + 16 * j + (lane & 15);
                if (c >= p.dim) continue;
                cx<T>* a = A + (long)r * p.ld + c;
                cx<T> o;
                if (q < 0) {
                    o = *a;
                } else if (si == sj) {
                    o = P[nd_pk<T, 64>(c - tj * 64, r - ti * 64)];
                    o = cx<T>{-o.x, -o.y};
                } else {
                    o = si > sj ? tp[nd_pk<T, NB>(c, r - c0)] : tp[nd_pk<T, NB>(r, c - c0)];
                }
                *a = csub(o, acc[i][j].get(v));
            }
        }
}

// A_ij of the tiles above the diagonal from those below, 64 x 64 tiles through
// LDS; the diagonal tiles' own upper halves too.
template <typename T>
__global__ __launch_bounds__(256) void k_nd_mirror(cx<T>* A, long sA, int ld, int items)
{
    const int nt = ld / 64, ntri = nt * (nt + 1) / 2;
    const long flat = xcd_flat((long)items * ntri);
    if (flat < 0) return;
    A += (flat / ntri) * sA;
    int ti, tj;
    tri_tile((int)(flat % ntri), ti, tj);
    __shared__ cx<T> t[64][33];
    for (int half = 0; half < 2; half++) {
        // columns 32 half .. + 31 of tile (ti, tj)
        for (int e = threadIdx.x; e < 2048; e += 256) {
            const int r = e >> 5, c = e & 31;
            t[r][c] = A[(long)(ti * 64 + r) * ld + tj * 64 + 32 * half + c];
        }
        __syncthreads();
        for (int e = threadIdx.x; e < 2048; e += 256) {
            const int c = e >> 6, r = e & 63;
            if (ti != tj || r > 32 * half + c)
                A[(long)(tj * 64 + 32 * half + c) * ld + ti * 64 + r] = t[r][c];
        }
        __syncthreads();
    }
}

// F = Z in T (tiles on and below the diagonal, zero past m), item 2 q the Z_L
// block of sample q, 2 q + 1 its Z_T block.
template <typename T>
__global__ __launch_bounds__(256) void k_nd_load(const c64* Z, long sZ, cx<T>* F, int ld, int m,
                                                  int items)
{
    const int nt = ld / 64, ntri = nt * (nt + 1) / 2;
    const long flat = xcd_flat((long)items * ntri);
    if (flat < 0) return;
    const long item = flat / ntri;
    int ti, tj;
    tri_tile((int)(flat % ntri), ti, tj);
    const c64* src = Z + (item >> 1) * sZ + (item & 1) * ((long)m * m + m);
    F += item * (long)ld * ld;
    for (int e = threadIdx.x; e < 4096; e += 256) {
        const int i = ti * 64 + (e >> 6), j = tj * 64 + (e & 63);
        cx<T> o{0, 0};
        if (i < m && j < m) {
            const c64 s = src[(long)i * m + j];
            o = cx<T>{(T)s.x, (T)s.y};
        }
        F[(long)i * ld + j] = o;
    }
}

// ---------------------------------------------------------------------------
// The node system
// ---------------------------------------------------------------------------
template <typename T>
struct NdArgs {
    int nb;
    long m, n, mp, np, N;
    const cx<T>* F;  // Y_L, Y_T (after the sweep)
    cx<T>* S;
    c64 *x, *r, *ysum, *dg, *cst;
    cx<T>*v, *z, *f, *y, *h, *c;
    const int *sn, *en, *node_ptr, *node_seg;
    int parts;
    const int *part, *root, *pseg_ptr, *pseg, *pnode_ptr, *pnode;  // see HemOp
    unsigned long long* norms;
    long snorm;
    const int* active;
    long inj;
};

__device__ inline c64 wave_sum(c64 a)
{
    for (int o = 32; o > 0; o >>= 1) {
        a.x += __shfl_xor(a.x, o);
        a.y += __shfl_xor(a.y, o);
    }
    return a;
}

// ysum_i = (Y_T 1)_i and the diagonal's share dg_i = 2 Y_L,ii + Y_T,ii / 2; one
// wave per row
template <typename T>
__global__ __launch_bounds__(256) void k_nd_rows(NdArgs<T> g)
{
    const long wg = (g.m + 3) / 4;
    const long item = blockIdx.x / wg, i = (blockIdx.x % wg) * 4 + (threadIdx.x >> 6);
    if (i >= g.m) return;
    const int lane = threadIdx.x & 63;
    const cx<T>* yl = g.F + 2 * item * g.mp * g.mp + i * g.mp;
    const cx<T>* yt = yl + g.mp * g.mp;
    c64 s{0, 0};
    for (long c = lane; c < g.m; c += 64) {
        s.x += yt[c].x;
        s.y += yt[c].y;
    }
    s = wave_sum(s);
    if (lane == 0) {
        g.ysum[item * g.m + i] = s;
        g.dg[item * g.m + i] = c64{2.0 * yl[i].x + 0.5 * yt[i].x, 2.0 * yl[i].y + 0.5 * yt[i].y};
    }
}

// sum over part j's segments of v, by a wave
template <typename T, typename V>
__device__ inline c64 nd_part_sum(const NdArgs<T>& g, int j, const V* v)
{
    c64 s{0, 0};
    for (int p = g.pseg_ptr[j] + (threadIdx.x & 63); p < g.pseg_ptr[j + 1]; p += 64) {
        const V a = v[g.pseg[p]];
        s = cadd(s, c64{a.x, a.y});
    }
    return wave_sum(s);
}

// The same with several parts: ysum's row j holds Y_T 1_j
template <typename T>
__global__ __launch_bounds__(256) void k_nd_part_rows(NdArgs<T> g)
{
    const long wg = (g.m + 3) / 4;
    const long item = blockIdx.x / wg, i = (blockIdx.x % wg) * 4 + (threadIdx.x >> 6);
    if (i >= g.m) return;
    const int lane = threadIdx.x & 63;
    const cx<T>* yl = g.F + 2 * item * g.mp * g.mp + i * g.mp;
    const cx<T>* yt = yl + g.mp * g.mp;
    for (int j = 0; j < g.parts; j++) {
        const c64 s = nd_part_sum(g, j, yt);
        if (lane == 0) g.ysum[(item * g.parts + j) * g.m + i] = s;
    }
    if (lane == 0)
        g.dg[item * g.m + i] = c64{2.0 * yl[i].x + 0.5 * yt[i].x, 2.0 * yl[i].y + 0.5 * yt[i].y};
}

// whether node u is the root of a part other than the first (parts > 1)
template <typename T>
__device__ inline bool nd_is_root(const NdArgs<T>& g, long u)
{
    const int j = g.part[u];
    return j > 0 && g.root[j] == u;
}

__device__ inline c64 wg_sum(c64 a, c64* red)
{
    a = wave_sum(a);
    const int nw = blockDim.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
    __syncthreads();
    c64 t{0, 0};
    for (int i = 0; i < nw; i++) t = cadd(t, red[i]);
    return t;
}

// tau, s and c of each item (one work-group)
template <typename T>
__global__ __launch_bounds__(1024) void k_nd_const(NdArgs<T> g)
{
    __shared__ c64 red[16];
    const long item = blockIdx.x;
    const c64 *ys = g.ysum + item * g.parts * g.m, *dg = g.dg + item * g.m;
    const bool multi = g.parts > 1;  // (then s, c and tau are the first part's)
    c64 a{0, 0}, d{0, 0};
    for (long i = threadIdx.x; i < g.m; i += 1024) {
        if (!multi || g.part[g.sn[i]] == 0) a = cadd(a, ys[i]);
        d = cadd(d, dg[i]);
    }
    a = wg_sum(a, red);
    d = wg_sum(d, red);
    if (threadIdx.x == 0) {
        const double s = 1.0 / ((double)g.n * (double)(multi ? g.pnode_ptr[1] : g.n));
        g.cst[4 * item] = c64{d.x * s, d.y * s};
        g.cst[4 * item + 1] = a;
    }
    for (long u = threadIdx.x; u < g.np; u += 1024) {
        c64 t{0, 0};
        if (multi && u < g.n && nd_is_root(g, u)) continue;
        if (u < g.n)
            for (int p = g.node_ptr[u]; p < g.node_ptr[u + 1]; p++)
                t = cadd(t, ys[g.node_seg[p] >> 1]);
        g.c[item * g.np + u] = cx<T>{(T)(0.5 * t.x), (T)(0.5 * t.y)};
    }
    for (int j = 1 + (threadIdx.x >> 6); j < g.parts; j += 16) {
        const c64 t = nd_part_sum(g, j, ys);
        if ((threadIdx.x & 63) == 0) g.c[item * g.np + g.root[j]] = cx<T>{(T)t.x, (T)t.y};
    }
}

// -S_p on and below the diagonal (zero past n): an entry of Y_L and of Y_T per
// pair of segment ends. 16 x 64 entries per work-group, a wave four rows: the
// rows' lists are scalar loads, a lane keeps the first two segments of its column
// (inside a conductor a node has two), and their four entries are loaded at once;
// a chain of list and entry loads per entry took 1.58 ms for 96 systems of 1221
// nodes, latency-bound.
template <typename T>
__global__ __launch_bounds__(256) void k_nd_schur(NdArgs<T> g)
{
    const int nt = (int)(g.np / 64), per = nt * (nt + 1) / 2 * 4;
    const long flat = xcd_flat((long)g.nb * per);
    if (flat < 0) return;
    const long item = flat / per;
    const int e = (int)(flat % per);
    int ti, tj;
    tri_tile(e >> 2, ti, tj);
    const int n = (int)g.n, w = tj * 64 + (threadIdx.x & 63);
    // (the wave's rows are uniform, so their lists are read by scalar loads)
    const int u0 = ti * 64 + (e & 3) * 16 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 4;
    const cx<T>* yl = g.F + 2 * item * g.mp * g.mp;
    const cx<T>* yt = yl + g.mp * g.mp;
    const c64 s0 = g.cst[4 * item];
    const bool first_part = g.parts == 1 || (w < n && g.part[w] == 0);
    int q0 = 0, q1 = 0, b0 = 0, b1 = 0;
    if (w < n) {
        q0 = g.node_ptr[w];
        q1 = g.node_ptr[w + 1];
        if (q1 > q0) b0 = g.node_seg[q0];
        b1 = q1 > q0 + 1 ? g.node_seg[q0 + 1] : b0;
    }
    const bool has0 = q1 > q0, has1 = q1 > q0 + 1;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int u = u0 + r;
        cx<T> o{0, 0};
        if (u < n) {
            c64 s = csel(first_part && (g.parts == 1 || g.part[u] == 0), s0, c64{0, 0});
            const int p1 = g.node_ptr[u + 1];
            for (int p = g.node_ptr[u]; p < p1; p++) {
                const int a = g.node_seg[p];
                const cx<T>* rl = yl + (a >> 1) * g.mp;
                const cx<T>* rt = yt + (a >> 1) * g.mp;
                auto add = [&](bool on, int b, cx<T> l, cx<T> t) {
                    const double sg = ((a ^ b) & 1) ? -1.0 : 1.0;
                    const c64 x{s.x + (sg * l.x + 0.25 * t.x), s.y + (sg * l.y + 0.25 * t.y)};
                    s = csel(on, x, s);
                };
                const cx<T> l0 = rl[b0 >> 1], t0 = rt[b0 >> 1], l1 = rl[b1 >> 1], t1 = rt[b1 >> 1];
                add(has0, b0, l0, t0);
                add(has1, b1, l1, t1);
                for (int q = q0 + 2; q < q1; q++) {
                    const int b = g.node_seg[q];
                    add(true, b, rl[b >> 1], rt[b >> 1]);
                }
            }
            if (w < n) o = cx<T>{(T)-s.x, (T)-s.y};
        }
        g.S[item * g.np * g.np + (long)u * g.np + w] = o;
    }
}

// Rows and columns of the other parts' roots (negated like the rest): one
// work-group per root. Of two roots the later node's work-group writes the entry.
template <typename T>
__global__ __launch_bounds__(256) void k_nd_roots(NdArgs<T> g)
{
    const long item = blockIdx.y;
    const int j = blockIdx.x + 1, r = g.root[j];
    const c64* ys = g.ysum + item * g.parts * g.m;
    cx<T>* S = g.S + item * g.np * g.np;
    ys += j * g.m;
    for (int u = threadIdx.x; u < g.n; u += 256) {
        if (nd_is_root(g, u)) continue;
        c64 s{0, 0};
        for (int p = g.node_ptr[u]; p < g.node_ptr[u + 1]; p++)
            s = cadd(s, ys[g.node_seg[p] >> 1]);
        S[(long)max(r, u) * g.np + min(r, u)] = cx<T>{(T)(-0.5 * s.x), (T)(-0.5 * s.y)};
    }
    for (int k = 1 + (threadIdx.x >> 6); k < g.parts; k += 4) {
        const int u = g.root[k];
        if (u > r) continue;
        const c64 s = nd_part_sum(g, k, ys);
        if ((threadIdx.x & 63) == 0) S[(long)r * g.np + u] = cx<T>{(T)-s.x, (T)-s.y};
    }
}

// out = M in for symmetric matrices, four rows per wave, 16 bytes per lane and
// row: HBM-bound (one read of M). BLK 2: the Y blocks of each item, with in /
// out of 2 mp values; BLK 1: the node inverse.
template <typename T, int BLK>
__device__ inline void nd_gemv_rows(const NdArgs<T>& g, const cx<T>* in, long item, int blk,
                                    long row0, cx<T> (&acc)[4])
{
    const long ld = BLK == 2 ? g.mp : g.np;
    const cx<T>* M = BLK == 2 ? g.F + (2 * item + blk) * ld * ld : g.S + item * ld * ld;
    const cx<T>* xv = in + (BLK == 2 ? (2 * item + blk) * ld : item * ld);
    constexpr int V = 16 / sizeof(cx<T>);
    struct alignas(16) Vec {
        cx<T> e[V];
    };
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q] = cx<T>{0, 0};
#pragma unroll 2
    for (long c = (long)lane * V; c < ld; c += 64 * V) {
        const Vec xx = *(const Vec*)(xv + c);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const Vec a = *(const Vec*)(M + (row0 + q) * ld + c);
#pragma unroll
            for (int e = 0; e < V; e++) {
                const cx<T> s = a.e[e], t = xx.e[e];
                acc[q].x = fma(s.x, t.x, fma(-s.y, t.y, acc[q].x));
                acc[q].y = fma(s.x, t.y, fma(s.y, t.x, acc[q].y));
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        for (int o = 32; o > 0; o >>= 1) {
            acc[q].x += __shfl_xor(acc[q].x, o);
            acc[q].y += __shfl_xor(acc[q].y, o);
        }
}

template <typename T, int BLK>
__global__ __launch_bounds__(256) void k_nd_gemv(NdArgs<T> g, const cx<T>* in, cx<T>* out)
{
    const long ld = BLK == 2 ? g.mp : g.np, wg = ld / 16;
    const long flat = xcd_flat((long)g.nb * BLK * wg);
    if (flat < 0) return;
    const long mat = flat / wg, item = mat / BLK;
    if (g.active && !g.active[item]) return;
    const long row0 = (flat % wg) * 16 + (threadIdx.x >> 6) * 4;
    cx<T> acc[4];
    nd_gemv_rows<T, BLK>(g, in, item, (int)(mat % BLK), row0, acc);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int q = 0; q < 4; q++) out[mat * ld + row0 + q] = acc[q];
    }
}

// 1 / (s - c^T h) (one work-group per item)
template <typename T>
__global__ __launch_bounds__(256) void k_nd_den(NdArgs<T> g)
{
    __shared__ c64 red[4];
    const long item = blockIdx.x;
    c64 a{0, 0};
    for (long u = threadIdx.x; u < g.n; u += 256) {
        const cx<T> c = g.c[item * g.np + u], h = g.h[item * g.np + u];
        a = cadd(a, cmul(c64{c.x, c.y}, c64{h.x, h.y}));
    }
    a = wg_sum(a, red);
    if (threadIdx.x == 0) g.cst[4 * item + 2] = crecip(csub(g.cst[4 * item + 1], a));
}

__device__ inline double nd_scale(const unsigned long long* rn, bool single)
{
    if (!single) return 1.0;
    const double s = __longlong_as_double((long long)*rn);
    return s > 0.0 ? s : 1.0;
}

// v = r_L, r_T (complex64: over |r|, so that the correction stays in range)
template <typename T>
__global__ __launch_bounds__(256) void k_nd_in(NdArgs<T> g, int kprev)
{
    const long item = blockIdx.y;
    if (g.active && !g.active[item]) return;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= 2 * g.m) return;
    const double s = 1.0 / nd_scale(g.norms + item * g.snorm + 4 * kprev, sizeof(T) == 4);
    const c64 r = g.r[item * g.N + i];
    const long o = i < g.m ? i : g.mp + i - g.m;
    g.v[2 * item * g.mp + o] = cx<T>{(T)(r.x * s), (T)(r.y * s)};
}

// f = r_U + A^T z_L + B^T z_T
template <typename T>
__global__ __launch_bounds__(256) void k_nd_node(NdArgs<T> g, int kprev)
{
    const long item = blockIdx.y;
    if (g.active && !g.active[item]) return;
    const long u = (long)blockIdx.x * 256 + threadIdx.x;
    if (u >= g.n) return;
    const double s = 1.0 / nd_scale(g.norms + item * g.snorm + 4 * kprev, sizeof(T) == 4);
    const c64 r = g.r[item * g.N + 2 * g.m + u];
    c64 t{r.x * s, r.y * s};
    const cx<T>* zl = g.z + 2 * item * g.mp;
    const cx<T>* zt = zl + g.mp;
    for (int p = g.node_ptr[u]; p < g.node_ptr[u + 1]; p++) {
        const int a = g.node_seg[p];
        const double sg = (a & 1) ? -1.0 : 1.0;
        t.x += sg * zl[a >> 1].x + 0.5 * zt[a >> 1].x;
        t.y += sg * zl[a >> 1].y + 0.5 * zt[a >> 1].y;
    }
    g.f[item * g.np + u] = cx<T>{(T)t.x, (T)t.y};
}

// f at the other parts' roots: the sums over the part of r_U and z_T; one wave per
// root
template <typename T>
__global__ __launch_bounds__(64) void k_nd_root_f(NdArgs<T> g, int kprev)
{
    const long item = blockIdx.y;
    if (g.active && !g.active[item]) return;
    const int j = blockIdx.x + 1;
    const double s = 1.0 / nd_scale(g.norms + item * g.snorm + 4 * kprev, sizeof(T) == 4);
    const c64* r = g.r + item * g.N + 2 * g.m;
    const cx<T>* zt = g.z + (2 * item + 1) * g.mp;
    c64 t{0, 0};
    for (int p = g.pnode_ptr[j] + threadIdx.x; p < g.pnode_ptr[j + 1]; p += 64)
        t = cadd(t, cscale(r[g.pnode[p]], s));
    t = cadd(wave_sum(t), nd_part_sum(g, j, zt));
    if (threadIdx.x == 0) g.f[item * g.np + g.root[j]] = cx<T>{(T)t.x, (T)t.y};
}

__device__ inline void dx_max(unsigned long long* p, unsigned long long a)
{
    a = wave_max(a);
    if ((threadIdx.x & 63) == 0) atomicMax(p, a);
}

// alpha and w (y is replaced by w), u += scale (w + alpha), and the segments'
// A w - r_L, B u - r_T into v; one work-group per item. first: r is the unit
// current at node inj, so f = e_inj, y is a row of the node inverse and r_L,
// r_T are zero. With several parts (MULTI) alpha is the first one's, every other
// part's constant is w at its root, and w counts as zero there; f = e_inj gains an
// entry at the root of inj's part.
template <typename T, bool MULTI>
__global__ __launch_bounds__(1024) void k_nd_alpha(NdArgs<T> g, int k, int first)
{
    __shared__ c64 red[16];
    const long item = blockIdx.x;
    if (g.active && !g.active[item]) return;
    const unsigned long long* rn = g.norms + item * g.snorm + 4 * (k - 1);
    const double scale = first ? 1.0 : nd_scale(rn, sizeof(T) == 4);
    cx<T>* y = g.y + item * g.np;
    const cx<T>*h = g.h + item * g.np, *c = g.c + item * g.np;
    const cx<T>* yin = first ? g.S + item * g.np * g.np + g.inj * g.np : y;
    const int jp = MULTI ? g.part[g.inj] : 0;  // inj's part
    // its root's row too, unless inj is the root
    const cx<T>* yr = MULTI && first && jp > 0 && g.root[jp] != g.inj
                          ? g.S + item * g.np * g.np + (long)g.root[jp] * g.np
                          : nullptr;
    auto y_at = [&](long u) {
        cx<T> v = yin[u];
        if (MULTI && yr) v = cadd(v, yr[u]);
        return v;
    };
    const c64* r = g.r + item * g.N;
    c64* x = g.x + item * g.N;
    c64 a{0, 0};
    for (long u = threadIdx.x; u < g.n; u += 1024) {
        const cx<T> cu = c[u], yu = y_at(u);
        a = csub(a, cmul(c64{cu.x, cu.y}, c64{yu.x, yu.y}));
        if (!first && (!MULTI || g.part[u] == 0))
            a = cadd(a, c64{r[2 * g.m + u].x / scale, r[2 * g.m + u].y / scale});
    }
    if (!first) {
        const cx<T>* zt = g.z + (2 * item + 1) * g.mp;
        for (long i = threadIdx.x; i < g.m; i += 1024)
            if (!MULTI || g.part[g.sn[i]] == 0) a = cadd(a, c64{zt[i].x, zt[i].y});
    }
    a = wg_sum(a, red);
    if (first && jp == 0) a.x += 1.0;
    const c64 al = cmul(a, g.cst[4 * item + 2]);
    unsigned long long dm = 0;
    for (long u = threadIdx.x; u < g.n; u += 1024) {
        const cx<T> hu = h[u], yu = y_at(u);
        const c64 w = csub(c64{yu.x, yu.y}, cmul(al, c64{hu.x, hu.y}));
        y[u] = cx<T>{(T)w.x, (T)w.y};
        if (MULTI) continue;
        const c64 d = cscale(cadd(w, al), scale);
        x[2 * g.m + u] = first ? d : cadd(x[2 * g.m + u], d);
        dm = max(dm, size_bits(sqrt(d.x * d.x + d.y * d.y)));
    }
    if (MULTI) __syncthreads();
    // the constant of node u's part, and w there
    auto const_at = [&](long u) {
        const int j = MULTI ? g.part[u] : 0;
        if (j == 0) return al;
        const cx<T> b = y[g.root[j]];
        return c64{b.x, b.y};
    };
    auto w_at = [&](long u) { return MULTI && nd_is_root(g, u) ? cx<T>{0, 0} : y[u]; };
    if (MULTI)
        for (long u = threadIdx.x; u < g.n; u += 1024) {
            const cx<T> w = w_at(u);
            const c64 d = cscale(cadd(c64{w.x, w.y}, const_at(u)), scale);
            x[2 * g.m + u] = first ? d : cadd(x[2 * g.m + u], d);
            dm = max(dm, size_bits(sqrt(d.x * d.x + d.y * d.y)));
        }
    dx_max(g.norms + item * g.snorm + 4 * k + 3, dm);
    __syncthreads();
    cx<T>* vl = g.v + 2 * item * g.mp;
    cx<T>* vt = vl + g.mp;
    const double inv = 1.0 / scale;
    for (long i = threadIdx.x; i < g.m; i += 1024) {
        const cx<T> ws = w_at(g.sn[i]), we = w_at(g.en[i]);
        const c64 b = const_at(g.sn[i]);
        c64 l{(double)ws.x - we.x, (double)ws.y - we.y};
        c64 t{0.5 * ((double)ws.x + we.x) + b.x, 0.5 * ((double)ws.y + we.y) + b.y};
        if (!first) {
            l = csub(l, cscale(r[i], inv));
            t = csub(t, cscale(r[g.m + i], inv));
        }
        vl[i] = cx<T>{(T)l.x, (T)l.y};
        vt[i] = cx<T>{(T)t.x, (T)t.y};
    }
}

// i_L, i_T += scale Y v
template <typename T>
__global__ __launch_bounds__(256) void k_nd_currents(NdArgs<T> g, int k, int first)
{
    const long wg = g.mp / 16;
    const long flat = xcd_flat((long)g.nb * 2 * wg);
    if (flat < 0) return;
    const long mat = flat / wg, item = mat >> 1;
    if (g.active && !g.active[item]) return;
    const long row0 = (flat % wg) * 16 + (threadIdx.x >> 6) * 4;
    if (row0 >= g.m) return;
    cx<T> acc[4];
    nd_gemv_rows<T, 2>(g, g.v, item, (int)(mat & 1), row0, acc);
    const int lane = threadIdx.x & 63;
    unsigned long long dm = 0;
    if (lane < 4 && row0 + lane < g.m) {
        const double s =
            first ? 1.0 : nd_scale(g.norms + item * g.snorm + 4 * (k - 1), sizeof(T) == 4);
        const cx<T> a = csel(lane < 2, csel(lane == 0, acc[0], acc[1]),
                             csel(lane == 2, acc[2], acc[3]));
        const c64 d{a.x * s, a.y * s};
        c64* xi = g.x + item * g.N + (mat & 1) * g.m + row0 + lane;
        *xi = first ? d : cadd(*xi, d);
        dm = size_bits(sqrt(d.x * d.x + d.y * d.y));
    }
    dx_max(g.norms + item * g.snorm + 4 * k + 3, dm);
}

// b = e_inj (unless null), zeroed norms, zero padding of the vectors
template <typename T>
__global__ __launch_bounds__(256) void k_nd_init(NdArgs<T> g, c64* b)
{
    const long item = blockIdx.y;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (b && i < g.N) b[item * g.N + i] = c64{i == 2 * g.m + g.inj ? 1.0 : 0.0, 0.0};
    if (i < g.snorm) g.norms[item * g.snorm + i] = 0;
    const cx<T> zero{0, 0};
    if (i < 2 * g.mp) g.v[2 * item * g.mp + i] = zero;
    if (i < g.np) g.f[item * g.np + i] = zero;
}

// What the host reads, written straight into its pinned copies (one launch in
// place of a gather and two copies of 4 us each)
template <typename T>
__global__ __launch_bounds__(256) void k_nd_pick(NdArgs<T> g, c64* u, unsigned long long* norms)
{
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q < g.nb) u[q] = g.x[q * g.N + 2 * g.m + g.inj];
    if (q < g.nb * g.snorm) norms[q] = g.norms[q];
}

// ---------------------------------------------------------------------------
// Small systems (at most 64 segments and 64 nodes) in one launch
// ---------------------------------------------------------------------------
__device__ inline void bits_max(unsigned long long& m, double a) { m = max(m, size_bits(a)); }

// Everything of a sample after the fill: both inverses (256 threads each), the
// node system, its inverse, and `spec` refinement steps, by one work-group, with
// the operations of the kernels above and the vectors in LDS. The blocks, S^-1
// and the vectors are left where those kernels take further steps from. As
// separate launches the same work is 25 of 4 to 6 us each beside two sweeps; here
// 59 us for one sample of 30 segments in complex128 (107 with a pivot at a time
// and the rows read again for every product), 64 for a hundred in complex64:
// chains of dependent steps.
template <typename T>
__global__ __launch_bounds__(512) void k_nd_small(NdArgs<T> g, const c64* Zall, long sZ, c64* ball,
                                                   int spec, c64* hu, unsigned long long* hnorms)
{
    const long item = blockIdx.x;
    const int t = threadIdx.x, grp = t >> 8;
    const int lane = t & 63, wave = (t & 255) >> 6, lr = lane & 15;
    const int m = (int)g.m, n = (int)g.n, N = (int)g.N;
    const c64* Z = Zall + item * sZ;
    const c64* Zg = Z + grp * (m * m + m);
    cx<T>* F = const_cast<cx<T>*>(g.F) + 2 * item * 4096;
    cx<T>* Fg = F + grp * 4096;
    cx<T>* S = g.S + item * 4096;
    c64 *xo = g.x + item * N, *ro = g.r + item * N;
    __shared__ NdSweep<T> sh[2];
    __shared__ cx<T> v[2][64], z[2][64], f[64], y[64], h[64], c[64];
    __shared__ c64 ys[64], dg[64], x[192], r[192], cst[3];
    __shared__ unsigned long long nrm[4 * 4];
    // the incidence lists, read many times by one lane after another
    __shared__ int nptr[65], nseg[128], end0[64], end1[64];
    if (t <= n) nptr[t] = g.node_ptr[t];
    if (t < 2 * m) nseg[t] = g.node_seg[t];
    if (t < m) {
        end0[t] = g.sn[t];
        end1[t] = g.en[t];
    }
    if (t < 16) nrm[t] = 0;
    if (t < 192) x[t] = c64{0, 0};
    if (t < 128) v[t >> 6][t & 63] = z[t >> 6][t & 63] = cx<T>{0, 0};
    if (t < 64) f[t] = y[t] = h[t] = c[t] = cx<T>{0, 0};
    // the matrix being inverted, 16 rows a wave in the layout of nd_sweep64
    cx<T> a[4][4];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                f(16 * wave + Mfma<T>::row(lane, v), 16 * j + lr, a[j][v]);
    };
    each([&](int p, int q, cx<T>& x) {
        x = cx<T>{0, 0};
        if (p < m && q < m) {
            const c64 s = Zg[max(p, q) * m + min(p, q)];
            x = cx<T>{(T)s.x, (T)s.y};
        }
    });
    nd_sweep64(a, sh[grp], m, wave, lane);
    each([&](int p, int q, cx<T>& x) { Fg[p * 64 + q] = p < m && q < m ? x : cx<T>{0, 0}; });
    __syncthreads();
    // four lanes per row of the own block from here on
    const int rw = (t & 255) >> 2, q4 = t & 3;
    if (grp == 1) {
        c64 s{0, 0};
#pragma unroll 4
        for (int k = q4; k < 64; k += 4) s = cadd(s, c64{Fg[rw * 64 + k].x, Fg[rw * 64 + k].y});
        for (int o = 2; o > 0; o >>= 1) s = cadd(s, c64{__shfl_xor(s.x, o), __shfl_xor(s.y, o)});
        if (q4 == 0) {
            const cx<T> l = F[rw * 65], u = Fg[rw * 65];
            ys[rw] = s;
            dg[rw] = c64{2.0 * l.x + 0.5 * u.x, 2.0 * l.y + 0.5 * u.y};
        }
    }
    __syncthreads();
    if (t < 64) {
        const c64 sa = wave_sum(t < m ? ys[t] : c64{0, 0}), sd = wave_sum(t < m ? dg[t] : c64{0, 0});
        if (t == 0) {
            const double w = 1.0 / ((double)n * (double)n);
            cst[0] = c64{sd.x * w, sd.y * w};
            cst[1] = sa;
        }
        if (t < n) {
            c64 s{0, 0};
            for (int p = nptr[t]; p < nptr[t + 1]; p++) s = cadd(s, ys[nseg[p] >> 1]);
            c[t] = cx<T>{(T)(0.5 * s.x), (T)(0.5 * s.y)};
        }
    }
    __syncthreads();
    // -S_p
    each([&](int p, int q, cx<T>& x) {
        const int u = max(p, q), w = min(p, q);
        x = cx<T>{0, 0};
        if (grp == 1 || u >= n) return;
        c64 s = cst[0];
        for (int i = nptr[u]; i < nptr[u + 1]; i++) {
            const int sa = nseg[i];
            for (int k = nptr[w]; k < nptr[w + 1]; k++) {
                const int sb = nseg[k];
                const double sg = ((sa ^ sb) & 1) ? -1.0 : 1.0;
                const cx<T> l = F[(sa >> 1) * 64 + (sb >> 1)];
                const cx<T> d = F[4096 + (sa >> 1) * 64 + (sb >> 1)];
                s.x += sg * l.x + 0.25 * d.x;
                s.y += sg * l.y + 0.25 * d.y;
            }
        }
        x = cx<T>{(T)-s.x, (T)-s.y};
    });
    nd_sweep64(a, sh[0], n, wave, lane, grp == 1);
    if (grp == 0)
        each([&](int p, int q, cx<T>& x) { S[p * 64 + q] = p < n && q < n ? x : cx<T>{0, 0}; });
    __syncthreads();
    // the four lanes' parts of row rw of the inverse and of the matrix (zero beyond
    // m; x is finite there)
    cx<T> fr[16];
    c64 zr[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int c = 4 * k + q4;
        fr[k] = Fg[rw * 64 + c];
        zr[k] = rw < m && c < m ? Zg[rw * m + c] : c64{0, 0};
    }
    auto gemv = [&](auto row, const cx<T>* in) {
        cx<T> s{0, 0};
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const cx<T> p = row(k), q = in[4 * k + q4];
            s.x = fma(p.x, q.x, fma(-p.y, q.y, s.x));
            s.y = fma(p.x, q.y, fma(p.y, q.x, s.y));
        }
        for (int o = 2; o > 0; o >>= 1) {
            s.x += __shfl_xor(s.x, o);
            s.y += __shfl_xor(s.y, o);
        }
        return s;
    };
    auto frow = [&](int k) { return fr[k]; };
    auto srow = [&](int k) { return S[rw * 64 + 4 * k + q4]; };
    {
        const cx<T> s = gemv(srow, c);
        if (grp == 0 && q4 == 0) h[rw] = s;
    }
    __syncthreads();
    if (t < 64) {
        c64 s{0, 0};
        if (t < n) s = cmul(c64{c[t].x, c[t].y}, c64{h[t].x, h[t].y});
        s = wave_sum(s);
        if (t == 0) cst[2] = crecip(csub(cst[1], s));
    }
    __syncthreads();
    for (int k = 1; k <= spec; k++) {
        const bool first = k == 1;
        const double scale = first ? 1.0 : nd_scale(&nrm[4 * (k - 1)], sizeof(T) == 4);
        const double inv = 1.0 / scale;
        unsigned long long nr = 0, nx = 0, na = 0, nd = 0;  // maxima of this thread
        if (first) {
            if (t < 64) y[t] = S[g.inj * 64 + t];
        } else {
            if ((t & 255) < m) {
                const c64 q = r[grp * m + (t & 255)];
                v[grp][t & 255] = cx<T>{(T)(q.x * inv), (T)(q.y * inv)};
            }
            __syncthreads();
            const cx<T> s = gemv(frow, v[grp]);
            if (q4 == 0) z[grp][rw] = s;
            __syncthreads();
            if (t < n) {
                c64 s{r[2 * m + t].x * inv, r[2 * m + t].y * inv};
                for (int p = nptr[t]; p < nptr[t + 1]; p++) {
                    const int sa = nseg[p];
                    const double sg = (sa & 1) ? -1.0 : 1.0;
                    s.x += sg * z[0][sa >> 1].x + 0.5 * z[1][sa >> 1].x;
                    s.y += sg * z[0][sa >> 1].y + 0.5 * z[1][sa >> 1].y;
                }
                f[t] = cx<T>{(T)s.x, (T)s.y};
            }
            __syncthreads();
            const cx<T> w = gemv(srow, f);
            if (grp == 0 && q4 == 0) y[rw] = w;
        }
        __syncthreads();
        // alpha (every wave alike), w and u
        c64 al{0, 0};
        {
            const int u = t & 63;
            if (u < n) {
                al = csub(al, cmul(c64{c[u].x, c[u].y}, c64{y[u].x, y[u].y}));
                if (!first) al = cadd(al, c64{r[2 * m + u].x / scale, r[2 * m + u].y / scale});
            }
            if (!first && u < m) al = cadd(al, c64{z[1][u].x, z[1][u].y});
            al = wave_sum(al);
            if (first) al.x += 1.0;
            al = cmul(al, cst[2]);
        }
        __syncthreads();
        if (t < n) {
            const c64 w = csub(c64{y[t].x, y[t].y}, cmul(al, c64{h[t].x, h[t].y}));
            y[t] = cx<T>{(T)w.x, (T)w.y};
            const c64 d = cscale(cadd(w, al), scale);
            x[2 * m + t] = first ? d : cadd(x[2 * m + t], d);
            bits_max(nd, sqrt(d.x * d.x + d.y * d.y));
        }
        __syncthreads();
        if ((t & 255) < m) {
            const int i = t & 255;
            const cx<T> ws = y[end0[i]], we = y[end1[i]];
            c64 l = grp ? c64{0.5 * ((double)ws.x + we.x) + al.x, 0.5 * ((double)ws.y + we.y) + al.y}
                        : c64{(double)ws.x - we.x, (double)ws.y - we.y};
            if (!first) l = csub(l, cscale(r[grp * m + i], inv));
            v[grp][i] = cx<T>{(T)l.x, (T)l.y};
        }
        __syncthreads();
        {
            const cx<T> s = gemv(frow, v[grp]);
            if (q4 == 0 && rw < m) {
                const c64 d{s.x * scale, s.y * scale};
                c64* xi = &x[grp * m + rw];
                *xi = first ? d : cadd(*xi, d);
                bits_max(nd, sqrt(d.x * d.x + d.y * d.y));
            }
        }
        __syncthreads();
        // r = b - W x, in double-double as k_hem_apply
        if (rw < m) {
            DD sx{0, 0}, sy{0, 0};
            double ta = 0;
#pragma unroll
            for (int k4 = 0; k4 < 16; k4++) {
                const c64 p = zr[k4], q = x[grp * m + 4 * k4 + q4];
                dd_mac(sx, p.x, q.x);
                dd_mac(sx, -p.y, q.y);
                dd_mac(sy, p.x, q.y);
                dd_mac(sy, p.y, q.x);
                if (first) ta += sqrt(p.x * p.x + p.y * p.y);
            }
            for (int o = 2; o > 0; o >>= 1) {
                sx = dd_plus(sx, dd_shfl_xor(sx, o));
                sy = dd_plus(sy, dd_shfl_xor(sy, o));
                ta += __shfl_xor(ta, o);
            }
            if (q4 == 0) {
                const c64 xs = x[2 * m + end0[rw]], xe = x[2 * m + end1[rw]];
                const double cs = grp ? 0.5 : 1.0, ce = grp ? 0.5 : -1.0;
                dd_add(sx, cs * xs.x);
                dd_add(sy, cs * xs.y);
                dd_add(sx, ce * xe.x);
                dd_add(sy, ce * xe.y);
                const int i = grp * m + rw;
                const c64 rr{dd_sub_from(0.0, sx), dd_sub_from(0.0, sy)};
                r[i] = rr;
                bits_max(nr, sqrt(rr.x * rr.x + rr.y * rr.y));
                bits_max(nx, sqrt(x[i].x * x[i].x + x[i].y * x[i].y));
                if (first) bits_max(na, ta + 2.0 * cs);
            }
        }
        if (t < n) {
            DD sx{0, 0}, sy{0, 0};
            double ta = 0;
            for (int p = nptr[t]; p < nptr[t + 1]; p++) {
                const int sa = nseg[p];
                const double cl = (sa & 1) ? -1.0 : 1.0;
                const c64 xl = x[sa >> 1], xt = x[m + (sa >> 1)];
                dd_add(sx, cl * xl.x);
                dd_add(sx, 0.5 * xt.x);
                dd_add(sy, cl * xl.y);
                dd_add(sy, 0.5 * xt.y);
                ta += 1.5;
            }
            const int i = 2 * m + t;
            const c64 rr{dd_sub_from(t == g.inj ? 1.0 : 0.0, sx), dd_sub_from(0.0, sy)};
            r[i] = rr;
            bits_max(nr, sqrt(rr.x * rr.x + rr.y * rr.y));
            bits_max(nx, sqrt(x[i].x * x[i].x + x[i].y * x[i].y));
            if (first) bits_max(na, ta);
        }
        for (int o = 32; o > 0; o >>= 1) {
            nr = max(nr, __shfl_xor(nr, o));
            nx = max(nx, __shfl_xor(nx, o));
            nd = max(nd, __shfl_xor(nd, o));
            if (first) na = max(na, __shfl_xor(na, o));
        }
        if ((t & 63) == 0) {
            atomicMax(&nrm[4 * k], nr);
            atomicMax(&nrm[4 * k + 1], nx);
            atomicMax(&nrm[4 * k + 2], na);
            atomicMax(&nrm[4 * k + 3], nd);
        }
        __syncthreads();
    }
    // what further steps start from
    for (int i = t; i < N; i += 512) {
        xo[i] = x[i];
        ro[i] = r[i];
        ball[item * N + i] = c64{i == 2 * m + g.inj ? 1.0 : 0.0, 0.0};
    }
    for (int i = t; i < g.snorm; i += 512) {
        const unsigned long long v = i < 4 * (spec + 1) ? nrm[i] : 0;
        g.norms[item * g.snorm + i] = v;
        hnorms[item * g.snorm + i] = v;
    }
    if (t == 0) hu[item] = x[2 * m + g.inj];
    if (t < 128) g.v[128 * item + t] = v[t >> 6][t & 63];
    if (t < 64) {
        g.f[64 * item + t] = f[t];
        g.h[64 * item + t] = h[t];
        g.c[64 * item + t] = c[t];
    }
    if (t < 3) g.cst[4 * item + t] = cst[t];
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
// Columns per sweep step. A step reads and writes every tile once, which at 64
// columns takes as long as its MFMAs; more blocks per step cost the panels'
// products with the step's earlier blocks. In complex64 256 columns win from
// order 300 on (200 samples of order 400: 5.39 against 5.71 ms with 128; 96 of
// order 1320: 38.1 against 40.6 ms); complex128, whose products take four times
// as long per byte, gains nothing past 128.
constexpr long kWide = 300;
static int nd_block(long dim, bool f64)
{
    if (dim <= 128) return 64;
    return !f64 && dim >= kWide ? 256 : 128;
}
static long up(long v, long a) { return (v + a - 1) / a * a; }

template <typename T>
size_t NodalSolver::partition(char* base, int batch)
{
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* p = base + off;
        off += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const size_t B = (size_t)batch, e = sizeof(cx<T>);
    const bool d = sizeof(T) == 8;
    const long bz = nd_block(m, d), bs = nd_block(n, d);
    const size_t panel = std::max(2 * (size_t)mp * bz, (size_t)np * bs);
    const size_t diag = 64 * (size_t)std::max(2 * bz, bs);
    sZ = nodal_z_items(m);
    Z = (c64*)take(sizeof(c64) * sZ * B);
    F = take(e * 2 * mp * mp * B);
    S = take(e * np * np * B);
    tp = take(e * panel * B);
    op_ = take(e * panel * B);
    P = take(e * diag * B);
    x = (c64*)take(sizeof(c64) * N * B);
    r = (c64*)take(sizeof(c64) * N * B);
    b = (c64*)take(sizeof(c64) * N * B);
    ysum = (c64*)take(sizeof(c64) * m * op.parts * B);
    dg = (c64*)take(sizeof(c64) * m * B);
    cst = (c64*)take(sizeof(c64) * 4 * B);
    v = take(e * 2 * mp * B);
    z = take(e * 2 * mp * B);
    f = take(e * np * B);
    y = take(e * np * B);
    h = take(e * np * B);
    c = take(e * np * B);
    norms = (unsigned long long*)take(sizeof(unsigned long long) * kNormStride * B);
    active = (int*)take(sizeof(int) * B);
    return off;
}

size_t NodalSolver::bytes(long m_, long n_, int parts, bool f64_, int batch)
{
    NodalSolver t;
    t.op.parts = parts;
    t.m = m_;
    t.n = n_;
    t.N = n_ + 2 * m_;
    t.mp = up(m_, 64);
    t.np = up(n_, 64);
    return f64_ ? t.partition<double>(nullptr, batch) : t.partition<float>(nullptr, batch);
}

int NodalSolver::ensure(const HemOp& hem, bool f64_, int batch)
{
    if (batch < 1 || hem.m < 1 || hem.n < 1) return TAGS_ERR_ARG;
    op = hem;
    op.zl_off = 0;
    op.zt_off = hem.m;
    op.node_off = 2 * hem.m;
    m = hem.m;
    n = hem.n;
    N = n + 2 * m;
    mp = up(m, 64);
    np = up(n, 64);
    f64 = f64_;
    const size_t need = bytes(m, n, op.parts, f64, batch);
    if (need > arena_bytes) {
        hipFree(arena);
        arena = nullptr;
        arena_bytes = 0;
        TAGS_HIP(dev_malloc((void**)&arena, need));
        arena_bytes = need;
    }
    if (f64) partition<double>(arena, batch);
    else partition<float>(arena, batch);
    if (batch > host_cap) {
        if (hnorms) hipHostFree(hnorms);
        if (hu) hipHostFree(hu);
        if (hactive) hipHostFree(hactive);
        hnorms = nullptr;
        hu = nullptr;
        hactive = nullptr;
        host_cap = 0;
        TAGS_HIP(hipHostMalloc(&hnorms, sizeof(unsigned long long) * kNormStride * batch, 0));
        TAGS_HIP(hipHostMalloc(&hu, sizeof(c64) * batch, 0));
        TAGS_HIP(hipHostMalloc(&hactive, sizeof(int) * batch, 0));
        host_cap = batch;
    }
    cap = batch;
    return 0;
}

void NodalSolver::release()
{
    hipFree(arena);
    if (hnorms) hipHostFree(hnorms);
    if (hu) hipHostFree(hu);
    if (hactive) hipHostFree(hactive);
    arena = nullptr;
    hnorms = nullptr;
    hu = nullptr;
    hactive = nullptr;
    arena_bytes = 0;
    host_cap = cap = 0;
}

template <typename T>
static NdArgs<T> nd_args(NodalSolver& s, bool masked)
{
    NdArgs<T> g;
    g.nb = s.nb;
    g.m = s.m;
    g.n = s.n;
    g.mp = s.mp;
    g.np = s.np;
    g.N = s.N;
    g.F = (const cx<T>*)s.F;
    g.S = (cx<T>*)s.S;
    g.x = s.x;
    g.r = s.r;
    g.ysum = s.ysum;
    g.dg = s.dg;
    g.cst = s.cst;
    g.v = (cx<T>*)s.v;
    g.z = (cx<T>*)s.z;
    g.f = (cx<T>*)s.f;
    g.y = (cx<T>*)s.y;
    g.h = (cx<T>*)s.h;
    g.c = (cx<T>*)s.c;
    g.sn = s.op.sn;
    g.en = s.op.en;
    g.node_ptr = s.op.node_ptr;
    g.node_seg = s.op.node_seg;
    g.parts = s.parts;
    g.part = s.op.part;
    g.root = s.op.root;
    g.pseg_ptr = s.op.pseg_ptr;
    g.pseg = s.op.pseg;
    g.pnode_ptr = s.op.pnode_ptr;
    g.pnode = s.op.pnode;
    g.norms = s.norms;
    g.snorm = NodalSolver::kNormStride;
    g.active = masked ? s.active : nullptr;
    g.inj = s.inj;
    return g;
}

// A = -A^-1 for every item of the phase, then both triangles
template <typename T, int NB>
static int nd_sweep(const NdPhase<T>& p, hipStream_t st, Profiler* pr)
{
    const long nt = p.ld / 64, ntri = nt * (nt + 1) / 2;
    if (nt == 1) {
        Timed tm(pr, FAM_PANEL, st);
        hipLaunchKernelGGL((k_nd_diag<T, NB>), dim3(p.items), dim3(256), 0, st, p, 0, 0, 1);
        tm.end();
        TAGS_HIP(hipGetLastError());
        return 0;
    }
    for (int c0 = 0; c0 < p.dim; c0 += NB) {
        const int nq = (int)std::min<long>(NB / 64, nt - c0 / 64);
        {
            Timed tm(pr, FAM_PANEL, st);
            for (int t = 0; t < nq; t++) {
                hipLaunchKernelGGL((k_nd_diag<T, NB>), dim3(p.items), dim3(256), 0, st, p, c0, t,
                                   0);
                hipLaunchKernelGGL((k_nd_panel<T, NB>), dim3(xcd_grid(p.items * nt)), dim3(256), 0,
                                   st, p, c0, t);
            }
            tm.end();
        }
        Timed tm(pr, FAM_GEMM, st);
        const double d = p.dim, w = std::min(NB, p.dim - c0);
        hipLaunchKernelGGL((k_nd_update<T, NB>), dim3(xcd_grid(p.items * ntri)), dim3(256), 0, st,
                           p, c0);
        tm.end(4.0 * d * d * w * p.items, true);
    }
    hipLaunchKernelGGL(k_nd_mirror<T>, dim3(xcd_grid(p.items * ntri)), dim3(256), 0, st, p.A, p.sA,
                       p.ld, p.items);
    TAGS_HIP(hipGetLastError());
    return 0;
}

template <typename T>
static int nd_invert(const NdPhase<T>& p, int nb, hipStream_t st, Profiler* pr)
{
    if constexpr (sizeof(T) == 4) {
        if (nb == 256) return nd_sweep<T, 256>(p, st, pr);
    }
    return nb == 128 ? nd_sweep<T, 128>(p, st, pr) : nd_sweep<T, 64>(p, st, pr);
}

template <typename T>
int NodalSolver::factor()
{
    const NdArgs<T> g = nd_args<T>(*this, false);
    const long nt = mp / 64, ntri = nt * (nt + 1) / 2;
    {
        Timed tm(pr, FAM_OTHER, st);
        hipLaunchKernelGGL(k_nd_load<T>, dim3(xcd_grid(2L * nb * ntri)), dim3(256), 0, st, Z, sZ,
                           (cx<T>*)F, (int)mp, (int)m, 2 * nb);
        tm.end();
    }
    int rc;
    const int bz = nd_block(m, f64), bs = nd_block(n, f64);
    const NdPhase<T> pz{(cx<T>*)F,   mp * mp, (int)mp,   (int)m,     2 * nb,     (cx<T>*)tp,
                        (cx<T>*)op_, mp * bz, (cx<T>*)P};
    if ((rc = nd_invert<T>(pz, bz, st, pr))) return rc;
    {
        Timed tm(pr, FAM_OTHER, st);
        const bool multi = parts > 1;
        const dim3 gr((unsigned)(nb * ((m + 3) / 4)));
        if (multi) hipLaunchKernelGGL(k_nd_part_rows<T>, gr, dim3(256), 0, st, g);
        else hipLaunchKernelGGL(k_nd_rows<T>, gr, dim3(256), 0, st, g);
        hipLaunchKernelGGL(k_nd_const<T>, dim3(nb), dim3(1024), 0, st, g);
        const long n64 = np / 64;
        hipLaunchKernelGGL(k_nd_schur<T>, dim3(xcd_grid((long)nb * (n64 * (n64 + 1) / 2 * 4))),
                           dim3(256), 0, st, g);
        if (multi)
            hipLaunchKernelGGL(k_nd_roots<T>, dim3(parts - 1, nb), dim3(256), 0, st, g);
        tm.end();
    }
    const NdPhase<T> ps{(cx<T>*)S,   np * np, (int)np,   (int)n,     nb,         (cx<T>*)tp,
                        (cx<T>*)op_, np * bs, (cx<T>*)P};
    if ((rc = nd_invert<T>(ps, bs, st, pr))) return rc;
    hipLaunchKernelGGL((k_nd_gemv<T, 1>), dim3(xcd_grid(nb * (np / 16))), dim3(256), 0, st, g,
                       (const cx<T>*)g.c, g.h);
    hipLaunchKernelGGL(k_nd_den<T>, dim3(nb), dim3(256), 0, st, g);
    TAGS_HIP(hipGetLastError());
    return 0;
}

template <typename T>
int NodalSolver::queue_step(int k, bool masked)
{
    const NdArgs<T> g = nd_args<T>(*this, masked);
    const int first = k == 1 && unit_;
    const unsigned gm = (unsigned)((2 * m + 255) / 256), gn = (unsigned)((n + 255) / 256);
    const unsigned gz = xcd_grid(2L * nb * (mp / 16));
    {
        Timed tm(pr, FAM_SOLVE, st);
        if (!first) {
            hipLaunchKernelGGL(k_nd_in<T>, dim3(gm, nb), dim3(256), 0, st, g, k - 1);
            hipLaunchKernelGGL((k_nd_gemv<T, 2>), dim3(gz), dim3(256), 0, st, g,
                               (const cx<T>*)g.v, g.z);
            hipLaunchKernelGGL(k_nd_node<T>, dim3(gn, nb), dim3(256), 0, st, g, k - 1);
            if (parts > 1)
                hipLaunchKernelGGL(k_nd_root_f<T>, dim3(parts - 1, nb), dim3(64), 0, st, g, k - 1);
            hipLaunchKernelGGL((k_nd_gemv<T, 1>), dim3(xcd_grid(nb * (np / 16))), dim3(256), 0, st,
                               g, (const cx<T>*)g.f, g.y);
        }
        if (parts > 1)
            hipLaunchKernelGGL((k_nd_alpha<T, true>), dim3(nb), dim3(1024), 0, st, g, k, first);
        else
            hipLaunchKernelGGL((k_nd_alpha<T, false>), dim3(nb), dim3(1024), 0, st, g, k, first);
        hipLaunchKernelGGL(k_nd_currents<T>, dim3(gz), dim3(256), 0, st, g, k, first);
        TAGS_HIP(hipGetLastError());
        tm.end();
    }
    Timed tm(pr, FAM_RESID, st);
    // |W| comes with the first residual
    const int rc = hem_apply(Z, m, op, x, N, b, r, N, norms + 4 * k, kNormStride, k == 1 ? 2 : 1,
                             nb, sZ, masked ? active : nullptr, st);
    tm.end();
    return rc;
}

int NodalSolver::issue(int nb_, long inj_)
{
    if (nb_ < 1 || nb_ > cap || inj_ < 0 || inj_ >= n) return TAGS_ERR_ARG;
    nb = nb_;
    inj = inj_;
    unit_ = true;
    // (in complex128 a small system of several parts is taken as one: its steps
    // still contract by 1e-9, and one launch does it. 54 segments in two parts, 200
    // samples: 0.39 ms, 0.53 told apart)
    const bool small = m <= 64 && n <= 64 && (op.parts == 1 || f64);
    parts = small ? 1 : op.parts;
    if (small) {
        step_ = f64 ? kSpec64 : kSpec32;
        Timed tm(pr, FAM_SOLVE, st);
        if (f64)
            hipLaunchKernelGGL(k_nd_small<double>, dim3(nb), dim3(512), 0, st,
                               nd_args<double>(*this, false), (const c64*)Z, sZ, b, step_, hu,
                               hnorms);
        else
            hipLaunchKernelGGL(k_nd_small<float>, dim3(nb), dim3(512), 0, st,
                               nd_args<float>(*this, false), (const c64*)Z, sZ, b, step_, hu,
                               hnorms);
        TAGS_HIP(hipGetLastError());
        tm.end();
        first_ = true;
        return 0;
    }
    const long w = std::max(std::max(N, 2 * mp), std::max(np, kNormStride));
    const dim3 gi((unsigned)((w + 255) / 256), nb);
    if (f64) hipLaunchKernelGGL(k_nd_init<double>, gi, dim3(256), 0, st, nd_args<double>(*this, false), b);
    else hipLaunchKernelGGL(k_nd_init<float>, gi, dim3(256), 0, st, nd_args<float>(*this, false), b);
    TAGS_HIP(hipGetLastError());
    return queue_spec();
}

int NodalSolver::issue_rhs()
{
    if (!f64 || cap < 1) return TAGS_ERR_ARG;
    nb = 1;
    inj = 0;
    parts = op.parts;
    const long w = std::max(std::max(N, 2 * mp), std::max(np, kNormStride));
    hipLaunchKernelGGL(k_nd_init<double>, dim3((unsigned)((w + 255) / 256)), dim3(256), 0, st,
                       nd_args<double>(*this, false), (c64*)nullptr);
    TAGS_HIP(hipGetLastError());
    TAGS_HIP(hipMemcpyAsync(r, b, sizeof(c64) * N, hipMemcpyDeviceToDevice, st));
    int rc = fill_c64(x, N, c64{0.0, 0.0}, st);
    if (rc) return rc;
    unit_ = false;
    return queue_spec();
}

// the factors, the first steps and their results
int NodalSolver::queue_spec()
{
    int rc = f64 ? factor<double>() : factor<float>();
    if (rc) return rc;
    step_ = f64 ? kSpec64 : kSpec32;
    for (int k = 1; k <= step_; k++)
        if ((rc = f64 ? queue_step<double>(k, false) : queue_step<float>(k, false))) return rc;
    first_ = true;
    return queue_results();
}

int NodalSolver::queue_results()
{
    const dim3 g((unsigned)(((long)nb * kNormStride + 255) / 256));
    if (f64)
        hipLaunchKernelGGL(k_nd_pick<double>, g, dim3(256), 0, st, nd_args<double>(*this, false),
                           hu, hnorms);
    else
        hipLaunchKernelGGL(k_nd_pick<float>, g, dim3(256), 0, st, nd_args<float>(*this, false), hu,
                           hnorms);
    TAGS_HIP(hipGetLastError());
    return 0;
}

double NodalSolver::norm_at(int q, int k, int i) const
{
    double d;
    std::memcpy(&d, &hnorms[kNormStride * q + 4 * k + i], 8);
    return d;
}
double NodalSolver::berr_at(int q, int k) const
{
    const double w = norm_at(q, 1, 2), rn = norm_at(q, k, 0), xn = norm_at(q, k, 1);
    if (rn == 0.0 && xn > 0.0) return 0.0;
    return w > 0 && xn > 0 ? rn / (w * xn) : NAN;
}
double NodalSolver::dx_at(int q, int k) const
{
    const double d = norm_at(q, k, 3), xn = norm_at(q, k, 1);
    return xn > 0 ? d / xn : NAN;
}
// rho / (1 - rho) |dx| / |x| with rho the last step's contraction; |dx| / |x|
// itself at the first step and where rho >= 1/2
double NodalSolver::fwd_at(int q, int k) const
{
    const double d = dx_at(q, k);
    if (k < 2 || d == 0.0) return d;
    const double dp = dx_at(q, k - 1), rho = dp > 0.0 ? d / dp : 1.0;
    return rho < 0.5 ? d * rho / (1.0 - rho) : d;
}
// Acceptance: backward error of a few ulps, and the error left in x below
// 1e-10 (complex64 blocks: 100 x below the 1e-8 bar) or 1e-14 (complex128: the
// level of a direct FP64 factorisation or better).
bool NodalSolver::accept(int q) const
{
    return berr[q] <= 1e-15 && fwd[q] <= (f64 ? 1e-14 : 1e-10);
}

int NodalSolver::advance(bool* complete)
{
    *complete = false;
    const int k = first_ ? step_ : ++step_;
    if (first_) {
        steps.assign(nb, k);
        accepted.assign(nb, 0);
        go.assign(nb, 1);
        berr.assign(nb, 0.0);
        fwd.assign(nb, 0.0);
        hist.assign(8 * (size_t)nb, -1.0);
        for (int q = 0; q < nb; q++)
            for (int i = 1; i < k; i++) hist[8 * q + i - 1] = berr_at(q, i);
    }
    first_ = false;
    int ngo = 0;
    for (int q = 0; q < nb; q++) {
        if (!go[q]) continue;
        steps[q] = k;
        berr[q] = berr_at(q, k);
        fwd[q] = fwd_at(q, k);
        if (k <= 8) hist[8 * q + k - 1] = berr[q];
        accepted[q] = accept(q);
        // on while a step still gains 20 % in either measure
        go[q] = !accepted[q] && k < kMaxSteps && berr[q] == berr[q] && fwd[q] == fwd[q] &&
                (k < 3 || berr[q] <= 0.8 * berr_at(q, k - 1) || dx_at(q, k) <= 0.8 * dx_at(q, k - 1));
        ngo += go[q];
    }
    if (ngo == 0) {
        *complete = true;
        return 0;
    }
    for (int q = 0; q < nb; q++) hactive[q] = go[q];
    TAGS_HIP(hipMemcpyAsync(active, hactive, sizeof(int) * nb, hipMemcpyHostToDevice, st));
    int rc = f64 ? queue_step<double>(k + 1, true) : queue_step<float>(k + 1, true);
    return rc ? rc : queue_results();
}

// ---------------------------------------------------------------------------
// Dense symmetric inverses and the structure of a host immittance matrix
// ---------------------------------------------------------------------------
// A = -src (upper triangle, row-major) on 64 x 64 tiles on and below the
// diagonal, transposed through LDS, zero beyond dim
__global__ __launch_bounds__(256) void k_sym_load(const c64* src, long lds, long ssrc, c64* A,
                                                   int ld, int dim, int items)
{
    const int nt = ld / 64, ntri = nt * (nt + 1) / 2;
    const long flat = xcd_flat((long)items * ntri);
    if (flat < 0) return;
    const long item = flat / ntri;
    int ti, tj;
    tri_tile((int)(flat % ntri), ti, tj);
    src += item * ssrc;
    A += item * (long)ld * ld;
    __shared__ c64 t[32][65];
    for (int half = 0; half < 2; half++) {
        for (int e = threadIdx.x; e < 2048; e += 256) {
            const int c = e >> 6, r = e & 63;
            const int i = ti * 64 + r, j = tj * 64 + 32 * half + c;
            c64 v{0, 0};
            if (i < dim && j < dim) v = src[(long)min(i, j) * lds + max(i, j)];
            t[c][r] = c64{-v.x, -v.y};
        }
        __syncthreads();
        for (int e = threadIdx.x; e < 2048; e += 256) {
            const int r = e >> 5, c = e & 31;
            A[(long)(ti * 64 + r) * ld + tj * 64 + 32 * half + c] = t[c][r];
        }
        __syncthreads();
    }
}

size_t sym_inverse_bytes(long dim, int items)
{
    const size_t ld = (size_t)up(dim, 64), nb = (size_t)nd_block(dim, true);
    return sizeof(c64) * (size_t)items * (2 * ld * nb + 64 * nb) + 1024;
}

int sym_inverse(const c64* src, long lds, long ssrc, c64* X, long dim, int items, char* work,
                hipStream_t st)
{
    if (dim < 1 || dim >= 65536 || items < 1) return TAGS_ERR_ARG;
    const long ld = up(dim, 64), nt = ld / 64;
    const int nb = nd_block(dim, true);
    hipLaunchKernelGGL(k_sym_load, dim3(xcd_grid(items * (nt * (nt + 1) / 2))), dim3(256), 0, st,
                       src, lds, ssrc, X, (int)ld, (int)dim, items);
    TAGS_HIP(hipGetLastError());
    c64* tp = (c64*)work;
    c64* op = tp + (size_t)items * ld * nb;
    c64* P = op + (size_t)items * ld * nb;
    const NdPhase<double> p{X, ld * ld, (int)ld, (int)dim, items, tp, op, ld * nb, P};
    return nd_invert<double>(p, nb, st, nullptr);
}

__global__ __launch_bounds__(256) void k_sym_apply(const c64* X, long ld, long n, const c64* r,
                                                    c64* x, unsigned long long* dmax)
{
    const long i = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    const int lane = threadIdx.x & 63;
    c64 s{0, 0};
    for (long c = lane; c < n; c += 64) s = cadd(s, cmul(X[i * ld + c], r[c]));
    s = wave_sum(s);
    if (lane) return;
    x[i] = cadd(x[i], s);
    atomicMax(dmax, (unsigned long long)__double_as_longlong(sqrt(s.x * s.x + s.y * s.y)));
}
int sym_apply(const c64* X, long ld, long n, const c64* r, c64* x, unsigned long long* dmax,
              hipStream_t st)
{
    hipLaunchKernelGGL(k_sym_apply, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, X, ld, n, r, x,
                       dmax);
    TAGS_HIP(hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void k_sub_identity(c64* R, long m, long total,
                                                       unsigned long long* dmax)
{
    unsigned long long a = 0;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
        const long q = e % (m * m);
        c64 v = R[e];
        if (q % (m + 1) == 0) {
            v.x -= 1.0;
            R[e] = v;
        }
        a = max(a, size_bits(fabs(v.x) + fabs(v.y)));
    }
    a = wave_max(a);
    if ((threadIdx.x & 63) == 0) atomicMax(dmax, a);
}
int sub_identity(c64* R, long m, int items, unsigned long long* dmax, hipStream_t st)
{
    const long total = m * m * items;
    hipLaunchKernelGGL(k_sub_identity, dim3((unsigned)std::min((total + 255) / 256, 1024L)),
                       dim3(256), 0, st, R, m, total, dmax);
    TAGS_HIP(hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void k_sym_pack(const c64* X, long ld, long m, c64* out)
{
    X += blockIdx.z * ld * ld;
    out += blockIdx.z * (m * (m + 1) / 2);
    for (long i = blockIdx.y; i < m; i += gridDim.y) {
        const long o = i * m - i * (i - 1) / 2 - i;
        for (long k = i + (long)blockIdx.x * 256 + threadIdx.x; k < m; k += (long)gridDim.x * 256)
            out[o + k] = X[i * ld + k];
    }
}
int sym_pack(const c64* X, long ld, long m, int items, c64* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_sym_pack, dim3((unsigned)std::min((m + 255) / 256, 16L),
                                        (unsigned)std::min(m, 16384L), (unsigned)items),
                       dim3(256), 0, st, X, ld, m, out);
    TAGS_HIP(hipGetLastError());
    return 0;
}

// row (column of the caller's array) c of W, entries r >= c
__global__ __launch_bounds__(256) void k_imm_structure(const c64* W, long N, long m, long n,
                                                        int* out)
{
    int *sn = out, *en = out + m, *cnt = out + 2 * m, *bad = out + 4 * m;
    int wrong = 0;
    for (long c = blockIdx.y; c < n + m; c += gridDim.y)
        for (long r = c + (long)blockIdx.x * 256 + threadIdx.x; r < N; r += (long)gridDim.x * 256) {
            if (c >= n && r < n + m) continue;  // Z_L
            const c64 v = W[c * N + r];
            if (r < n || c >= n || r >= n + m) {
                if (c < n && r >= n + m) {
                    // B: 1/2 exactly where A is not zero
                    const c64 a = W[c * N + r - m];
                    wrong += v.y != 0.0 || v.x != (a.x != 0.0 ? 0.5 : 0.0);
                } else {
                    wrong += v.x != 0.0 || v.y != 0.0;
                }
            } else if (v.x != 0.0 || v.y != 0.0) {
                // A: +1 at the start node, -1 at the end node
                const long s = r - n;
                if (v.y == 0.0 && v.x == 1.0) {
                    sn[s] = (int)c;
                    atomicAdd(&cnt[s], 1);
                } else if (v.y == 0.0 && v.x == -1.0) {
                    en[s] = (int)c;
                    atomicAdd(&cnt[m + s], 1);
                } else {
                    wrong++;
                }
            }
        }
    // (NaN entries compare unequal to everything and count as wrong)
    if (wrong) atomicAdd(bad, wrong);
}
__global__ void k_int_zero(int* p, long n)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}
int imm_structure(const c64* W, long N, long m, long n, int* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_int_zero, dim3((unsigned)((4 * m + 256) / 256)), dim3(256), 0, st, out,
                       4 * m + 1);
    hipLaunchKernelGGL(k_imm_structure, dim3((unsigned)std::min((N + 255) / 256, 16L),
                                             (unsigned)std::min(n + m, 8192L)),
                       dim3(256), 0, st, W, N, m, n, out);
    TAGS_HIP(hipGetLastError());
    return 0;
}

__global__ __launch_bounds__(256) void k_imm_blocks(const c64* W, long N, long m, long n, c64* Z)
{
    const long blk = blockIdx.z;
    const c64* src = W + (n + blk * m) * N + n + blk * m;
    c64* dst = Z + blk * (m * m + m);
    for (long i = blockIdx.y; i < m; i += gridDim.y)
        for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < m; k += (long)gridDim.x * 256)
            dst[i * m + k] = src[min(i, k) * N + max(i, k)];
}
int imm_blocks(const c64* W, long N, long m, long n, c64* Z, hipStream_t st)
{
    hipLaunchKernelGGL(k_imm_blocks, dim3((unsigned)std::min((m + 255) / 256, 16L),
                                          (unsigned)std::min(m, 16384L), 2),
                       dim3(256), 0, st, W, N, m, n, Z);
    TAGS_HIP(hipGetLastError());
    return 0;
}

}  // namespace tags
