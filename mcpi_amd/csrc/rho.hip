// One- and two-body density matrices and the Hellmann-Feynman adjoint.
//
// Reference: OBrho_XM, onebodyMatrix.h:190-251 (rho1), and TBrho_XX,
// twobodyMatrix.h:991-1487 (rho2, rules 1-8 plus symmetry copies).
//
// The reference walks the rows of the basis and adds, for every term its
// maps reach, conj(C_v') C_v times the bosonic factors into the matrix entry
// of the term: about M^4/4 gathered terms per row for rho2.  Here both
// densities are Gram matrices over the basis with fewer particles.  With the
// identity sum_u |u><u| over N-1 or N-2 particles inserted between the
// creators and the annihilators,
//
//   rho1[k + M l]                 = <a*_k a_l>         = sum_u conj(f_u(k)) f_u(l),
//       f_u(k)   = <u| a_k |C>     = sqrt(u_k + 1) C[rank(u + e_k)],          u in B(N-1, M)
//   rho2[a + bM + cM^2 + dM^3]    = <a*_a a*_b a_c a_d> = sum_u conj(g_u(ab)) g_u(cd),
//       g_u(ql)  = <u| a_q a_l |C> = sqrt((u_q + 1)(u_l + 1 + [q = l]))
//                                     C[rank(u + e_q + e_l)],                  u in B(N-2, M)
//
// (bosonic operators commute, so g_u depends on the unordered pair {q, l}).
// Every u + e_q + e_l is a state of the basis, so a row of the matrix
// Phi = [g_u(p)] needs M(M+1)/2 gathers of C and no occupation test, and
// rho2 is the Hermitian product Phi^H Phi: at N = M = 12, 27.5 M gathers and
// 2.1e9 complex multiply-adds (half of them computed, by Hermitian symmetry)
// in place of 2.2e9 gathered terms.  The result is the reference's sum
// regrouped, equal to it up to rounding.
//
// Targets: rank(v) = nc - 1 - sum_{j=1}^{M-1} B[j][P_j] with P_j the
// particles in orbitals below j (closed form of FockToIndex,
// configurationsMap.h:273-305).  Adding e_q + e_l (q <= l) to u raises P_j
// by 1 for q < j <= l and by 2 for j > l, so with the running sums
// S_d(x) = sum_{j=1}^{x} B[j][P_j(u) + d]:
//   rank(u + e_q + e_l) = nc - 1 - S_2(M-1) - (S_0(q) - S_1(q)) - (S_1(l) - S_2(l))
//   rank(u + e_k)       = nc - 1 - S_1(M-1) - (S_0(k) - S_1(k))
// Each row u of a tile has its two difference tables and the roots of its
// occupations made once, in LDS (pair_rows.h), so a gather costs four LDS reads,
// two subtractions and a product.
//
// Kernel k_gram: a block owns one tile pair (TI, TJ) of 80 x 80 entries of
// the Gram matrix and loops over tiles of U rows of Phi (32 for rho2, 128
// for rho1, whose Phi has at most 32 columns).  The row tables come from the
// basis's occupation table, two threads a row (without it, and for rho1, a
// thread unranks a row: greedy over B, the combinatorial number system), during
// the previous tile's products; the entries are gathered into LDS (lanes over
// consecutive rows of one column: neighbouring targets; all of a thread's loads
// in flight together), and the product runs on the FP64 matrix cores in 16 x 16
// sub-blocks: the sub-blocks i <= j of a diagonal tile pair, all of them off it,
// dealt out to the block's eight wavefronts (GramSplit).  Phi stays in LDS in one layout for both operands, because
// v_mfma_f64_16x16x4f64 takes A[i][k] and B[k][j] from the same lanes
// (i or j = lane % 16, k = lane / 16): lane (i, k) of step s reads column i of
// row 4 s + k.
// The bound is FP64: a complex product is three real ones here (Gauss), 6
// operations for each entry of the sub-blocks and row, against 8 on the vector
// units.  Eight wavefronts a block with at most two sub-blocks each leave room
// for two blocks a CU, so that one block's gathers and row tables run beside
// the other's products (four wavefronts with four sub-blocks each: 2.34 ms at
// N = 16, M = 12; three such blocks without gathers in flight over the
// products: 2.38 ms).  rho1 and rho2 together, kernels, sums and expansion, at
// M = 12: N = 12 (352,716 rows of 78 columns) 0.45 -> 0.20 ms, of which the
// product 0.32 -> 0.18; N = 16 (4,457,400 rows) 5.26 -> 2.12 ms, the product
// 4.2 -> 2.1 ms or 49 TFLOP/s issued (before: vector FMAs, unranked rows and a
// Gram product of its own for rho1).
// Rounding: the three products' errors are relative to |x| |y|, also in the part
// of a product that is small beside the other.  Over random complex vectors the
// result's relative error is 0.81 (rho2) and 0.62 (rho1) of that of the vector
// FMAs before (against 80-bit sums, 13 sizes from N = 2, M = 24 to N = 60, M = 3), a
// real vector has no imaginary part, but one whose imaginary parts are 1e-6 of
// the real ones keeps them to 1e-9 of themselves instead of 1e-15.  Four real
// products would keep them: 2.50 instead of 2.15 ms at N = 16, M = 12, 0.267
// instead of 0.237 at N = 12.
// Each block writes its sub-blocks once; two fixed-order stages sum the
// blocks (deterministic result), the second one inside the kernel that
// expands the Gram matrix into the full rho1 / rho2 arrays on the device.
// With rho2 at hand rho1 needs no Gram product of its own: on N >= 2
// particles sum_s a*_k a*_s a_s a_l = (N - 1) a*_k a_l.  No map is read, so
// the densities run on every storage mode, and the vectors are in the
// reference order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "mcpi_internal.h"
#include "pair_rows.h"

namespace mcpi {

namespace {

constexpr int GT = 80;            // Gram tile side (columns of Phi per tile)
constexpr int GG = GT / 16;       // 16 x 16 sub-blocks per tile side
constexpr int GU2 = 32;           // rows of Phi per LDS tile, rho2
constexpr int GU1 = 128;          // rows of Phi per LDS tile, rho1 (16 or 32 columns)
constexpr int GWAVES = 8;         // wavefronts of a block
constexpr int GTHREADS = 64 * GWAVES;
constexpr int GSEG = 8;           // segments of the first stage of the block sums

typedef double mcpi_v4d __attribute__((ext_vector_type(4)));

// sub-blocks of a tile pair with ng column groups a side
__host__ __device__ constexpr int gram_subblocks(int ng, bool diag) { return diag ? ng * (ng + 1) / 2 : ng * ng; }

// LDS row stride of a tile of Phi in complex entries: odd, so that the lanes
// of a gather write rows on distinct banks
__host__ __device__ constexpr int gram_stride(int ng) { return 16 * ng + 1; }

struct GramArgs {
    int N, M, ord;       // particles and orbitals of the basis; annihilators (1: rho1, 2: rho2)
    int np;              // columns of Phi: M (ord 1) or M(M+1)/2 (ord 2)
    int ntile;           // tiles of GT columns
    int ng;              // 16-column groups of a full tile (<= GG)
    int64_t nc;          // states of the basis
    int64_t nu;          // rows of Phi: states of B(N - ord, M)
    int64_t nut;         // tiles of U rows
    const int32_t *B;    // rank table B[j*(N+1) + p]
    const uint8_t *occ;  // occupations of the rows (null: unrank them)
    const cplx *C;       // vector, reference order
    cplx *partial;       // [block][entries]: the sub-blocks of the diagonal
                         // tile pairs, then of the others, 256 entries each
    int64_t entries;     // entries of one block's partial
};

__device__ inline cplx ldc(const cplx *p)
{
    double2 t = *reinterpret_cast<const double2 *>(p);
    return cmake(t.x, t.y);
}

// tile pair of an off-diagonal index: TI < TJ, lexicographic
__host__ __device__ inline void off_pair(int idx, int T, int &TI, int &TJ)
{
    TI = 0;
    while (idx >= T - 1 - TI) {
        idx -= T - 1 - TI;
        TI++;
    }
    TJ = TI + 1 + idx;
}

__host__ __device__ inline int off_index(int TI, int TJ, int T)
{
    return TI * (2 * T - TI - 1) / 2 + (TJ - TI - 1);
}

// LDS layout of a block (dynamic shared memory, in this order); red: the
// wavefronts' sums where they split the rows, over the tiles (which are
// done with by then)
struct GramLds {
    size_t phiA, phiB, g, sq, ql, tt, dd, bt, bytes;
};

__host__ __device__ inline GramLds gram_lds(int N, int M, int np, int ng, bool diag, int GU, int ord, size_t red)
{
    GramLds L;
    size_t o = 0;
    auto take = [&o](size_t n, size_t al) {
        o = (o + al - 1) / al * al;
        size_t r = o;
        o += n;
        return r;
    };
    L.phiA = take(sizeof(cplx) * GU * gram_stride(ng), 16);
    L.phiB = diag ? L.phiA : take(sizeof(cplx) * GU * gram_stride(ng), 16);
    if (o < red) o = red;
    L.g = take(sizeof(double) * GU * M * ord, 8);
    L.sq = take(sizeof(double) * (N + 3), 8);
    L.ql = take(sizeof(uint2) * np, 8);
    L.tt = take(sizeof(int32_t) * GU, 4);
    L.dd = take(sizeof(int32_t) * GU * M * ord, 4);
    L.bt = take(sizeof(int32_t) * M * (N + 1), 4);
    L.bytes = (o + 15) / 16 * 16;
    return L;
}

// How the wavefronts share the sub-blocks of a tile pair: WK of them split
// the rows (steps of four) and GWAVES / WK split the sub-blocks, at most NB
// each.  Few sub-blocks leave wavefronts without one, so they split the rows
// there and add their sums in LDS at the end.
template <bool DIAG, int NG>
struct GramSplit {
    static constexpr int SB = gram_subblocks(NG, DIAG);
    static constexpr int WK = SB <= 3 ? 8 : (SB <= 6 ? 4 : (SB <= 10 ? 2 : 1));
    static constexpr int WB = GWAVES / WK;
    static constexpr int NB = (SB + WB - 1) / WB;
    static constexpr size_t red = WK > 1 ? sizeof(cplx) * 256 * NB * WB * (WK - 1) : 0;
    // per SIMD: sub-blocks take 24 registers each, and 4 wavefronts (two
    // blocks of a CU in turn) leave 128
    static constexpr int WAVES = NB <= 2 ? 4 : 2;
};

// Block partials of one tile pair of Phi^H Phi.  DIAG: tile pair (TI, TI)
// from blockIdx.y, sub-blocks i <= j; else the off-diagonal pair
// off_pair(blockIdx.y), all sub-blocks.  OW > 0: the rows come
// from the occupation table, OW words each (rho2 only), else they are
// unranked.
template <bool DIAG, int GU, int NG, int OW>
__global__ __launch_bounds__(GTHREADS) __attribute__((amdgpu_waves_per_eu(GramSplit<DIAG, NG>::WAVES))) void
k_gram(GramArgs a)
{
    using S = GramSplit<DIAG, NG>;
    constexpr int NB = S::NB, RS = gram_stride(NG);
    extern __shared__ __align__(16) unsigned char lds[];
    const GramLds L = gram_lds(a.N, a.M, a.np, NG, DIAG, GU, a.ord, S::red);
    cplx *phiA = (cplx *)(lds + L.phiA);
    cplx *phiB = (cplx *)(lds + L.phiB);
    double *g = (double *)(lds + L.g);        // sqrt(u_o + 1), then sqrt(u_o + 2): [orbital][row]
    double *sq = (double *)(lds + L.sq);
    uint2 *ql = (uint2 *)(lds + L.ql);        // a column's places in dd and g (see below)
    int32_t *tt = (int32_t *)(lds + L.tt);    // rank(u + ord e_0), -1 past the last row
    int32_t *dd = (int32_t *)(lds + L.dd);    // S_0 - S_1, then S_1 - S_2: [orbital][row]
    int32_t *Bt = (int32_t *)(lds + L.bt);

    const int t = threadIdx.x;
    const int N = a.N, M = a.M, NB1 = N + 1, Np = N - a.ord;
    int TI, TJ;
    if (DIAG) TI = TJ = blockIdx.y;
    else off_pair(blockIdx.y, a.ntile, TI, TJ);

    for (int x = t; x < M * NB1; x += GTHREADS) Bt[x] = a.B[x];
    for (int x = t; x < N + 3; x += GTHREADS) sq[x] = sqrt((double)x);
    // column p = pair (q, l) or orbital q: its entries of dd at x (low half
    // q, high half l), the second root at y (sqrt(u_l + 1), or sqrt(u_l + 2)
    // for q = l; the first is at q)
    for (int x = t; x < a.np; x += GTHREADS) {
        int q = x, l = 0;
        if (a.ord == 2) {
            while ((l + 1) * (l + 2) / 2 <= x) l++;
            q = x - l * (l + 1) / 2;
        }
        ql[x] = make_uint2((unsigned)(q * GU) | (unsigned)((M + l) * GU) << 16,
                           (unsigned)((q == l ? M + l : l) * GU));
    }
    __syncthreads();
    // columns of the two sides (NG groups of 16, a.ng == NG; the columns of
    // a narrower last tile past wA / wB hold zeros, so every sub-block is
    // computed without a test)
    const int wA = min(GT, a.np - TI * GT), wB = min(GT, a.np - TJ * GT);

    // row r of a tile without an occupation table: unrank (greedy over B),
    // targets and roots
    auto unrank_row = [&](int64_t tile, int r) {
        const int64_t u = tile * GU + r;
        if (u >= a.nu) {
            tt[r] = -1;
            return;
        }
        // one step per iteration (lower p, or settle orbital j and move
        // down), so the lanes of a wavefront stay together: at most
        // Np + M - 1 iterations.  P_j falls with j: the occupation of
        // orbital j is known when P_j is.  dd holds P_j meanwhile.
        int32_t *dq = dd + r, *dl = dd + M * GU + r;
        double *gq = g + r, *gl = g + M * GU + r;
        int32_t R = (int32_t)(a.nu - 1 - u);
        int pj = Np, pa = Np, j = M - 1;
        while (j >= 1) {
            const int32_t bj = Bt[j * NB1 + pj];
            if (bj > R) {
                pj--;
            } else {
                dq[j * GU] = pj;
                gq[j * GU] = sq[pa - pj + 1];
                if (a.ord == 2) gl[j * GU] = sq[pa - pj + 2];
                pa = pj;
                R -= bj;
                j--;
            }
        }
        gq[0] = sq[pa + 1];
        if (a.ord == 2) gl[0] = sq[pa + 2];
        int32_t s0 = 0, s1 = 0, s2 = 0;
        dq[0] = 0;
        if (a.ord == 2) dl[0] = 0;
        for (int o = 1; o < M; o++) {
            const int b = o * NB1 + dq[o * GU];
            s0 += Bt[b];
            s1 += Bt[b + 1];
            dq[o * GU] = s0 - s1;
            if (a.ord == 2) {
                s2 += Bt[b + 2];
                dl[o * GU] = s1 - s2;
            }
        }
        tt[r] = (int32_t)(a.nc - 1) - (a.ord == 2 ? s2 : s1);
    };
    // rows of a tile from the occupation table (pair amplitudes only): two
    // threads a row, one for each table of differences; occ_row's load is
    // issued a tile earlier
    const bool duty = t < 2 * GU;
    const int dr = t % GU, dh = t / GU;
    constexpr int NW = OW ? OW : 1;
    uint32_t ow[NW];
    auto occ_row = [&](int64_t tile) {
        const int64_t u = min(tile * GU + dr, a.nu - 1);
        const uint4 *o = reinterpret_cast<const uint4 *>(a.occ + u * occ_stride(M));
#pragma unroll
        for (int k = 0; k < OW / 4; k++) {
            const uint4 w = o[k];
            ow[4 * k] = w.x;
            ow[4 * k + 1] = w.y;
            ow[4 * k + 2] = w.z;
            ow[4 * k + 3] = w.w;
        }
    };
    auto occ_tables = [&](int64_t tile) {
        const int32_t s = pair_row_tables<NW>(ow, M, NB1, Bt, sq, dh, dd + dh * M * GU + dr, GU,
                                              g + dh * M * GU + dr, GU);
        if (dh == 1) tt[dr] = tile * GU + dr < a.nu ? (int32_t)(a.nc - 1) - s : -1;
    };

    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int il = lane & 15, kl = lane >> 4;
    const int wk = wave / S::WB, wb = wave % S::WB;
    // this wavefront's sub-blocks: NB, or one fewer
    const int sb0 = wb * S::SB / S::WB;
    const bool last = (wb + 1) * S::SB / S::WB - sb0 == NB;
    int bi[NB], bj[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int b = min(sb0 + j, S::SB - 1);
        int I = 0, J = b;
        if (DIAG) {
            while (J >= NG - I) {
                J -= NG - I;
                I++;
            }
            J += I;
        } else {
            I = b / NG;
            J = b % NG;
        }
        bi[j] = 16 * I;
        bj[j] = 16 * J;
    }

    mcpi_v4d T1[NB], T2[NB], T3[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) T1[j] = T2[j] = T3[j] = mcpi_v4d{0, 0, 0, 0};

    constexpr int SIDES = DIAG ? 1 : 2;
    constexpr int CS = GTHREADS / GU, NK = 16 * NG / CS;   // columns side by side, and a thread's columns
    const int ul = t % GU, c0 = t / GU;
    // Gathers of a tile of Phi: a thread keeps to one row and takes every
    // CS-th column (lanes over consecutive rows of one column): targets and
    // loads, all in flight together, then (put) the LDS stores
    cplx v[SIDES][NK];
    double f[SIDES][NK];
    auto get = [&]() {
        const int32_t base = tt[ul];
#pragma unroll
        for (int h = 0; h < SIDES; h++) {
            const int p0 = (h ? TJ : TI) * GT + c0, pw = (h ? TJ : TI) * GT + (h ? wB : wA);
            int32_t tg[NK];
#pragma unroll
            for (int k = 0; k < NK; k++) {
                const int p = p0 + k * CS;
                const uint2 x = ql[p < pw ? p : 0];
                const int xq = x.x & 0xffff;
                tg[k] = base - dd[xq + ul];
                f[h][k] = g[xq + ul];
                if (a.ord == 2) {
                    tg[k] -= dd[(x.x >> 16) + ul];
                    f[h][k] *= g[x.y + ul];
                }
                // columns and rows past the last: the load goes to entry 0, put
                // stores zero (no branch: all loads are in flight together)
                if (base < 0 || p >= pw) {
                    tg[k] = 0;
                    f[h][k] = -1;
                }
            }
#pragma unroll
            for (int k = 0; k < NK; k++) v[h][k] = ldc(a.C + tg[k]);
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int h = 0; h < SIDES; h++) {
            cplx *row = (h ? phiB : phiA) + ul * RS + c0;
#pragma unroll
            for (int k = 0; k < NK; k++) row[k * CS] = f[h][k] < 0 ? cmake(0, 0) : cscale(v[h][k], f[h][k]);
        }
    };

    auto rows = [&](int64_t tile) {
        if (tile >= a.nut) return;
        if (OW == 0) {
            if (t < GU) unrank_row(tile, t);
        } else if (duty) {
            occ_tables(tile);
            occ_row(tile + gridDim.x);
        }
    };
    // The gathers of a tile are in flight during the previous tile's
    // products, and the row tables of the one after are made beside them (by
    // the wavefront with the fewest sub-blocks)
    if (OW > 0 && duty) occ_row(blockIdx.x);
    rows(blockIdx.x);
    if (blockIdx.x < a.nut) {
        __syncthreads();
        get();
        __syncthreads();
        rows(blockIdx.x + gridDim.x);
    }
    for (int64_t tile = blockIdx.x; tile < a.nut; tile += gridDim.x) {
        const int64_t next = tile + gridDim.x;
        put();
        __syncthreads();   // the tile and the next one's row tables are written
        // (the loaded occupations are taken first: waiting for them after the
        // gathers would wait for those too)
        if (OW > 0)
#pragma unroll
            for (int k = 0; k < NW; k++) asm volatile("" : "+v"(ow[k]));
        if (next < a.nut) get();
        __syncthreads();   // the next tile's row tables are read
        rows(next + gridDim.x);
        // conj(x + iy) (u + iv) = (k1 + k3) + i (k1 + k2) with k1 = u (x - y),
        // k2 = x (v - u), k3 = y (u + v)
#pragma unroll 2
        for (int s = 0; s < GU / 4 / S::WK; s++) {
            const cplx *ra = phiA + (4 * (s * S::WK + wk) + kl) * RS + il;
            const cplx *rb = phiB + (4 * (s * S::WK + wk) + kl) * RS + il;
#pragma unroll
            for (int j = 0; j < NB; j++) {
                if (j == NB - 1 && !last) continue;
                const cplx x = ra[bi[j]], y = rb[bj[j]];
                T1[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re - x.im, y.re, T1[j], 0, 0, 0);
                T2[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.im - y.re, T2[j], 0, 0, 0);
                T3[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.re + y.im, T3[j], 0, 0, 0);
            }
        }
        __syncthreads();   // the tile's products are done
    }
    // re = T1 + T3, im = T1 + T2; register r of lane j + 16 g holds entry
    // (g + 4 r, j) of the sub-block
    const int at = kl * 16 + il;
    cplx *out = a.partial + (int64_t)blockIdx.x * a.entries +
                256 * ((int64_t)(DIAG ? 0 : a.ntile * gram_subblocks(GG, true)) + (int64_t)blockIdx.y * S::SB);
    if (S::WK > 1) {
        cplx *red = (cplx *)lds;   // [row split - 1][sub-block][256]
        __syncthreads();
        if (wk > 0) {
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    red[(((wk - 1) * S::WB + wb) * NB + j) * 256 + at + 64 * r] =
                        cmake(T1[j][r] + T3[j][r], T1[j][r] + T2[j][r]);
        }
        __syncthreads();
        if (wk > 0) return;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
        if (j == NB - 1 && !last) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            cplx z = cmake(T1[j][r] + T3[j][r], T1[j][r] + T2[j][r]);
            if (S::WK > 1) {
                const cplx *red = (const cplx *)lds;
#pragma unroll
                for (int w = 0; w < S::WK - 1; w++)
                    z = cadd(z, red[((w * S::WB + wb) * NB + j) * 256 + at + 64 * r]);
            }
            out[(sb0 + j) * 256 + at + 64 * r] = z;
        }
    }
}

// Block sums in two fixed-order stages.  Stage 1 (this kernel): segment s of
// the blocks (blocks s*seg .. s*seg+seg-1), in four parts of consecutive
// blocks side by side, summed into the partial of its first block; stage 2:
// the segment sums, in order, where they are read (GramSums).
__global__ __launch_bounds__(256) void k_gram_sum1(int64_t entries, int nblocks, int seg, cplx *__restrict__ partial)
{
    __shared__ cplx part[4][64];
    const int64_t x = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
    const int w = threadIdx.x >> 6;
    const int s0 = blockIdx.y * seg, s1 = min(nblocks, s0 + seg), q = (seg + 3) / 4;
    const int b0 = s0 + w * q, b1 = min(s1, b0 + q);
    double re = 0, im = 0;
    for (int b = b0; b < b1; b++) {
        const cplx z = ldc(partial + b * entries + x);
        re += z.re;
        im += z.im;
    }
    part[w][threadIdx.x & 63] = cmake(re, im);
    __syncthreads();
    if (w || s0 >= s1) return;
    for (int k = 1; k < 4; k++) {
        re += part[k][threadIdx.x].re;
        im += part[k][threadIdx.x].im;
    }
    partial[s0 * entries + x] = cmake(re, im);
}

// the segment sums of a Gram matrix held as the sub-blocks of its upper triangle
struct GramSums {
    const cplx *p;      // null: the matrix is zero
    int64_t step;       // entries from one segment's sums to the next's
    int nseg;
    int T, ng;          // tiles a side, column groups of a tile
};

// entry (p1, p2) of the Hermitian Gram matrix; a diagonal entry is real
__device__ inline cplx gram_entry(const GramSums &G, int p1, int p2)
{
    const bool lower = p1 > p2;
    const int a = lower ? p2 : p1, b = lower ? p1 : p2;
    const int TI = a / GT, TJ = b / GT, I = a % GT / 16, J = b % GT / 16;
    const int sb = gram_subblocks(G.ng, true);
    const int at = TI == TJ ? TI * sb + I * G.ng - I * (I - 1) / 2 + (J - I)
                            : G.T * sb + off_index(TI, TJ, G.T) * gram_subblocks(G.ng, false) + I * G.ng + J;
    const cplx *p = G.p + (int64_t)at * 256 + (a % 16) * 16 + b % 16;
    cplx y[GSEG];
#pragma unroll
    for (int s = 0; s < GSEG; s++) y[s] = s < G.nseg ? ldc(p + s * G.step) : cmake(0, 0);
    cplx z = y[0];
#pragma unroll
    for (int s = 1; s < GSEG; s++) z = cadd(z, y[s]);
    if (a == b) return cmake(z.re, 0);
    return lower ? cmake(z.re, -z.im) : z;
}

__device__ inline int pair_of(int x, int y)
{
    const int lo = x < y ? x : y, hi = x < y ? y : x;
    return hi * (hi + 1) / 2 + lo;
}

// rho1[k + M l] = G1(k, l), or with G2 at hand sum_s G2({k,s}, {s,l}) / (N -
// 1) (the first blocks1 blocks, 32 lanes an entry, lane s the term of s); a
// null matrix gives zeros (fewer particles than annihilators)
// rho2[a + bM + cM^2 + dM^3] = s2 * G2({a,b}, {c,d}) (the other blocks)
__global__ __launch_bounds__(256) void k_gram_expand(int N, int M, int blocks1, GramSums G1, cplx *__restrict__ rho1,
                                                     GramSums G2, cplx *__restrict__ rho2, double s2)
{
    const int64_t M2 = (int64_t)M * M;
    if ((int)blockIdx.x < blocks1) {
        const int x = blockIdx.x * 8 + threadIdx.x / 32, s = threadIdx.x % 32;
        const int k = x % M, l = x / M;
        cplx z = cmake(0, 0);
        if (x < M2 && s < M) {
            if (G2.p) z = gram_entry(G2, pair_of(k, s), pair_of(s, l));
            else if (G1.p && s == 0) z = gram_entry(G1, k, l);
        }
        for (int o = 16; o > 0; o >>= 1) {
            z.re += __shfl_xor(z.re, o, 64);
            z.im += __shfl_xor(z.im, o, 64);
        }
        if (x < M2 && s == 0) rho1[x] = G2.p ? cmake(z.re / (N - 1), z.im / (N - 1)) : z;
        return;
    }
    const int64_t x = (int64_t)(blockIdx.x - blocks1) * 256 + threadIdx.x;
    if (x >= M2 * M2) return;
    const int a = (int)(x % M), b = (int)(x / M % M), c = (int)(x / M2 % M), d = (int)(x / (M2 * M));
    rho2[x] = G2.p ? cscale(gram_entry(G2, pair_of(a, b), pair_of(c, d)), s2) : cmake(0, 0);
}

}  // namespace

// launch geometry of one Gram product
struct GramPlan {
    GramArgs a;
    int U = GU2;         // rows of Phi per LDS tile
    int ntp = 0;         // tile pairs: ntile diagonal, then the off-diagonal ones
    int nblocks = 0;     // blocks per tile pair
    size_t partial_entries() const { return (size_t)nblocks * a.entries; }
};

// plan Phi^H Phi for ord annihilators on basis b; nblocks at most max_blocks
static mcpi_status plan_gram(const BasisDev &b, int ord, int max_blocks, GramPlan *pl)
{
    GramArgs &a = pl->a;
    a.N = b.N;
    a.M = b.M;
    a.ord = ord;
    a.np = ord == 2 ? b.M * (b.M + 1) / 2 : b.M;
    a.ntile = (a.np + GT - 1) / GT;
    a.ng = std::min(GG, (a.np + 15) / 16);
    a.nc = b.nc;
    a.nu = b.N >= ord ? nc_of(b.N - ord, b.M) : 0;
    pl->U = ord == 2 ? GU2 : GU1;
    a.nut = (a.nu + pl->U - 1) / pl->U;
    a.B = b.B;
    a.occ = ord == 2 ? b.occ2 : nullptr;
    a.C = nullptr;
    a.partial = nullptr;
    const int noff = a.ntile * (a.ntile - 1) / 2;
    pl->ntp = a.ntile + noff;
    a.entries = 256 * ((int64_t)a.ntile * gram_subblocks(a.ng, true) + (int64_t)noff * gram_subblocks(a.ng, false));
    int dev = 0, ncu = 0;
    MCPI_HIP(hipGetDevice(&dev));
    MCPI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    // two blocks per CU (their registers fill it) over all tile pairs, at most one per row tile
    const int64_t want = std::max<int64_t>(1, (int64_t)2 * ncu / pl->ntp);
    pl->nblocks = (int)std::max<int64_t>(1, std::min<int64_t>({want, a.nut, (int64_t)max_blocks}));
    return MCPI_OK;
}

template <bool DIAG, int U, int NG, int OW>
static mcpi_status launch_gram_k(const GramPlan &pl, int ny, hipStream_t s)
{
    const size_t sm =
        gram_lds(pl.a.N, pl.a.M, pl.a.np, NG, DIAG, U, pl.a.ord, GramSplit<DIAG, NG>::red).bytes;
    MCPI_ARG(sm <= 160 * 1024, "density-matrix tiles exceed LDS");
    (void)hipFuncSetAttribute((const void *)k_gram<DIAG, U, NG, OW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
    hipLaunchKernelGGL((k_gram<DIAG, U, NG, OW>), dim3(pl.nblocks, ny), dim3(GTHREADS), sm, s, pl.a);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

template <bool DIAG, int U, int NG>
static mcpi_status launch_gram(const GramPlan &pl, int ny, hipStream_t s)
{
    if (U == GU2 && pl.a.occ) {
        if (pl.a.M <= 16) return launch_gram_k<DIAG, U, NG, U == GU2 ? 4 : 0>(pl, ny, s);
        return launch_gram_k<DIAG, U, NG, U == GU2 && NG == GG ? 8 : 0>(pl, ny, s);
    }
    return launch_gram_k<DIAG, U, NG, 0>(pl, ny, s);
}

// the block-partial kernels of a plan: rho1 (U = GU1, one tile of at most
// 32 columns) or rho2 (U = GU2: the diagonal tile pairs, then the others)
static mcpi_status launch_gram_kernels(const GramPlan &pl, hipStream_t s)
{
    const int T = pl.a.ntile;
    if (pl.U == GU1) {
        MCPI_ARG(T == 1 && pl.a.ng <= 2, "one-body Gram matrix wider than two column groups");
        return pl.a.ng == 1 ? launch_gram<true, GU1, 1>(pl, 1, s) : launch_gram<true, GU1, 2>(pl, 1, s);
    }
    switch (pl.a.ng) {
    case 1: MCPI_CHECK((launch_gram<true, GU2, 1>(pl, T, s))); break;
    case 2: MCPI_CHECK((launch_gram<true, GU2, 2>(pl, T, s))); break;
    case 3: MCPI_CHECK((launch_gram<true, GU2, 3>(pl, T, s))); break;
    case 4: MCPI_CHECK((launch_gram<true, GU2, 4>(pl, T, s))); break;
    default: MCPI_CHECK((launch_gram<true, GU2, GG>(pl, T, s))); break;
    }
    // off-diagonal tile pairs exist only when the columns fill more than one tile
    if (T > 1) MCPI_CHECK((launch_gram<false, GU2, GG>(pl, T * (T - 1) / 2, s)));
    return MCPI_OK;
}

// segment sums of Phi^H Phi in partial, on stream s
static mcpi_status run_gram(GramPlan pl, const cplx *C, cplx *partial, GramSums *G, hipStream_t s)
{
    pl.a.C = C;
    pl.a.partial = partial;
    MCPI_CHECK(launch_gram_kernels(pl, s));
    const int seg = (pl.nblocks + GSEG - 1) / GSEG, nseg = (pl.nblocks + seg - 1) / seg;
    if (seg > 1) {
        hipLaunchKernelGGL(k_gram_sum1, dim3((unsigned)(pl.a.entries / 64), (unsigned)nseg), dim3(256), 0, s,
                           pl.a.entries, pl.nblocks, seg, partial);
        MCPI_HIP(hipGetLastError());
    }
    *G = GramSums{partial, (int64_t)seg * pl.a.entries, nseg, pl.a.ntile, pl.a.ng};
    return MCPI_OK;
}

// Densities of C on the device: rho1 (M*M, if want1) and / or rho2 (M^4,
// scaled by s2, if want2) into device memory, on stream s.  ws: device
// workspace of ws_entries complex entries (null: only report the need in
// *need); the number of blocks shrinks to fit a given workspace.
static mcpi_status densities_dev(const BasisDev &b, const cplx *C, bool want1, bool want2, cplx *rho1, cplx *rho2,
                                 double s2, cplx *ws, size_t ws_entries, size_t *need, hipStream_t s)
{
    const int M = b.M;
    // one product: rho2's where it exists (rho1 is its contraction), else rho1's
    const bool do2 = want2 && b.N >= 2, do1 = want1 && b.N >= 1 && !do2;
    GramPlan pl;
    MCPI_CHECK(plan_gram(b, do2 ? 2 : 1, 1 << 20, &pl));
    if (!ws) {
        *need = do1 || do2 ? pl.partial_entries() : 1;
        return MCPI_OK;
    }
    GramSums none{}, G{};
    if (do1 || do2) {
        if (pl.partial_entries() > ws_entries) {
            MCPI_ARG(ws_entries >= (size_t)pl.a.entries, "density workspace too small");
            MCPI_CHECK(plan_gram(b, do2 ? 2 : 1, (int)(ws_entries / pl.a.entries), &pl));
        }
        MCPI_CHECK(run_gram(pl, C, ws, &G, s));
    }
    const int64_t M2 = (int64_t)M * M;
    const int blocks1 = want1 ? (int)((M2 + 7) / 8) : 0, blocks2 = want2 ? (int)((M2 * M2 + 255) / 256) : 0;
    hipLaunchKernelGGL(k_gram_expand, dim3((unsigned)(blocks1 + blocks2)), dim3(256), 0, s, b.N, M, blocks1,
                       do1 ? G : none, rho1, do2 ? G : none, rho2, s2);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

// The tables the density kernels read: rank table and sizes only; vectors
// are in the reference order also for a sector-ordered basis.
static BasisDev density_view(mcpi_basis bs)
{
    BasisDev b = bs->d;
    b.perm = nullptr;
    return b;
}

// rho1 / rho2 (rho2 scaled by s2) into host arrays; either may be null
static mcpi_status densities(mcpi_basis bs, const cplx *C, cplx *rho1, cplx *rho2, double s2)
{
    std::lock_guard<std::mutex> lock(bs->rho_mu);
    const BasisDev b = density_view(bs);
    const int64_t M2 = (int64_t)b.M * b.M, M4 = M2 * M2;
    size_t need = 0;
    MCPI_CHECK(densities_dev(b, C, rho1, rho2, nullptr, nullptr, s2, nullptr, 0, &need, 0));
    const size_t total = need + (rho1 ? M2 : 0) + (rho2 ? M4 : 0);
    if (bs->rho_ws_bytes < total * sizeof(cplx)) {
        if (bs->rho_ws) MCPI_HIP(hipFree(bs->rho_ws));
        bs->rho_ws = nullptr;
        bs->rho_ws_bytes = 0;
        MCPI_HIP(hipMalloc(&bs->rho_ws, total * sizeof(cplx)));
        bs->rho_ws_bytes = total * sizeof(cplx);
    }
    cplx *ws = (cplx *)bs->rho_ws;
    cplx *d1 = rho1 ? ws + need : nullptr;
    cplx *d2 = rho2 ? ws + need + (rho1 ? M2 : 0) : nullptr;
    MCPI_CHECK(densities_dev(b, C, rho1, rho2, d1, d2, s2, ws, need, &need, 0));
    if (rho1) MCPI_HIP(hipMemcpy(rho1, d1, sizeof(cplx) * M2, hipMemcpyDeviceToHost));
    if (rho2) MCPI_HIP(hipMemcpy(rho2, d2, sizeof(cplx) * M4, hipMemcpyDeviceToHost));
    return MCPI_OK;
}

// ------------------------------------------------ allocation-free adjoint --
// For callers that cannot allocate device memory (code under stream capture,
// serving loops): the block partials and the Gram tiles live in a file-scope
// device array instead of the basis's workspace (fewer blocks when the
// partials would not fit), and the outputs are written on the device, so
// the call allocates nothing and copies nothing to the host.  Every call on
// a GPU shares that GPU's array: calls that overlap on one GPU race.
#define MCPI_NOALLOC_SCRATCH_BYTES (16u << 20)
static __device__ __align__(256) cplx scratch[MCPI_NOALLOC_SCRATCH_BYTES / sizeof(cplx)];

#define MCPI_NOALLOC_MAXDEV 64
static std::mutex g_scratch_mu;
static cplx *g_scratch_dev[MCPI_NOALLOC_MAXDEV];

// device address of this device's copy of `scratch` (looked up once per
// device, with that device current)
static mcpi_status noalloc_scratch(cplx **p)
{
    int dev = 0;
    MCPI_HIP(hipGetDevice(&dev));
    MCPI_ARG(dev >= 0 && dev < MCPI_NOALLOC_MAXDEV, "device ordinal beyond the supported range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *a = nullptr;
        MCPI_HIP(hipGetSymbolAddress(&a, HIP_SYMBOL(scratch)));
        g_scratch_dev[dev] = (cplx *)a;
    }
    *p = g_scratch_dev[dev];
    return MCPI_OK;
}

static mcpi_status vjp_noalloc(mcpi_basis bs, const cplx *C, cplx *g1, cplx *g2, hipStream_t s)
{
    cplx *scr = nullptr;
    MCPI_CHECK(noalloc_scratch(&scr));
    const size_t cap = MCPI_NOALLOC_SCRATCH_BYTES / sizeof(cplx);
    const mcpi_status st = densities_dev(density_view(bs), C, true, true, g1, g2, 0.5, scr, cap, nullptr, s);
    if (st == MCPI_ERR_ARG)
        set_error("basis has too many orbitals for the allocation-free adjoint (scratch holds 16 MiB)");
    return st;
}

}  // namespace mcpi

using namespace mcpi;

extern "C" {

mcpi_status mcpi_hip_rho1(mcpi_basis b, const mcpi_cplx *C_dev, mcpi_cplx *rho1)
{
    MCPI_ARG(b && C_dev && rho1, "null argument");
    return densities(b, (const cplx *)C_dev, (cplx *)rho1, nullptr, 1.0);
}

mcpi_status mcpi_hip_rho2(mcpi_basis b, const mcpi_cplx *C_dev, mcpi_cplx *rho2)
{
    MCPI_ARG(b && C_dev && rho2, "null argument");
    return densities(b, (const cplx *)C_dev, nullptr, (cplx *)rho2, 1.0);
}

mcpi_status mcpi_hip_vjp(mcpi_basis b, const mcpi_cplx *C_dev, mcpi_cplx *dE_dHo, mcpi_cplx *dE_dHint)
{
    MCPI_ARG(b && C_dev && dE_dHo && dE_dHint, "null argument");
    // Hellmann-Feynman: E = sum Ho . rho1 + 1/2 sum Hint . rho2
    return densities(b, (const cplx *)C_dev, (cplx *)dE_dHo, (cplx *)dE_dHint, 0.5);
}

mcpi_status mcpi_hip_vjp_noalloc(mcpi_basis b, const mcpi_cplx *C_dev, mcpi_cplx *dE_dHo_dev,
                                 mcpi_cplx *dE_dHint_dev, void *stream)
{
    MCPI_ARG(b && C_dev && dE_dHo_dev && dE_dHint_dev, "null argument");
    return vjp_noalloc(b, (const cplx *)C_dev, (cplx *)dE_dHo_dev, (cplx *)dE_dHint_dev, (hipStream_t)stream);
}

}  // extern "C"
