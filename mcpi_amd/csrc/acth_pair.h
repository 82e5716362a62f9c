// H.v through the pair space (schedules 6 and 7): every term of the
// reference's operator (hamiltonianMatrix.h:1431-1970, the folded rules of
// acth.hip), evaluated as two gathers around a pair-space step instead of
// one gather per term.
//
// In pair form (build_coefficients) the operator is
//   H = sum_{k,l} h1[k][l] a*_k a_l + sum_{P,Q} W[P][Q] a*_{P1} a*_{P2} a_{Q1} a_{Q2}
// over unordered orbital pairs.  On N >= 2 particles the one-body part is a
// pair term too (a*_k a_l = sum_s a*_k a*_s a_s a_l / (N - 1)).  Inserting
// the identity over the basis with N-2 particles after the creators,
//   (H C)(v) = sum_P <v|a*_{P1} a*_{P2}|u> Y2_u(P),  u = v - e_{P1} - e_{P2}
//   Y2_u(P)  = sum_Q W[P][Q] X[Q][u],  X[Q][u] = <u|a_{Q1} a_{Q2}|C>
// and <u|a_q a_l|C> = sqrt((u_q + 1)(u_l + 1 + [q = l])) C[rank(u + e_q + e_l)]
// is the pair amplitude of the densities' Gram matrix (rho.hip).  At N = M =
// 12 a row has up to 1,636 double-jump terms; here it costs 78 output
// gathers, and the 352,716 rows of 10 particles cost 78 gathers and a 78 x
// 78 complex matrix-vector product each, on the FP64 MFMA (schedule 6).
// When W is block diagonal with rank-one blocks, W = a b^T on each block r
// (a contact interaction that conserves a pair charge), and h1 is diagonal,
// Y2_u(P) = a[P] Z[r(P)][u] with Z[r][u] = sum_{Q in r} b[Q] X[Q][u]: one
// sum per block and no product (schedule 7).
//
// k_pair_mul<M>: Y2 = W X on the MFMA, X gathered.
// k_pairz_amp<>: Z, gathered and summed per block.
// k_pair_out<M, FAC>: one thread per row v of the basis ranks the v - e_P
// in the smaller basis from its prefix-count tables and sums the factors
// times Y2 (or a[P] Z).  k_pair_y1<M, U>: for N = 1 only, the one-body
// part over the empty basis of N - 1 particles.  Y2, Z and X are stored
// column-major (Y[col * ld + u]) so that every pass reads and writes them
// coalesced.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mcpi_internal.h"
#include "pair_rows.h"

namespace mcpi {

namespace {

constexpr int PT = 256;   // threads per block

struct PairArgs {
    int N;                // particles of the basis
    int64_t nc;           // its states
    int64_t nu;           // states of the basis with N - 2 (or N - 1) particles
    int64_t nut;          // tiles of U rows
    const int32_t *B;     // rank table B[j*(N+1) + p]
    const cplx *C;
    const cplx *W;        // pair matrix in fragment order (c.pwf), or h1 as ph1[l * 16 + k] (M <= 12)
    cplx *Y;              // Y[col * ld + u]
    int64_t ld;           // row stride of Y (and of the pair amplitudes X), >= nu
    const uint8_t *occ;   // occupations of the N - 2 particle states (BasisDev::occ2)
    const PairOff *ql;    // pairs: their places in the row tables
    const PairRec *rec;   // factorized form: pairs block by block
    const PairRun *run;   // 4 gridDim.y runs of blocks
    int zR;               // blocks
    unsigned G;           // tiles dealt to an XCD in one piece
    int64_t mC, mY;       // factorized form, several members: entries between
                          // the members' C vectors and between their Z tables
};

__device__ inline cplx ldcp(const cplx *p)
{
    double2 t = *reinterpret_cast<const double2 *>(p);
    return cmake(t.x, t.y);
}

// 16-byte load at byte offset off of the buffer [p, p + bytes) (bytes <
// 2^31); an offset at or past the end reads zero without a memory access
__device__ inline cplx ldbuf(const cplx *p, int bytes, uint32_t off)
{
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, bytes, 0x00020000);
    const v4u w = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return cmake(__builtin_bit_cast(double, (unsigned long long)w.x | ((unsigned long long)w.y << 32)),
                 __builtin_bit_cast(double, (unsigned long long)w.z | ((unsigned long long)w.w << 32)));
}

template <int M, int U>
struct PairLds {
    static constexpr int RS = M + 1;   // LDS row stride of the tile (odd)
    static size_t bytes(int N)
    {
        size_t o = sizeof(cplx) * ((size_t)M * 16 + (size_t)U * RS);
        o += sizeof(int64_t) * ((size_t)U + (size_t)U * M);
        o += sizeof(double) * (N + 3) + sizeof(int32_t) * M * (N + 1) + (size_t)U * (M + 1);
        return (o + 15) / 16 * 16;
    }
};

// Y1[k][u] = sum_l h1[k][l] <u|a_l|C> over the basis with N-1 particles
template <int M, int U>
__global__ __launch_bounds__(PT) void k_pair_y1(PairArgs a)
{
    using L = PairLds<M, U>;
    constexpr int RS = L::RS, UR = U / 16;
    extern __shared__ __align__(16) unsigned char lds[];
    cplx *Wl = (cplx *)lds;                                   // [M][16]: h1[k][l] at l * 16 + k
    cplx *phi = Wl + M * 16;                                   // [U][RS]
    int64_t *tt = (int64_t *)(phi + U * RS);                  // [U]
    int64_t *dq = tt + U;                                      // [U][M]
    double *sq = (double *)(dq + U * M);                       // [N + 3]
    int32_t *Bt = (int32_t *)(sq + a.N + 3);                   // [M][N + 1]
    uint8_t *pp = (uint8_t *)(Bt + M * (a.N + 1));            // [U][M + 1]

    const int t = threadIdx.x;
    const int N = a.N, NB = N + 1, Np = N - 1;
    for (int x = t; x < M * 16; x += PT) Wl[x] = ldcp(a.W + x);
    for (int x = t; x < M * NB; x += PT) Bt[x] = a.B[x];
    for (int x = t; x < N + 3; x += PT) sq[x] = sqrt((double)x);
    const int pg = t & 15, ug = t >> 4;

    for (int64_t tile = blockIdx.x; tile < a.nut; tile += gridDim.x) {
        __syncthreads();   // the previous tile's product has read phi and the row tables
        const int64_t u0 = tile * U;
        if (t < U) {
            const int64_t u = u0 + t;
            uint8_t *P = pp + t * (M + 1);
            if (u < a.nu) {
                // greedy unranking, one step per iteration (lanes stay together)
                int64_t R = a.nu - 1 - u;
                int pj = Np, j = M - 1;
                P[M] = (uint8_t)Np;
                while (j >= 1) {
                    const int64_t bj = Bt[j * NB + pj];
                    if (bj > R) {
                        pj--;
                    } else {
                        P[j] = (uint8_t)pj;
                        R -= bj;
                        j--;
                    }
                }
                P[0] = 0;
                int64_t s0 = 0, s1 = 0;
                int64_t *Dq = dq + t * M;
                Dq[0] = 0;
                for (int j2 = 1; j2 < M; j2++) {
                    const int b = j2 * NB + P[j2];
                    s0 += Bt[b];
                    s1 += Bt[b + 1];
                    Dq[j2] = s0 - s1;
                }
                tt[t] = a.nc - 1 - s1;
            } else {
                tt[t] = -1;
            }
        }
        __syncthreads();
        // amplitudes of the tile: lanes over consecutive rows of one column,
        // five loads in flight per thread
        constexpr int NE = U * M, GBP = 5;
        for (int e0 = t; e0 < NE; e0 += GBP * PT) {
            int64_t tg[GBP];
            double f[GBP];
#pragma unroll
            for (int k = 0; k < GBP; k++) {
                const int e = e0 + k * PT;
                const int col = e / U, ul = e % U;
                const int64_t base = e < NE ? tt[ul] : -1;
                tg[k] = -1;
                f[k] = 0;
                if (base >= 0) {
                    const uint8_t *P = pp + ul * (M + 1);
                    tg[k] = base - dq[ul * M + col];
                    f[k] = sq[P[col + 1] - P[col] + 1];
                }
            }
            cplx v[GBP];
#pragma unroll
            for (int k = 0; k < GBP; k++) v[k] = tg[k] >= 0 ? ldcp(a.C + tg[k]) : cmake(0, 0);
#pragma unroll
            for (int k = 0; k < GBP; k++) {
                const int e = e0 + k * PT;
                if (e < NE) phi[(e % U) * RS + e / U] = cscale(v[k], f[k]);
            }
        }
        __syncthreads();
        // thread (pg, ug) forms column pg (an orbital k < M) of the rows
        // ug + 16 j
        cplx acc[UR];
#pragma unroll
        for (int j = 0; j < UR; j++) acc[j] = cmake(0, 0);
#pragma unroll 2
        for (int l = 0; l < M; l++) {
            const cplx w = Wl[l * 16 + pg];
            cplx x[UR];
#pragma unroll
            for (int j = 0; j < UR; j++) x[j] = phi[(ug + 16 * j) * RS + l];
#pragma unroll
            for (int j = 0; j < UR; j++) acc[j] = cfma(w, x[j], acc[j]);
        }
        if (pg < M) {
#pragma unroll
            for (int j = 0; j < UR; j++) {
                const int64_t u = u0 + ug + 16 * j;
                if (u < a.nu) {
                    double2 o;
                    o.x = acc[j].re;
                    o.y = acc[j].im;
                    *reinterpret_cast<double2 *>(a.Y + (int64_t)pg * a.ld + u) = o;
                }
            }
        }
    }
}

// Row tables of a tile of PAIR_U states u of N - 2 particles in LDS, PAIR_ORB
// bytes per orbital o: the differences of the rank sums for o the lower (dq)
// and the higher (dl) orbital of a pair, sqrt(u_o + 1), and sqrt(u_o + 2) for
// the pairs q = l.  A pair and row take two differences and two roots, at
// offsets that depend on the pair alone (PairOff): four LDS reads.
constexpr int PAIR_DL = 4, PAIR_G = PAIR_SLOT;   // of an orbital's entries: dl, the roots

static size_t pair_amp_lds(int N, int M)
{
    const size_t o = (size_t)PAIR_ORB * M + sizeof(double) * (N + 3) + sizeof(int32_t) * (PAIR_U + M * (N + 1));
    return (o + 15) / 16 * 16;
}

// tables the launches pass are read through constant pointers: uniform
// indices then give scalar loads although the kernels write memory
template <class T>
__device__ inline const __attribute__((address_space(4))) T *kptr(const T *p)
{
    return (const __attribute__((address_space(4))) T *)p;
}

// The tables of a row with occupations w (NW words of bytes, orbital 0 first)
// at tab; returns rank(u + 2 e_0).  Four orbitals' entries are in flight
// together.
template <int NW>
__device__ inline int32_t pair_rows(const uint32_t (&w)[NW], int M, int NB1, int32_t top, const int32_t *Bt,
                                    const double *sq, unsigned char *tab)
{
    int p = 0;
    int32_t s01 = 0, s12 = 0, s2 = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        if (4 * k >= M) continue;
        int32_t b0[4], b1[4], b2[4];
        double g[4], g2[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // (orbitals past M - 1 read its entry again and are not stored)
            const int o = 4 * k + j, b = (o < M ? o : M - 1) * NB1 + p;
            const int v = (int)((w[k] >> (8 * j)) & 255u);
            b0[j] = Bt[b];
            b1[j] = Bt[b + 1];
            b2[j] = Bt[b + 2];
            g[j] = sq[v + 1];
            g2[j] = sq[v + 2];
            p += v;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int o = 4 * k + j;
            if (o >= M) continue;
            if (o) {
                s01 += b0[j] - b1[j];
                s12 += b1[j] - b2[j];
                s2 += b2[j];
            }
            unsigned char *t = tab + o * PAIR_ORB;
            *(int2 *)t = make_int2(s01, s12);
            *(double *)(t + PAIR_G) = g[j];
            *(double *)(t + PAIR_G + PAIR_SLOT) = g2[j];
        }
    }
    return top - s2;
}

// target of a pair and row (tab: the row's entries) and its amplitude's factor
__device__ inline uint32_t pair_target(const unsigned char *tab, int oq, int ol, int e, int32_t base, double &f)
{
    f = *(const double *)(tab + oq + PAIR_G) * *(const double *)(tab + ol + e + PAIR_G);
    return (uint32_t)(base - *(const int32_t *)(tab + oq) - *(const int32_t *)(tab + ol + PAIR_DL));
}

// Z[r][u] = sum_{Q in block r} zb[Q] <u|a_{Q1} a_{Q2}|C> of the factorized pair
// form; Z has R rows of ld entries.  MV > 1: the same for MV members that share
// zb and the blocks, their C vectors mC and their Z tables mY entries apart
// (the row tables and the targets are shared); grid row z serves members z MV
// .. z MV + MV - 1.  RC: zb is real.
//
// A block tabulates 64 rows from the occupation table (one wavefront) and its
// four wavefronts share the list of pairs (a.rec, block by block), cut at block
// borders into 4 gridDim.y runs of about the same length (a.run): with few rows
// gridDim.y > 1 gives every CU something to do.  A wavefront walks its run in
// batches of BT pairs whose loads are in flight together, across the borders
// of the blocks r.  Per pair and row: four LDS reads, two differences, one
// gather.  What bounds it is the L2: neighbouring tiles gather from
// neighbouring parts of C, so chunks of them go to one XCD each.
// Measured (before: rows unranked in the kernel, two pairs in flight, tiles
// dealt out one by one; blocks of one pair included): N = 12, M = 12 88 -> 38
// us, 11 TB/s of gathered entries; N = 16, M = 12 1220 -> 630 us (chunks of 128
// tiles; single tiles 14 % more); 24 members of N = 10, M = 13, four at a time,
// 688 -> 530 us (chunks of 32 tiles, whose part of four C vectors an L2 holds;
// 128 tiles 36 % more); N = 5, M = 21 60 -> 6 us (eleven runs of 28 tiles).
template <int NW, int MV, bool RC>
__global__ __launch_bounds__(PT) void k_pairz_amp(PairArgs a, int M)
{
    constexpr int U = PAIR_U, BT = 8;

    extern __shared__ __align__(16) unsigned char lds[];
    double *sq = (double *)(lds + PAIR_ORB * M);               // [N + 3]
    int32_t *tt = (int32_t *)(sq + a.N + 3);                   // [U]
    int32_t *Bt = tt + U;                                      // [M][N + 1]
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int N = a.N, NB1 = N + 1;
    const int64_t m0 = MV > 1 ? (int64_t)blockIdx.z * MV : 0;   // first member of this grid row
    // one tile a block; its occupations' load goes first
    const int64_t u = (int64_t)chunk_xcd(blockIdx.x, gridDim.x, a.G) * U + lane;
    uint32_t w[NW];
    if (wave == 0) {
        const uint4 *o = reinterpret_cast<const uint4 *>(a.occ + (u < a.nu ? u : a.nu - 1) * (4 * NW));
#pragma unroll
        for (int k = 0; k < NW / 4; k++) {
            const uint4 x = o[k];
            w[4 * k] = x.x;
            w[4 * k + 1] = x.y;
            w[4 * k + 2] = x.z;
            w[4 * k + 3] = x.w;
        }
    }
    // this wavefront's run of blocks
    const auto rec = kptr(a.rec);
    const auto run = kptr(a.run) + 4 * blockIdx.y + wave;
    const int r0 = run[0].r, j0 = run[0].j, j1 = run[1].j;
    for (int x = t; x < M * NB1; x += PT) Bt[x] = a.B[x];
    for (int x = t; x < N + 3; x += PT) sq[x] = sqrt((double)x);
    unsigned char *tab = lds + 8 * lane;
    __syncthreads();
    if (wave == 0) tt[lane] = pair_rows<NW>(w, M, NB1, (int32_t)(a.nc - 1), Bt, sq, tab);
    __syncthreads();
    {
        const int32_t base = tt[lane];
        cplx acc[MV];
#pragma unroll
        for (int m = 0; m < MV; m++) acc[m] = cmake(0, 0);
        int r = r0;
        // B pairs from j on (past the run's end its last pair again, unused)
        auto batch = [&](auto size, int j) {
            constexpr int B = decltype(size)::value;
            double f[B];
            cplx v[MV][B];
#pragma unroll
            for (int k = 0; k < B; k++) {
                const auto &x = rec[j + k < j1 ? j + k : j1 - 1];
                const uint32_t tg = pair_target(tab, x.oq, x.ol, x.e, base, f[k]);
#pragma unroll
                for (int m = 0; m < MV; m++) v[m][k] = ldcp(a.C + (m0 + m) * a.mC + tg);
            }
#pragma unroll
            for (int k = 0; k < B; k++) {
                if (j + k >= j1) continue;
                const auto &x = rec[j + k];
#pragma unroll
                for (int m = 0; m < MV; m++) {
                    if (RC) {
                        acc[m].re = fma(x.br * f[k], v[m][k].re, acc[m].re);
                        acc[m].im = fma(x.br * f[k], v[m][k].im, acc[m].im);
                    } else {
                        acc[m] = cfma(cscale(cmake(x.br, x.bi), f[k]), v[m][k], acc[m]);
                    }
                }
                if (x.last) {
                    if (u < a.nu) {
#pragma unroll
                        for (int m = 0; m < MV; m++) {
                            double2 o;
                            o.x = acc[m].re;
                            o.y = acc[m].im;
                            *reinterpret_cast<double2 *>(a.Y + (m0 + m) * a.mY + (int64_t)r * a.ld + u) = o;
                        }
                    }
#pragma unroll
                    for (int m = 0; m < MV; m++) acc[m] = cmake(0, 0);
                    r++;
                }
            }
        };
        int j = j0;
        for (; j + BT <= j1; j += BT) batch(std::integral_constant<int, BT>(), j);
#pragma clang loop unroll(disable)
        for (; j < j1; j += 2) batch(std::integral_constant<int, 2>(), j);
    }
}

// Y2 = W X, X[Q][u] = <u|a_{Q1} a_{Q2}|C> gathered on the fly, through FP64 MFMA
// (v_mfma_f64_16x16x4f64: lane i + 16k holds A[i][k] and B[k][i]; the result
// D[g + 4r][j] sits in register r of lane j + 16g), three real products per
// complex one (Gauss): T1 = (Xr + Xi) Wr, T2 = Xr (Wi - Wr), T3 = Xi (Wr + Wi),
// then Re = T1 - T3 and Im = T1 + T2.  A = W: the block keeps it in LDS as
// fragments in the order the lanes read them, [s][g][lane] = W[16g + i][4s +
// k], KS = ceil(NP/4) steps of four Q times NG groups of 16 pair rows P, zero
// past NP (c.pwf, laid out with the Hamiltonian, its one-body part folded in:
// folding it in every block took 25 us of the kernel's 82 at N = 10, M = 12).
// B = X: each wavefront takes 16 rows u on its own, tabulates them (the tables
// of pair_rows, 16 rows wide) and keeps the NP x 16 result in accumulators;
// lane (j, k) of step s gathers X[4s + k][u_j], four steps ahead of its use, so
// X is never written.  Wavefronts share nothing but W: while one starts a row
// block, the other one of its SIMD has the matrix core.
// Each XCD takes a contiguous eighth of the row blocks (neighbouring rows
// gather from neighbouring parts of C).
// Measured (before: X written by a kernel of its own, W folded and staged by
// every block): N = 10, M = 12 amplitudes and product 30 + 82 -> 66 us; N = 12,
// M = 12 0.13 + 0.28 -> 0.27 ms; 51 TFLOP/s issued of the 64 that this loop
// reaches without memory; the workspace halves.
typedef double mcpi_v4d __attribute__((ext_vector_type(4)));

constexpr int PAIR_MUL_WAVES = 8;

template <int M>
struct PairMulLds {
    static constexpr int NP = pair_count(M), KS = pair_x_rows(M) / 4, NG = pair_stride(M) / 16;
    static constexpr int ORB = PAIR_ORB / 4, SLOT = PAIR_SLOT / 4;   // tables of 16 rows
    static size_t bytes(int N)
    {
        const size_t o = sizeof(cplx) * NG * KS * 64 + (size_t)PAIR_MUL_WAVES * ORB * M + sizeof(double) * (N + 3) +
                         sizeof(int4) * 4 * KS + sizeof(int32_t) * M * (N + 1);
        return (o + 31) / 16 * 16;
    }
};

template <int M>
__global__ __launch_bounds__(64 * PAIR_MUL_WAVES) void k_pair_mul(PairArgs a)
{
    using L = PairMulLds<M>;
    constexpr int NP = L::NP, KS = L::KS, NG = L::NG, ORB = L::ORB, SLOT = L::SLOT;
    static_assert(M <= 16, "16-byte occupation rows");
    extern __shared__ __align__(16) unsigned char lds[];
    cplx *wl = (cplx *)lds;                                            // [KS][NG][64]
    int4 *off = (int4 *)(wl + NG * KS * 64);                           // [4 KS]
    unsigned char *tabs = (unsigned char *)(off + 4 * KS);             // [wave][M][3][16] of 8 bytes
    double *sq = (double *)(tabs + PAIR_MUL_WAVES * ORB * M);          // [N + 3]
    int32_t *Bt = (int32_t *)(sq + a.N + 3);                           // [M][N + 1]
    const int N = a.N, NB1 = N + 1, nt = 64 * PAIR_MUL_WAVES, t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int jl = lane & 15, kl = lane >> 4;

    // this wavefront's row blocks: the XCD's eighth, dealt to its blocks, then
    // to their wavefronts
    const int64_t nrb = (a.nu + 15) / 16;
    const int nx = gridDim.x >= 8 ? 8 : 1, x = blockIdx.x % nx, bx = blockIdx.x / nx;
    const int nbx = ((int)gridDim.x - x + nx - 1) / nx;   // blocks of this XCD
    const int64_t end = nrb * (x + 1) / nx, step = (int64_t)nbx * PAIR_MUL_WAVES;
    int64_t rb = nrb * x / nx + bx + (int64_t)nbx * wave;

    // occupations of a row block: lanes 0..15 and 16..31 hold the same rows
    // (one half of the tables each)
    uint32_t ow[4] = {0, 0, 0, 0};
    auto occ_row = [&](int64_t r) {
        if (lane >= 32) return;
        int64_t u = r * 16 + jl;
        u = u < a.nu ? u : a.nu - 1;
        const uint4 w = *reinterpret_cast<const uint4 *>(a.occ + u * 16);
        ow[0] = w.x;
        ow[1] = w.y;
        ow[2] = w.z;
        ow[3] = w.w;
    };
    if (rb < end) occ_row(rb);
    for (int k = t; k < NG * KS * 64; k += nt) wl[k] = ldcp(a.W + k);
    for (int k = t; k < 4 * KS; k += nt) {
        const PairOff o = a.ql[k < NP ? k : NP - 1];
        off[k] = make_int4(o.oq / 4, o.ol / 4, o.e / 4, 0);
    }
    for (int k = t; k < M * NB1; k += nt) Bt[k] = a.B[k];
    for (int k = t; k < N + 3; k += nt) sq[k] = sqrt((double)k);
    __syncthreads();
    unsigned char *tab = tabs + wave * (ORB * M);
    int32_t base = 0;
    // targets and factors of step s, and the gather
    auto get = [&](int s, cplx &v, double &f) {
        const int4 o = off[4 * (s < KS ? s : KS - 1) + kl];
        const unsigned char *p = tab + 8 * jl;
        f = *(const double *)(p + o.x + SLOT) * *(const double *)(p + o.y + o.z + SLOT);
        v = ldcp(a.C + (uint32_t)(base - *(const int32_t *)(p + o.x) - *(const int32_t *)(p + o.y + PAIR_DL)));
    };
    for (; rb < end; rb += step) {
        if (lane < 32) {
            const int d = lane >> 4;
            const int32_t s = pair_row_tables<4>(ow, M, NB1, Bt, sq, d, (int32_t *)(tab + 8 * jl + 4 * d), ORB / 4,
                                                 (double *)(tab + 8 * jl + SLOT * (1 + d)), ORB / 8);
            base = (int32_t)(a.nc - 1) - s;   // of lanes 16..31: rank(u + 2 e_0)
        }
        base = __shfl(base, 16 + jl, 64);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (rb + step < end) occ_row(rb + step);
        cplx x0, x1, x2, x3;
        double f0, f1, f2, f3;
        get(0, x0, f0);
        get(1, x1, f1);
        get(2, x2, f2);
        get(3, x3, f3);
        mcpi_v4d acc[3 * NG];
#pragma unroll
        for (int g = 0; g < 3 * NG; g++) acc[g] = mcpi_v4d{0, 0, 0, 0};
        auto mul = [&](int s, const cplx v, double f) {
            const double xr = v.re * f, xi = v.im * f, xs = xr + xi;
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const cplx w = wl[(s * NG + g) * 64 + lane];
                acc[3 * g] = __builtin_amdgcn_mfma_f64_16x16x4f64(w.re, xs, acc[3 * g], 0, 0, 0);
                acc[3 * g + 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(w.im - w.re, xr, acc[3 * g + 1], 0, 0, 0);
                acc[3 * g + 2] = __builtin_amdgcn_mfma_f64_16x16x4f64(w.re + w.im, xi, acc[3 * g + 2], 0, 0, 0);
            }
        };
#pragma unroll
        for (int s = 0; s < KS; s += 4) {
            mul(s, x0, f0);
            if (s + 4 < KS) get(s + 4, x0, f0);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < KS) mul(s + 1, x1, f1);
            if (s + 5 < KS) get(s + 5, x1, f1);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 2 < KS) mul(s + 2, x2, f2);
            if (s + 6 < KS) get(s + 6, x2, f2);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 3 < KS) mul(s + 3, x3, f3);
            if (s + 7 < KS) get(s + 7, x3, f3);
            __builtin_amdgcn_sched_barrier(0);
        }
        // (Y has 16 NG rows of ld >= 16 nrb entries: no bounds)
#pragma unroll
        for (int g = 0; g < NG; g++) {
            cplx *y = a.Y + (int64_t)(16 * g + kl) * a.ld + rb * 16 + jl;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                double2 o;
                o.x = acc[3 * g][r] - acc[3 * g + 2][r];
                o.y = acc[3 * g][r] + acc[3 * g + 1][r];
                *reinterpret_cast<double2 *>(y + 4 * r * a.ld) = o;
            }
        }
    }
}

// out[v] = sum_k sqrt(v_k) Y1[k][rank'(v - e_k)] + sum_P f_P(v) Y2[P][rank''(v - e_P)];
// FAC (factorized pair form, Y2 = Z with one row per block):
// out[v] = (sum_k h1[k][k] v_k + sum_diag w v_q (v_l - [q = l])) C[v]
//          + sum_P f_P(v) za[P] Z[zblk[P]][rank''(v - e_P)]
// RC (FAC only): za is real.  MV > 1 (FAC only): MV members that share the
// basis, zb and the blocks (a group of Lieb-Liniger couplings): the row's
// occupations, prefix sums, pair offsets and factors serve every member;
// member m reads its C, Z, za and h1 at C + m mC, Z + m mZ and (bytes) za + m
// mK, h1 + m mK, and writes out + m mC; grid row y serves members y MV .. y MV
// + MV - 1.
//
// One thread per row.  The lanes of a wavefront are consecutive rows, which
// share the occupations of all but the first few orbitals, so an orbital that
// is empty in one of them is mostly empty in all: the pairs of a higher orbital
// c2 are passed over by the wavefront as a whole where no row has c2 (a load
// takes the vector memory pipeline the same time whether one lane or 64 take
// part; at N = 16, M = 12 about 50 of 78 loads remain).  Testing c1 too (42
// loads) costs as much in branches as it saves.  Where an orbital is empty in
// some lanes only, their offset lies past the column, which the buffer's range
// check turns into a zero without a memory access: no branch between the
// loads of a batch.  Occupations stay packed, a byte each, and the roots in
// LDS: registers are wavefronts, which hide the gathers.  Measured (before: all
// pairs, in batches of 13): N = 12, M = 12 88 -> 68 us, N = 16, M = 12 970 -> 780
// us (then bound by the nearly 6 GB that the L2s miss: the rows that read one
// entry of Z lie far apart), 24 members of N = 10, M = 13, four at a time, 918 ->
// 675 us.  Slower: each lane walking the pairs its own row has, through tables
// in LDS (N = 12 110 us, N = 16 1310 us, N = 5, M = 21 18 us as here).
struct PairOutArgs {
    int N;
    int64_t nc;
    const int32_t *IF, *B;
    int64_t nu1, nu2, ld2;
    const cplx *Y1, *Y2, *za;
    const int32_t *zblk;
    const cplx *h1, *C;
    const PairDiag *diag;   // pairs that are a block by themselves
    int nd;
    cplx *out;
    int64_t mC, mZ, mK;
    int S;   // wavefronts that share a row's pairs: 1, 2 or 4
    PairEpi ep;   // (one member) a Lanczos step's next vector operation, if ep.partial
};

template <int M, bool FAC, bool RC, int MV>
__global__ __launch_bounds__(PT) __attribute__((amdgpu_waves_per_eu(MV == 1 && M <= 16 ? 4 : 3))) void
k_pair_out(PairOutArgs a)
{
    static_assert(FAC || (MV == 1 && !RC), "several members: factorized form only");
    extern __shared__ __align__(16) unsigned char lds[];
    const int N = a.N;
    double *sq = (double *)lds;                      // [N + 3]
    int32_t *Bt = (int32_t *)(sq + N + 3);          // [M][N + 1]
    const int NB = N + 1;
    for (int x = threadIdx.x; x < N + 3; x += PT) sq[x] = sqrt((double)x);
    for (int x = threadIdx.x; x < M * NB; x += PT) Bt[x] = a.B[x];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = wave % a.S;   // this wavefront's share of its rows
    const int64_t i0 = ((int64_t)blockIdx.x * (PT / 64 / a.S) + wave / a.S) * 64 + lane;
    const int64_t i = i0 < a.nc ? i0 : a.nc - 1;
    const int64_t m0 = MV > 1 ? (int64_t)blockIdx.y * MV : 0;   // this grid row's first member
    const cplx *C = a.C + m0 * a.mC, *Z = a.Y2 + m0 * a.mZ;
    // the coefficients' uniform indices give scalar loads
    typedef const __attribute__((address_space(4))) char *kchar;
    typedef const __attribute__((address_space(4))) cplx *kcplx;
    const kchar za = (kchar)((const char *)a.za + m0 * a.mK), h1 = (kchar)((const char *)a.h1 + m0 * a.mK);
    const auto zblk = kptr(a.zblk);
    typedef const __attribute__((address_space(4))) PairDiag *kdiag;
    const kchar dgp = (kchar)((const char *)a.diag + m0 * a.mK);
    // occupations, a byte each (v(k)): the registers go to the gathers
    uint64_t pk[(M + 7) / 8];
#pragma unroll
    for (int k = 0; k < (M + 7) / 8; k++) pk[k] = 0;
#pragma unroll
    for (int k = 0; k < M; k++) pk[k / 8] |= (uint64_t)a.IF[i * M + k] << (8 * (k % 8));
    auto v = [&](int k) { return (int)((uint32_t)(pk[k / 8] >> (8 * (k % 8))) & 255u); };
    // the same for a run-time (uniform) orbital
    auto vrt = [&](int k) {
        uint64_t w = pk[0];
#pragma unroll
        for (int x = 1; x < (M + 7) / 8; x++) w = k >= 8 * x ? pk[x] : w;
        return (int)((uint32_t)(w >> (8 * (k & 7))) & 255u);
    };
    // D1[o] = S_0(o) - S_1(o), D2[o] = S_1(o) - S_2(o) of S_d(x) = sum_{j=1..x}
    // B[j][P_j - d] (P_j: particles below orbital j), modulo 2^32 (every rank
    // is below 2^31)
    uint32_t D1[M], D2[M], s1 = 0, s2 = 0;
    {
        int pj = 0;
        uint32_t d1 = 0, d2 = 0;
        D1[0] = D2[0] = 0;
#pragma unroll
        for (int j = 1; j < M; j++) {
            pj += v(j - 1);
            const int b = j * NB + pj;
            const uint32_t b0 = (uint32_t)Bt[b], b1 = (uint32_t)Bt[pj >= 1 ? b - 1 : b];
            const uint32_t b2 = (uint32_t)Bt[pj >= 2 ? b - 2 : b];
            s1 += b1;
            s2 += b2;
            D1[j] = d1 += b0 - b1;
            D2[j] = d2 += b1 - b2;
        }
    }
    // orbitals occupied in any row of the wavefront
    uint32_t any = 0;
#pragma unroll
    for (int k = 0; k < M; k++) any |= __ballot(v(k) > 0) ? 1u << k : 0u;
    any = __builtin_amdgcn_readfirstlane(any);
    // with S wavefronts a row, the orbitals c2 this one takes: dealt from the
    // highest (most pairs) to and fro
    uint32_t mine = any;
    if (a.S > 1) {
        mine = 0;
#pragma unroll
        for (int k = 0; k < M; k++) {
            const int x = (M - 1 - k) & (2 * a.S - 1);
            if ((x < a.S ? x : 2 * a.S - 1 - x) == sub) mine |= any & 1u << k;
        }
    }
    constexpr uint32_t OUT = 0x80000000u;   // beyond every column (< 2 GiB)
    cplx acc[MV];
#pragma unroll
    for (int m = 0; m < MV; m++) {
        acc[m] = cmake(0, 0);
        if (FAC && sub == 0) {   // the diagonal one-body part
            const kcplx h = (kcplx)(h1 + m * a.mK);
            cplx d = cmake(0, 0);
#pragma unroll
            for (int k = 0; k < M; k++) {
                const int x = k * (pair_h1_stride(M) + 1);
                d.re = fma(h[x].re, (double)v(k), d.re);
                if (!RC) d.im = fma(h[x].im, (double)v(k), d.im);
            }
            const kdiag dg = (kdiag)(dgp + m * a.mK);
            for (int x = 0; x < a.nd; x++) {
                const int q = dg[x].q, l = dg[x].l;
                const double w = (double)(vrt(q) * (vrt(l) - (q == l)));
                d.re = fma(dg[x].wr, w, d.re);
                if (!RC) d.im = fma(dg[x].wi, w, d.im);
            }
            const cplx c = ldcp(C + m * a.mC + i);
            acc[m] = RC ? cscale(c, d.re) : cfma(d, c, acc[m]);
        }
    }
    if (!FAC && a.nu1 > 0 && sub == 0) {
        const uint32_t top1 = (uint32_t)(a.nu1 - 1) - s1;
        const int bytes1 = (int)(a.nu1 * (int64_t)sizeof(cplx));
        cplx y[M];
#pragma unroll
        for (int k = 0; k < M; k++) {
            const uint32_t off = v(k) >= 1 ? (top1 - D1[k]) * (uint32_t)sizeof(cplx) : OUT;
            y[k] = ldbuf(a.Y1 + (int64_t)k * a.nu1, bytes1, off);
        }
#pragma unroll
        for (int k = 0; k < M; k++) {
            const double f = sq[v(k)];
            acc[0].re = fma(f, y[k].re, acc[0].re);
            acc[0].im = fma(f, y[k].im, acc[0].im);
        }
    }
    if (a.nu2 > 0) {
        const uint32_t top2 = (uint32_t)(a.nu2 - 1) - s2;
        const int bytes2 = (int)(a.nu2 * (int64_t)sizeof(cplx));
        // pairs c1 <= c2, c2 by c2 in batches of BT: every index below is a
        // constant (full unroll), the loads of a batch are in flight together
        constexpr int BT = MV == 1 ? 12 : (MV == 2 ? 6 : 4);
#pragma clang loop unroll(full)
        for (int c2 = 0; c2 < M; c2++) {
            if (!(mine >> c2 & 1)) continue;
            const uint32_t t2 = v(c2) >= 1 ? (top2 - D2[c2]) * (uint32_t)sizeof(cplx) : OUT;
            cplx sum[MV];   // over c1, without the root of v_c2
#pragma unroll
            for (int m = 0; m < MV; m++) sum[m] = cmake(0, 0);
#pragma clang loop unroll(full)
            for (int b0 = 0; b0 <= c2; b0 += BT) {
                cplx y[MV][BT];
#pragma unroll
                for (int k = 0; k < BT; k++) {
                    const int c1 = b0 + k;
                    if (c1 > c2) break;
                    const int P = c2 * (c2 + 1) / 2 + c1, blk = FAC ? zblk[P] : P;
                    const bool occ = v(c1) >= (c1 < c2 ? 1 : 2) && v(c2) >= 1 && blk >= 0;
                    const uint32_t off = occ ? t2 - D1[c1] * (uint32_t)sizeof(cplx) : OUT;
#pragma unroll
                    for (int m = 0; m < MV; m++) y[m][k] = ldbuf(Z + m * a.mZ + (int64_t)(blk >= 0 ? blk : 0) * a.ld2, bytes2, off);
                }
#pragma unroll
                for (int k = 0; k < BT; k++) {
                    const int c1 = b0 + k;
                    if (c1 > c2) break;
                    const int P = c2 * (c2 + 1) / 2 + c1;
                    const double f = sq[c1 < c2 ? v(c1) : (v(c1) >= 1 ? v(c1) - 1 : 0)];
#pragma unroll
                    for (int m = 0; m < MV; m++) {
                        if (!FAC) {
                            sum[m].re = fma(f, y[m][k].re, sum[m].re);
                            sum[m].im = fma(f, y[m][k].im, sum[m].im);
                            continue;
                        }
                        const kcplx zp = (kcplx)(za + m * a.mK) + P;
                        const cplx z = cmake(zp->re, RC ? 0.0 : zp->im);
                        if (RC) {
                            sum[m].re = fma(z.re * f, y[m][k].re, sum[m].re);
                            sum[m].im = fma(z.re * f, y[m][k].im, sum[m].im);
                        } else {
                            sum[m] = cfma(cscale(z, f), y[m][k], sum[m]);
                        }
                    }
                }
            }
            const double g2 = sq[v(c2)];
#pragma unroll
            for (int m = 0; m < MV; m++) {
                acc[m].re = fma(g2, sum[m].re, acc[m].re);
                acc[m].im = fma(g2, sum[m].im, acc[m].im);
            }
        }
    }
    if (a.S > 1) {   // the shares' sums, in order (over the tables, which are done with)
        cplx *red = (cplx *)lds;   // [member][wave][64]
        __syncthreads();
        if (sub > 0) {
#pragma unroll
            for (int m = 0; m < MV; m++) red[(m * (PT / 64) + wave) * 64 + lane] = acc[m];
        }
        __syncthreads();
        for (int w = 1; w < a.S && sub == 0; w++)
#pragma unroll
            for (int m = 0; m < MV; m++) acc[m] = cadd(acc[m], red[(m * (PT / 64) + wave + w) * 64 + lane]);
    }
    const bool own = sub == 0 && i0 < a.nc;
    if (MV == 1 && a.ep.partial) {
        double re = 0, im = 0;
        if (own) {
            const cplx x = ldcp(a.ep.lvec + (int64_t)*a.ep.it * a.nc + i), y = ldcp(C + i);
            const double beta = *a.ep.beta;
            acc[0].re -= beta * x.re;
            acc[0].im -= beta * x.im;
            re = y.re * acc[0].re + y.im * acc[0].im;
            im = y.re * acc[0].im - y.im * acc[0].re;
        }
#pragma unroll
        for (int k = 32; k > 0; k >>= 1) {
            re += __shfl_xor(re, k, 64);
            im += __shfl_xor(im, k, 64);
        }
        double *red = (double *)lds;   // [wave][2]
        __syncthreads();
        if (lane == 0) {
            red[2 * wave] = re;
            red[2 * wave + 1] = im;
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            double s = 0;
            for (int w = 0; w < PT / 64; w++) s += red[2 * w + threadIdx.x];
            a.ep.partial[2 * blockIdx.x + threadIdx.x] = s;
        }
    }
    if (!own) return;
#pragma unroll
    for (int m = 0; m < MV; m++) {
        double2 o;
        o.x = acc[m].re;
        o.y = acc[m].im;
        *reinterpret_cast<double2 *>(a.out + (m0 + m) * a.mC + i) = o;
    }
}

// launch of the output pass for `chunks` grid rows.  A row's pairs are a serial
// chain of batches, which few rows leave exposed: up to four wavefronts share
// a row's pairs until there are two blocks a CU, two where four would be more
// wavefronts than the registers of all CUs hold (three a SIMD beyond M = 16:
// N = 5, M = 21 H.v 20.9 us with two, 22.1 with four; N = 5, M = 20, whose four
// fit, 19.2 and 17.3).  Lanczos steps, us, without
// and with: N = 5, M = 21 (208 blocks of whole rows) 118, 110; N = 6, M = 9 (12)
// 43.0, 40.5; N = 7, M = 13 (197) 66.3, 63.2; with eight blocks a CU N = 10, M =
// 11 (722) slows from 125 to 129.
template <int M, bool FAC, bool RC, int MV>
mcpi_status launch_pair_out(PairOutArgs o, int chunks, int ncu, hipStream_t st, PairEpi *e)
{
    const int64_t rows = (o.nc + 63) / 64;   // wavefronts of whole rows
    o.S = 1;
    const int64_t resident = (int64_t)(M > 16 ? 3 : 4) * 4 * ncu;
    if (rows * chunks < (int64_t)2 * 4 * ncu) o.S = rows * chunks * 4 <= resident ? 4 : 2;
    const int64_t nb = (rows * o.S + PT / 64 - 1) / (PT / 64);
    size_t sm = sizeof(double) * (o.N + 3) + sizeof(int32_t) * M * (o.N + 1);
    sm = std::max(sm, o.S > 1 ? sizeof(cplx) * PT * MV : 2 * sizeof(double) * (PT / 64));
    if (MV == 1 && e && nb <= e->cap) {
        e->blocks = (int)nb;
        o.ep = *e;
    }
    hipLaunchKernelGGL((k_pair_out<M, FAC, RC, MV>), dim3((unsigned)nb, (unsigned)chunks), dim3(PT), sm, st, o);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

template <int M, int U>
mcpi_status launch_y1(const PairArgs &a, int ncu, hipStream_t st)
{
    const size_t sm = PairLds<M, U>::bytes(a.N);
    MCPI_ARG(sm <= 160 * 1024, "pair-space tile exceeds LDS");
    const int per_cu = std::max(1, (int)(160 * 1024 / sm));
    const int64_t nb = std::max<int64_t>(1, std::min<int64_t>(a.nut, (int64_t)ncu * per_cu));
    (void)hipFuncSetAttribute((const void *)k_pair_y1<M, U>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
    hipLaunchKernelGGL((k_pair_y1<M, U>), dim3((unsigned)nb), dim3(PT), sm, st, a);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

template <int M>
mcpi_status launch_pair_m(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                          hipStream_t st, PairEpi *e)
{
    int dev = 0, ncu = 0;
    MCPI_HIP(hipGetDevice(&dev));
    MCPI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const int N = b.N;
    const int64_t nu1 = N >= 1 ? nc_of(N - 1, M) : 0, nu2 = N >= 2 ? nc_of(N - 2, M) : 0;
    const int64_t ld2 = pair_ld(nu2);
    static_assert(pair_h1_stride(M) == 16, "the pair product reads h1 with row stride 16");
    // with N >= 2 the one-body part rides in the pair product (h1 folded
    // into W); the pass over N - 1 particles runs only for N = 1
    const int64_t nu1p = N == 1 ? nu1 : 0;
    cplx *Y1 = ws, *Y2 = ws + (size_t)M * nu1p;
    if (nu1p > 0) {
        PairArgs a{};
        a.N = N;
        a.nc = b.nc;
        a.nu = a.ld = nu1;
        a.nut = (nu1 + 127) / 128;
        a.B = b.B;
        a.C = C;
        a.W = c.ph1;
        a.Y = Y1;
        MCPI_CHECK((launch_y1<M, 128>(a, ncu, st)));
    }
    if (nu2 > 0) {
        PairArgs a{};
        a.N = N;
        a.nc = b.nc;
        a.nu = nu2;
        a.B = b.B;
        a.C = C;
        a.W = c.pwf;
        a.Y = Y2;
        a.ld = ld2;
        a.occ = b.occ2;
        a.ql = c.pql;
        const size_t smw = PairMulLds<M>::bytes(N);
        MCPI_ARG(smw <= 160 * 1024, "pair matrix exceeds LDS");
        (void)hipFuncSetAttribute((const void *)k_pair_mul<M>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)smw);
        const int nt = 64 * PAIR_MUL_WAVES;
        int per_cu = 0;
        MCPI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_pair_mul<M>, nt, smw));
        const int64_t nrb = (nu2 + 15) / 16;
        const int64_t nb = std::max<int64_t>(1, std::min<int64_t>(nrb, (int64_t)ncu * std::max(per_cu, 1)));
        hipLaunchKernelGGL(k_pair_mul<M>, dim3((unsigned)nb), dim3(nt), smw, st, a);
        MCPI_HIP(hipGetLastError());
    }
    PairOutArgs o{};
    o.N = N;
    o.nc = b.nc;
    o.IF = b.IF;
    o.B = b.B;
    o.nu1 = nu1p;
    o.nu2 = nu2;
    o.ld2 = ld2;
    o.Y1 = Y1;
    o.Y2 = Y2;
    o.C = C;
    o.out = out;
    return launch_pair_out<M, false, false, 1>(o, 1, ncu, st, e);
}

// Z of the factorized form for chunks x MV members: the rows' tiles, the runs
// of pairs (as many as give about eight blocks a CU where there are few tiles)
// and the chunks; tiles dealt to the XCDs in equal chunks of at most G
template <int NW, int MV, bool RC>
mcpi_status launch_pairz_amp(PairArgs a, int M, int chunks, int ncu, hipStream_t st)
{
    const size_t sm = pair_amp_lds(a.N, M);
    MCPI_ARG(sm <= 160 * 1024, "pair-space tile exceeds LDS");
    (void)hipFuncSetAttribute((const void *)k_pairz_amp<NW, MV, RC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)sm);
    const int64_t want = (8 * ncu + a.nut * chunks - 1) / (a.nut * chunks);
    const int runs = (int)std::max<int64_t>(1, std::min<int64_t>({want, (a.zR + 3) / 4, PAIR_RUNS}));
    a.run += pair_run(runs);
    const int64_t G = MV == 1 ? 128 : 32, rounds = (a.nut + 8 * G - 1) / (8 * G);
    a.G = (unsigned)std::max<int64_t>(1, a.nut / (8 * rounds));
    hipLaunchKernelGGL((k_pairz_amp<NW, MV, RC>), dim3((unsigned)a.nut, (unsigned)runs, (unsigned)chunks), dim3(PT), sm,
                       st, a, M);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

// the factorized pair form (schedule 7) for chunks x MV members: Z (pzR rows
// of ld2 a member) at the start of the workspace, then the output pass.
// Vectors mC entries and coefficient blocks mK bytes apart, member 0's tables
// in c
template <int M, int MV, bool RC>
mcpi_status launch_pairz_m(const BasisDev &b, const HamCoefDev &c, int chunks, const cplx *C, cplx *out, int64_t mC,
                           int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    int dev = 0, ncu = 0;
    MCPI_HIP(hipGetDevice(&dev));
    MCPI_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    const int N = b.N;
    const int64_t nu2 = nc_of(N - 2, M), ld2 = pair_ld(nu2), mZ = (int64_t)c.pzR * ld2;
    constexpr int U = PAIR_U;
    PairArgs a{};
    a.N = N;
    a.nc = b.nc;
    a.nu = nu2;
    a.nut = (nu2 + U - 1) / U;
    a.B = b.B;
    a.C = C;
    a.Y = ws;
    a.ld = ld2;
    a.occ = b.occ2;
    a.rec = c.pzrec;
    a.run = c.pzrun;
    a.zR = c.pzR;
    a.mC = mC;
    a.mY = mZ;
    MCPI_CHECK((launch_pairz_amp<M <= 16 ? 4 : 8, MV, RC>(a, M, chunks, ncu, st)));
    PairOutArgs o{};
    o.N = N;
    o.nc = b.nc;
    o.IF = b.IF;
    o.B = b.B;
    o.nu2 = nu2;
    o.ld2 = ld2;
    o.Y2 = ws;
    o.za = c.pza;
    o.zblk = c.pzblk;
    o.h1 = c.ph1;
    o.diag = c.pzdiag;
    o.nd = c.pznd;
    o.C = C;
    o.out = out;
    o.mC = mC;
    o.mZ = mZ;
    o.mK = mK;
    return launch_pair_out<M, true, RC, MV>(o, chunks, ncu, st, e);
}

template <int M, int MV>
mcpi_status launch_pairz_r(const BasisDev &b, const HamCoefDev &c, int chunks, const cplx *C, cplx *out, int64_t mC,
                           int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    return c.real ? launch_pairz_m<M, MV, true>(b, c, chunks, C, out, mC, mK, ws, st, e)
                  : launch_pairz_m<M, MV, false>(b, c, chunks, C, out, mC, mK, ws, st, e);
}

}  // namespace

#define MCPI_PAIR_CASE(MM) case MM: return launch_pair_m<MM>(b, c, C, out, ws, st, e);
// members: one, or chunks of mv
#define MCPI_PAIRZ_CASE(MM) case MM: return launch_pairz_r<MM, 1>(b, c, 1, C, out, 0, 0, ws, st, e);
#define MCPI_PAIRZ_MV_CASE(MM) \
    case MM: \
        if (mv == 1) return launch_pairz_r<MM, 1>(b, c, 1, C, out, 0, 0, ws, st, e); \
        return mv == 4 ? launch_pairz_r<MM, 4>(b, c, chunks, C, out, mC, mK, ws, st, nullptr) \
                       : launch_pairz_r<MM, 2>(b, c, chunks, C, out, mC, mK, ws, st, nullptr);

}  // namespace mcpi
