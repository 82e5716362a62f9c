// Pair-space H.v (schedules 6 and 7): where it applies, and the launch for a
// number of orbitals.  The kernels are in acth_pair.h, compiled for their M in
// acth_pair_a.hip (3..9) to acth_pair_d.hip (20..24); the one for bases of few
// rows is here.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mcpi_internal.h"

namespace mcpi {

#define MCPI_PAIR_ARGS const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws, hipStream_t st, PairEpi *e
#define MCPI_PAIRZ_ARGS const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out, \
                        int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e
mcpi_status launch_pair_a(MCPI_PAIR_ARGS);
mcpi_status launch_pair_b(MCPI_PAIR_ARGS);
mcpi_status launch_pairz_a(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_b(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_c(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_d(MCPI_PAIRZ_ARGS);

namespace {

constexpr int DW = 4;   // rows (wavefronts) a block

// H.v in the factorized form on a basis of few rows, without the pair space:
// out[v] = sum_k h1[k][k] v_k C[v] + sum_terms w f_P(v) f_Q(v - e_P) C[v - e_P + e_Q].
// With a few thousand rows the two passes through the pair space are two
// launches, each one dependent chain (row tables, ranks, gathers) on a device
// that they do not fill.  Here a wavefront has one row: it lists the terms
// whose pair the row has (a quarter of them on average), then a lane takes
// every 64th.  The occupations are packed bytes, the same in all lanes, the
// target's prefix counts one multiplication a word, its rank M - 1 reads of
// the rank table in LDS; the lanes' sums meet in a fixed order.  What bounds it
// is latency, then the integer work of the targets, which the two passes share
// between the rows of a pair state.  Measured (before: the two passes): N = 6, M
// = 9 8.5 -> 5.0 us, N = 20, M = 4 6.2 -> 3.7, N = 4, M = 13 9.9 -> 5.2 (without
// the list 6.0, 3.1 and 8.7).
template <int NW, bool RC>
__global__ __launch_bounds__(64 * DW) void k_pair_terms(int N, int M, int64_t nc, int nt, const int32_t *IF,
                                                        const int32_t *B, const PairTerm *term, const cplx *h1,
                                                        const cplx *C, cplx *out, PairEpi ep)
{
    constexpr int CW = RC ? 1 : 2;   // doubles of a coefficient
    extern __shared__ __align__(16) unsigned char lds[];
    double *sq = (double *)lds;                            // [N + 3]
    double *wl = sq + N + 3;                               // [nt][CW]
    uint32_t *orb = (uint32_t *)(wl + CW * nt);            // [nt]
    int32_t *Bt = (int32_t *)(orb + nt);                   // [M][N + 1]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, NB = N + 1;
    uint16_t *list = (uint16_t *)(Bt + M * NB) + wave * nt;   // [DW][nt]
    const int64_t i0 = (int64_t)blockIdx.x * DW + wave, i = i0 < nc ? i0 : nc - 1;
    const int vk = lane < M ? IF[i * M + lane] : 0;
    const cplx c0 = C[i];
    const double hr = lane < M ? h1[lane * (pair_h1_stride(M) + 1)].re : 0.0;
    const double hi = !RC && lane < M ? h1[lane * (pair_h1_stride(M) + 1)].im : 0.0;
    for (int x = threadIdx.x; x < nt; x += 64 * DW) {
        orb[x] = term[x].orb;
        wl[CW * x] = term[x].wr;
        if (!RC) wl[CW * x + 1] = term[x].wi;
    }
    for (int x = threadIdx.x; x < M * NB; x += 64 * DW) Bt[x] = B[x];
    for (int x = threadIdx.x; x < N + 3; x += 64 * DW) sq[x] = sqrt((double)x);
    uint64_t pk[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) {
        pk[w] = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) pk[w] |= (uint64_t)(uint32_t)__builtin_amdgcn_readlane(vk, 8 * w + k) << (8 * k);
    }
    const uint32_t one = (uint32_t)__ballot(vk >= 1), two = (uint32_t)__ballot(vk >= 2);
    __syncthreads();
    // the terms whose pair the row has
    int n = 0;
    for (int x0 = 0; x0 < nt; x0 += 64) {
        const int x = x0 + lane;
        const uint32_t o = orb[x < nt ? x : 0], c1 = o & 255, c2 = o >> 8 & 255;
        const bool occ = x < nt && (one >> c2 & 1) && ((c1 < c2 ? one : two) >> c1 & 1);
        const uint64_t m = __ballot(occ);
        if (occ) list[n + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0))] = (uint16_t)x;
        n += __popcll(m);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    auto at = [](const uint64_t *p, int k) {
        uint64_t x = p[0];
#pragma unroll
        for (int w = 1; w < NW; w++) x = k >= 8 * w ? p[w] : x;
        return (int)((uint32_t)(x >> (8 * (k & 7))) & 255u);
    };
    // the diagonal one-body part, an orbital a lane; its sum meets C[v] once, so
    // that an infinite entry does not meet the zeros of the empty orbitals
    double dr = hr * vk, di = hi * vk;
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) {
        dr += __shfl_xor(dr, k, 64);
        if (!RC) di += __shfl_xor(di, k, 64);
    }
    cplx acc = cmake(0, 0);
    if (lane == 0) acc = RC ? cscale(c0, dr) : cfma(cmake(dr, di), c0, acc);
    for (int x = lane; x < n; x += 64) {
        const int id = list[x];
        const uint32_t o = orb[id];
        const int c1 = o & 255, c2 = o >> 8 & 255, q1 = o >> 16 & 255, q2 = o >> 24;
        const cplx w = cmake(wl[CW * id], RC ? 0.0 : wl[CW * id + 1]);
        const int v1 = at(pk, c1), v2 = at(pk, c2);
        uint64_t u[NW];   // v - e_P + e_Q
#pragma unroll
        for (int k = 0; k < NW; k++) {
            u[k] = pk[k];
            u[k] -= (c1 >> 3) == k ? (uint64_t)1 << (8 * (c1 & 7)) : 0;
            u[k] -= (c2 >> 3) == k ? (uint64_t)1 << (8 * (c2 & 7)) : 0;
            u[k] += (q1 >> 3) == k ? (uint64_t)1 << (8 * (q1 & 7)) : 0;
            u[k] += (q2 >> 3) == k ? (uint64_t)1 << (8 * (q2 & 7)) : 0;
        }
        const int u1 = at(u, q1), u2 = at(u, q2);
        // rank = nc - 1 - sum_{j >= 1} B[j][particles below j]; the counts fit
        // a byte (N <= MCPI_MAXN)
        uint32_t s = 0, below = 0;
#pragma unroll
        for (int k = 0; k < NW; k++) {
            const uint64_t p = u[k] * 0x0101010101010101ull + below * 0x0101010101010101ull;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (8 * k + j + 1 < M) s += (uint32_t)Bt[(8 * k + j + 1) * NB + (int)(p >> (8 * j) & 255)];
            below = (uint32_t)(p >> 56);
        }
        const double f = sq[c1 < c2 ? v1 : v1 - 1] * sq[v2] * (sq[q1 < q2 ? u1 : u1 - 1] * sq[u2]);
        const cplx x0 = C[(uint32_t)(nc - 1) - s];
        if (RC) {
            acc.re = fma(w.re * f, x0.re, acc.re);
            acc.im = fma(w.re * f, x0.im, acc.im);
        } else {
            acc = cfma(cscale(w, f), x0, acc);
        }
    }
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) {
        acc.re += __shfl_xor(acc.re, k, 64);
        acc.im += __shfl_xor(acc.im, k, 64);
    }
    if (ep.partial) {
        double re = 0, im = 0;
        if (i0 < nc) {
            const cplx x = ep.lvec[(int64_t)*ep.it * nc + i];
            const double beta = *ep.beta;
            acc.re -= beta * x.re;
            acc.im -= beta * x.im;
            re = c0.re * acc.re + c0.im * acc.im;
            im = c0.re * acc.im - c0.im * acc.re;
        }
        double *red = (double *)lds;   // (over the tables, which are done with)
        __syncthreads();
        if (lane == 0) {
            red[2 * wave] = re;
            red[2 * wave + 1] = im;
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            double s = 0;
            for (int w = 0; w < DW; w++) s += red[2 * w + threadIdx.x];
            ep.partial[2 * blockIdx.x + threadIdx.x] = s;
        }
    }
    if (lane == 0 && i0 < nc) out[i0] = acc;
}

template <int NW>
mcpi_status launch_pair_terms(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, hipStream_t st, PairEpi *e)
{
    const size_t sm = sizeof(double) * (b.N + 3 + (c.real ? 1 : 2) * c.pznt) + 4 * (size_t)(c.pznt + b.M * (b.N + 1)) +
                      2 * (size_t)DW * c.pznt;
    const dim3 grid((unsigned)((b.nc + DW - 1) / DW)), blk(64 * DW);
    PairEpi ep{};
    if (e && grid.x <= (unsigned)e->cap) {
        e->blocks = (int)grid.x;
        ep = *e;
    }
    if (c.real)
        hipLaunchKernelGGL((k_pair_terms<NW, true>), grid, blk, sm, st, b.N, b.M, b.nc, c.pznt, b.IF, b.B, c.pzterm,
                           c.ph1, C, out, ep);
    else
        hipLaunchKernelGGL((k_pair_terms<NW, false>), grid, blk, sm, st, b.N, b.M, b.nc, c.pznt, b.IF, b.B, c.pzterm,
                           c.ph1, C, out, ep);
    MCPI_HIP(hipGetLastError());
    return MCPI_OK;
}

}  // namespace

// complex entries of the pair-space workspace of a basis: Y1 (M rows of
// NC(N-1, M), for N = 1 only), then Y2 (pair_stride(M) rows of
// pair_ld(NC(N-2, M)) entries)
size_t pair_workspace_entries(int N, int M)
{
    const int64_t nu1 = N == 1 ? nc_of(N - 1, M) : 0, nu2 = N >= 2 ? nc_of(N - 2, M) : 0;
    return (size_t)M * nu1 + (size_t)pair_stride(M) * pair_ld(nu2);
}

bool pair_applicable(const BasisDev &b, const HamCoefDev &c)
{
    // (the output pass reads Y1 and Y2 columns as buffers of < 2 GiB:
    // NC(N-1, M) >= NC(N-2, M) entries of 16 bytes)
    return c.ph1 && (b.N < 2 || (c.pwf && b.occ2)) && b.M >= 3 && b.M <= MCPI_PAIR_MAXM && !b.perm && b.IF && b.nc <= INT32_MAX &&
           b.N <= MCPI_MAXN && (b.N < 1 || nc_of(b.N - 1, b.M) < ((int64_t)1 << 27));
}

mcpi_status launch_pair(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                        hipStream_t st, PairEpi *e)
{
    MCPI_ARG(pair_applicable(b, c), "the pair-space H.v does not apply to this basis");
    return b.M <= 9 ? launch_pair_a(b, c, C, out, ws, st, e) : launch_pair_b(b, c, C, out, ws, st, e);
}

// By terms while every row's wavefront is resident at once (32 a CU); us a
// H.v through the pair space and by terms: N = 6, M = 9 (3,003 rows) 8.5, 5.0;
// N = 6, M = 11 (8,008) 9.4, 9.0; N = 8, M = 9 (12,870) 8.8, 11.0.
int64_t pair_terms_rows()
{
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return (int64_t)32 * ncu;
}

bool pairz_applicable(const BasisDev &b, const HamCoefDev &c)
{
    return c.pza && c.pzR > 0 && b.occ2 && b.M >= 3 && b.M <= MCPI_PAIRZ_MAXM && !b.perm && b.IF && b.nc <= INT32_MAX &&
           b.N >= 2 && b.N <= MCPI_MAXN && nc_of(b.N - 1, b.M) < ((int64_t)1 << 27);
}

static mcpi_status launch_pairz_any(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C,
                                    cplx *out, int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    if (b.M <= 9) return launch_pairz_a(b, c, mv, chunks, C, out, mC, mK, ws, st, e);
    if (b.M <= 13) return launch_pairz_b(b, c, mv, chunks, C, out, mC, mK, ws, st, e);
    if (b.M <= 19) return launch_pairz_c(b, c, mv, chunks, C, out, mC, mK, ws, st, e);
    return launch_pairz_d(b, c, mv, chunks, C, out, mC, mK, ws, st, e);
}

mcpi_status launch_pairz(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                        hipStream_t st, PairEpi *e)
{
    MCPI_ARG(pairz_applicable(b, c), "the factorized pair-space H.v does not apply to this basis and Hamiltonian");
    if (pairz_by_terms(c))   // (there are terms on bases of few rows only)
        return b.M <= 8    ? launch_pair_terms<1>(b, c, C, out, st, e)
               : b.M <= 16 ? launch_pair_terms<2>(b, c, C, out, st, e)
                           : launch_pair_terms<3>(b, c, C, out, st, e);
    MCPI_ARG(ws, "no workspace for the factorized pair-space H.v");
    return launch_pairz_any(b, c, 1, 1, C, out, 0, 0, ws, st, e);
}

mcpi_status launch_pairz_multi(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                               int64_t mC, int64_t mK, cplx *ws, hipStream_t st)
{
    MCPI_ARG(pairz_applicable(b, c) && b.M <= MCPI_PAIRZ_MULTI_MAXM && (mv == 2 || mv == 4),
             "the factorized pair form for several members does not apply");
    MCPI_ARG(mK % 16 == 0 && mC >= b.nc && chunks >= 1 && chunks <= 65535, "member strides and chunks");
    return launch_pairz_any(b, c, mv, chunks, C, out, mC, mK, ws, st, nullptr);
}

}  // namespace mcpi

// H.v of h through the pair space on every size, as if it had more terms than
// are kept; what was tuned with them is tuned again (for tests; not part of the
// public interface).
extern "C" mcpi_status mcpi_hip_ham_drop_terms(mcpi_ham h)
{
    MCPI_ARG(h, "null Hamiltonian");
    h->c.pznt = 0;
    h->tuned[0] = h->tuned[1] = 0;
    return MCPI_OK;
}
