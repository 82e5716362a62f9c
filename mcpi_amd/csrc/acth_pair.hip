// Pair-space H.v (schedules 6 and 7): where it applies, and the launch for a
// number of orbitals.  The kernels are in acth_pair.h, compiled for their M in
// acth_pair_a.hip (3..9) to acth_pair_d.hip (20..24).
#include <hip/hip_runtime.h>

#include "mcpi_internal.h"

namespace mcpi {

#define MCPI_PAIR_ARGS const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws, hipStream_t st
#define MCPI_PAIRZ_ARGS const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out, \
                        int64_t mC, int64_t mK, cplx *ws, hipStream_t st
mcpi_status launch_pair_a(MCPI_PAIR_ARGS);
mcpi_status launch_pair_b(MCPI_PAIR_ARGS);
mcpi_status launch_pairz_a(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_b(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_c(MCPI_PAIRZ_ARGS);
mcpi_status launch_pairz_d(MCPI_PAIRZ_ARGS);

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
                        hipStream_t st)
{
    MCPI_ARG(pair_applicable(b, c), "the pair-space H.v does not apply to this basis");
    return b.M <= 9 ? launch_pair_a(b, c, C, out, ws, st) : launch_pair_b(b, c, C, out, ws, st);
}

bool pairz_applicable(const BasisDev &b, const HamCoefDev &c)
{
    return c.pza && c.pzR > 0 && b.occ2 && b.M >= 3 && b.M <= MCPI_PAIRZ_MAXM && !b.perm && b.IF && b.nc <= INT32_MAX &&
           b.N >= 2 && b.N <= MCPI_MAXN && nc_of(b.N - 1, b.M) < ((int64_t)1 << 27);
}

static mcpi_status launch_pairz_any(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C,
                                    cplx *out, int64_t mC, int64_t mK, cplx *ws, hipStream_t st)
{
    if (b.M <= 9) return launch_pairz_a(b, c, mv, chunks, C, out, mC, mK, ws, st);
    if (b.M <= 13) return launch_pairz_b(b, c, mv, chunks, C, out, mC, mK, ws, st);
    if (b.M <= 19) return launch_pairz_c(b, c, mv, chunks, C, out, mC, mK, ws, st);
    return launch_pairz_d(b, c, mv, chunks, C, out, mC, mK, ws, st);
}

mcpi_status launch_pairz(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                        hipStream_t st)
{
    MCPI_ARG(pairz_applicable(b, c), "the factorized pair-space H.v does not apply to this basis and Hamiltonian");
    return launch_pairz_any(b, c, 1, 1, C, out, 0, 0, ws, st);
}

mcpi_status launch_pairz_multi(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                               int64_t mC, int64_t mK, cplx *ws, hipStream_t st)
{
    MCPI_ARG(pairz_applicable(b, c) && b.M <= MCPI_PAIRZ_MULTI_MAXM && (mv == 2 || mv == 4),
             "the factorized pair form for several members does not apply");
    MCPI_ARG(mK % 16 == 0 && mC >= b.nc && chunks >= 1 && chunks <= 65535, "member strides and chunks");
    return launch_pairz_any(b, c, mv, chunks, C, out, mC, mK, ws, st);
}

}  // namespace mcpi
