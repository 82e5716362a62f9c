// Pair-space H.v kernels (acth_pair.h) for M = 20..24.
#include "acth_pair.h"

namespace mcpi {

mcpi_status launch_pairz_d(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                           int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIRZ_CASE(20) MCPI_PAIRZ_CASE(21) MCPI_PAIRZ_CASE(22) MCPI_PAIRZ_CASE(23)
        MCPI_PAIRZ_CASE(24)
    default: return MCPI_ERR_ARG;
    }
}

}  // namespace mcpi
