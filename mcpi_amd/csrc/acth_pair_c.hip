// Pair-space H.v kernels (acth_pair.h) for M = 14..19.
#include "acth_pair.h"

namespace mcpi {

mcpi_status launch_pairz_c(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                           int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIRZ_CASE(14) MCPI_PAIRZ_CASE(15) MCPI_PAIRZ_CASE(16) MCPI_PAIRZ_CASE(17)
        MCPI_PAIRZ_CASE(18) MCPI_PAIRZ_CASE(19)
    default: return MCPI_ERR_ARG;
    }
}

}  // namespace mcpi
