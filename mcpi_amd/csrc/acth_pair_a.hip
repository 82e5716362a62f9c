// Pair-space H.v kernels (acth_pair.h) for M = 3..9.
#include "acth_pair.h"

namespace mcpi {

mcpi_status launch_pair_a(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                          hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIR_CASE(3) MCPI_PAIR_CASE(4) MCPI_PAIR_CASE(5) MCPI_PAIR_CASE(6) MCPI_PAIR_CASE(7) MCPI_PAIR_CASE(8) MCPI_PAIR_CASE(9)
    default: return MCPI_ERR_ARG;
    }
}

mcpi_status launch_pairz_a(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                           int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIRZ_MV_CASE(3) MCPI_PAIRZ_MV_CASE(4) MCPI_PAIRZ_MV_CASE(5) MCPI_PAIRZ_MV_CASE(6)
        MCPI_PAIRZ_MV_CASE(7) MCPI_PAIRZ_MV_CASE(8) MCPI_PAIRZ_MV_CASE(9)
    default: return MCPI_ERR_ARG;
    }
}

}  // namespace mcpi
