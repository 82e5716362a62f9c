// Pair-space H.v kernels (acth_pair.h) for M = 10..13.
#include "acth_pair.h"

namespace mcpi {

mcpi_status launch_pair_b(const BasisDev &b, const HamCoefDev &c, const cplx *C, cplx *out, cplx *ws,
                          hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIR_CASE(10) MCPI_PAIR_CASE(11) MCPI_PAIR_CASE(12)
    default: return MCPI_ERR_ARG;
    }
}

mcpi_status launch_pairz_b(const BasisDev &b, const HamCoefDev &c, int mv, int chunks, const cplx *C, cplx *out,
                           int64_t mC, int64_t mK, cplx *ws, hipStream_t st, PairEpi *e)
{
    switch (b.M) {
        MCPI_PAIRZ_MV_CASE(10) MCPI_PAIRZ_MV_CASE(11) MCPI_PAIRZ_MV_CASE(12) MCPI_PAIRZ_MV_CASE(13)
    default: return MCPI_ERR_ARG;
    }
}

}  // namespace mcpi
