// Row tables of the pair space: the states u of N - 2 particles that the pair
// amplitudes <u|a_q a_l|C> run over (density matrices, pair-space H.v).
//
// rank(u + e_q + e_l) = rank(u + 2 e_0) - (S_0(q) - S_1(q)) - (S_1(l) - S_2(l))
// for q <= l, with S_d(x) = sum_{j=1..x} B[j][P_j(u) + d] and P_j(u) the
// particles below orbital j, so a row needs two tables of differences and the
// roots of its occupations.  They are made from the basis's occupation table
// (BasisDev::occ2, one byte per orbital): the B entries of all orbitals are
// read side by side, where unranking the row would walk N + M dependent ones.
#pragma once

#include "mcpi_internal.h"

namespace mcpi {

// One half of the tables of a row with occupations w (bytes, orbital 0
// first): D[o * sd] = S_d(o) - S_{d+1}(o) and G[o * sg] = sqrt(v_o + 1 + d) for
// every orbital o < M; returns S_{d+1}(M - 1).  NW words of w cover M
// orbitals.  d = 0: the tables of q (and of l > q for the roots), d = 1: of l.
// Four orbitals' entries are in flight together (all of them took more
// registers than the products beside leave).
template <int NW>
__device__ inline int32_t pair_row_tables(const uint32_t (&w)[NW], int M, int NB1, const int32_t *Bt, const double *sq,
                                          int d, int32_t *D, int sd, double *G, int sg)
{
    // (an empty statement that takes the sizes: without it what depends on
    // them alone moves out of the caller's loop, and every scalar register
    // goes with it)
    M = __builtin_amdgcn_readfirstlane(M);
    NB1 = __builtin_amdgcn_readfirstlane(NB1);
    asm volatile("" : "+s"(M), "+s"(NB1));
    int p = d;
    int32_t s = 0, s1 = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) {
        if (4 * k >= M) continue;
        int32_t lo[4], hi[4];
        double r[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // (orbitals past M - 1 read its entry again and are not stored)
            const int o = 4 * k + j, b = (o < M ? o : M - 1) * NB1 + p;
            const int v = (int)((w[k] >> (8 * j)) & 255u);
            lo[j] = Bt[b];
            hi[j] = Bt[b + 1];
            r[j] = sq[v + 1 + d];
            p += v;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int o = 4 * k + j;
            if (o >= M) continue;
            if (o) {
                s += lo[j] - hi[j];
                s1 += hi[j];
            }
            D[o * sd] = s;
            G[o * sg] = r[j];
        }
    }
    return s1;
}

// bytes of a row of the occupation table
__host__ __device__ constexpr int occ_stride(int M) { return M <= 16 ? 16 : 32; }

}  // namespace mcpi
