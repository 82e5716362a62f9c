// Host test of the coefficient block (build_coefficients in acth.hip): the
// tables that the batched H.v reads at a fixed stride from the first member's
// have the same offsets in every Hamiltonian with M orbitals, whatever the
// form of the pair matrix, and hold what a block of their own would.  The
// device allocation and copy are replaced by host ones.  Prints "all passed" or
// the first difference.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "mcpi_internal.h"

using namespace mcpi;

extern "C" hipError_t hipMalloc(void **p, size_t n)
{
    *p = malloc(n);
    return hipSuccess;
}
extern "C" hipError_t hipFree(void *p)
{
    free(p);
    return hipSuccess;
}
extern "C" hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}

// Ho diagonal; Hint couples pairs of total momentum lo .. hi (lo > hi: none),
// all of one momentum alike (factorized), or unalike (not factorized)
static HamCoefDev build(int N, int M, int lo, int hi, bool alike, char **block, size_t *bytes)
{
    std::vector<cplx> Ho(M * M, cmake(0, 0)), Hi((size_t)M * M * M * M, cmake(0, 0));
    for (int k = 0; k < M; k++) Ho[k + M * k] = cmake(1.0 + k, 0);
    for (int a = 0; a < M; a++)
        for (int b = 0; b < M; b++)
            for (int d = 0; d < M; d++)
                for (int e = 0; e < M; e++)
                    if (a + b == d + e && a + b >= lo && a + b <= hi)
                        Hi[a + M * (b + M * (d + (size_t)M * e))] = cmake(alike ? 5.0 : 5.0 + a * b + d * e, 0);
    HamCoefDev c;
    memset(&c, 0, sizeof c);
    void *p = nullptr;
    if (build_coefficients(M, Ho.data(), Hi.data(), &c, &p, bytes, N) != MCPI_OK) {
        std::printf("build failed\n");
        exit(1);
    }
    *block = (char *)p;
    return c;
}

int main()
{
    for (int M = 3; M <= 13; M++) {
        char *b0;
        size_t n0;
        const HamCoefDev c0 = build(5, M, 0, 2 * M, true, &b0, &n0);
        for (int N : {1, 5})
            for (int lo = 0; lo <= 4; lo++)
                for (int hi : {2 * M, 2 * M - 4, lo - 1})
                    for (bool alike : {true, false}) {
                        char *b;
                        size_t n;
                        const HamCoefDev c = build(N, M, lo, hi, alike, &b, &n);
                        const void *x0[] = {c0.dk, c0.d1, c0.d2, c0.A0, c0.A, c0.ot, c0.tt, c0.otc, c0.ttc, c0.nz_c, c0.ph1,
                                            c0.nz_1j, c0.nz_ot, c0.nz_tt, c0.m1j, c0.ot_off, c0.tt_off, c0.nz_e, c0.pql};
                        const void *x[] = {c.dk, c.d1, c.d2, c.A0, c.A, c.ot, c.tt, c.otc, c.ttc, c.nz_c, c.ph1,
                                           c.nz_1j, c.nz_ot, c.nz_tt, c.m1j, c.ot_off, c.tt_off, c.nz_e, c.pql};
                        for (size_t t = 0; t < sizeof x / sizeof x[0]; t++)
                            if ((const char *)x[t] - b != (const char *)x0[t] - b0) {
                                std::printf("M=%d N=%d lo=%d hi=%d alike=%d: table %zu at %td, not %td (%zu and %zu bytes)\n", M, N,
                                            lo, hi, (int)alike, t, (const char *)x[t] - b, (const char *)x0[t] - b0, n, n0);
                                return 1;
                            }
                        // the last table lies inside, aligned
                        if (c.pzblk && ((size_t)c.pza % 16 || (char *)(c.pzoff + c.pzR + 1) > b + n)) {
                            std::printf("M=%d N=%d lo=%d: factorized form's tables\n", M, N, lo);
                            return 1;
                        }
                        free(b);
                    }
        free(b0);
    }
    std::printf("all passed\n");
    return 0;
}
