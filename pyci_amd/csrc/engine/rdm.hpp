// Accumulators shared by the density-matrix kernels (rdm.hip, rdm_full.hip).
#pragma once

#include "internal.hpp"

namespace pe {

// Sizes and the layout of one accumulator copy: a1, b1 (n x n, single excitations one
// way round), caa, cbb (pairs p < q by pairs r < s, each connected pair of strings or
// determinants once), cab (n x n by pairs q <= s); GenCI has a1 and caa of its one string.
struct RfShape {
    int n, nup, ndn, na, nb;
    int ldc, ldt;  // row strides of C and C^T: string counts rounded up to 16, padding zero
    int npd, npr;  // pairs p < q, pairs q <= s
    const i64 *binom;
    i64 oaa, obb, oab, stride;
    bool genci;
};

RfShape rf_shape(const pyci_wfn *w);
// copies of the accumulators that blocks take in turn, to spread contention
int rf_copies(const RfShape &S);
void rf_result(pyci_ctx *ctx, const RfShape &S, int R, const double *acc, double *rdm1, double *rdm2);

}  // namespace pe
