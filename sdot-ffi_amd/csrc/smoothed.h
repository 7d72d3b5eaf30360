// The flexible CG preconditioned by a smoothed-aggregation V-cycle: the default solver of the Newton systems.
#pragma once

#include "multigrid.h"
#include "graph_cache.h"

namespace sdot_amd {

/// `A d = b` from `d = 0` to the relative residual `tol` in at most `maxit` iterations, the outer iteration in FP64, the cycle in
/// FP32 ( `valf`, `diaf`: the rows' values and diagonal in float, laid out as `L`'s ) or in FP64 ( both null ). `prev_its`: the
/// iterations of the caller's last system ( 0: unknown ), launched without waiting in between. `drop`: how much more than usual of the
/// prolongations' small entries is dropped ( 1: none; the result is `bad` when a coarse row outgrows its room )
FcgResult smoothed_solve( const Csr &L, const float *valf, const float *diaf, const double *b, double *d, double tol, int maxit,
                          const MgOptions &o, hipStream_t st, int &nb_levels, int prev_its, double drop );

/// the device bytes of the hierarchy and the vectors of a system of `n` rows ( `wide`: 3D rows ), its values of `s` bytes
double smoothed_bytes( I64 n, bool wide, double s );

/// the rows below which the K-cycle's dense coarsest level is all there is ( the smoothed hierarchy needs a level above its bottom )
constexpr I64 SA_MIN_ROWS = 64;

} // namespace sdot_amd
