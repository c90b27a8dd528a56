// solver.hpp — stage orchestration entry points.
#pragma once

#include "context.hpp"

namespace cuev {

void options_defaults(cuev_options &o);

// Smallest merge (rows) of the device D&C that waits for a back-transform running
// beside it (the gate of dc_solve).
int kDcGateFrom(int n);

// Order from which the device D&C beats host LAPACK's: whole solves of n = 129, 140 and 159 take 1.20,
// 1.33 and 1.69 ms with ?stedc in FP64 (0.97, 1.12 and 1.43 in FP32) and 1.08, 1.12 and 1.30 (0.99,
// 1.05 and 1.27) with the device form; at n = 1000 the stage alone takes 19.7 (11.5) and 1.3
// (1.0) ms. Up to 128 only solves with stage options get here.
constexpr int kDeviceDcFrom = 129;

// D&C on device (d, e): eval <- eigenvalues, evec (ld ldv) <- Q_d; host ?stedc
// or the device-resident form, as ctx.dc_mode says.
template <typename T>
int tridi_dc(Context<T> &ctx, T *d, T *e, T *eval, T *evec, i64 ldv, double *dc_ms);
// evec <- Q_s Q_b evec (direct order).
template <typename T>
int back_transform(Context<T> &ctx, const T *Y, const T *W, const T *U, T *evec,
                   cuev_solve_timer *timer);
// Eigenvalues il..iu only (0-based, ascending) into eval[0 .. iu-il]: DBBR, bulge
// chasing, then Sturm multisection on the GPU; no back-transform.
template <typename T>
int solve_values(Context<T> &ctx, T *A, int il, int iu, T *eval, cuev_solve_timer *timer);
// Full solve in the precision T.
template <typename T>
int solve_native(Context<T> &ctx, T *A, T *eval, T *evec, cuev_solve_timer *timer, int bt_mode,
                 int dc_mode, int dc_leaf);

} // namespace cuev
