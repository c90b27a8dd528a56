// bulge.hpp — band -> tridiagonal stage.
#pragma once

#include "workspace.hpp"

namespace cuev {

// Bp (2b x n packed band) -> tridiagonal (d[0:n], e[0:n-1], e[n-1] = 0); reflectors stored in
// ws.U (shifted layout). write_band: the tridiagonal matrix is left in Bp as well, whichever form
// of the chase runs; without it Bp's contents are unspecified afterwards.
template <typename T> int bc_chase(Workspace<T> &ws, T *Bp, T *d, T *e, bool write_band = false);

// bytes of ws.chmsg, the message buffers of the resident chase (either precision)
size_t bc_chase_msg_bytes(int n, int b);

} // namespace cuev
