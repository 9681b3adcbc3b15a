// Dip estimation of a 2-D section that stays resident on the chip (dip2.hip).
#pragma once
#include "dipcore.hpp"

// dipc with n3 == 1 in one launch.  *ran = 0: the section or the radii do not
// fit, or the stream is being captured; nothing was done.  mask (one byte a
// sample) and init may be null; rec (device, REC_INTS ints, may be null)
// receives the iterations' decisions.
constexpr int REC_INTS = 2 * 64;
int dip2_resident(sh_ctx *ctx, int n1, int n2, int r1, int r2, int order, const float *x, const unsigned char *mask,
                  const float *init, int niter, int liter, int *rec, float *dip, int *ran);
