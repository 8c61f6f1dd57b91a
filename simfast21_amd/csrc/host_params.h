// Internal to the library: the growth factors of several redshifts in one sweep
// (host_params.c).
#pragma once
#include "../../include/sf21_hii.h"

#ifdef __cplusplus
extern "C" {
#endif
#pragma GCC visibility push(hidden)
// growth[k] = D(z[k]), k < nz <= 3: sf21_growth of each, bit for bit
void sf21_growth_many(const sf21_params *p, int nz, const double *z, double *growth);
// dD/dt at z from D(z + 0.0005) and D(z - 0.0005)
double sf21_dgrowth_of(const sf21_params *p, double z, double hi, double lo);
#pragma GCC visibility pop
#ifdef __cplusplus
}
#endif
