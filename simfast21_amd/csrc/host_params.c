/* Host logic that needs no GPU: parameter file parsing, the radius ladder,
 * the ball bound and the background cosmology of the 21-cm step.  Part of
 * libsf21hii. */
#define _GNU_SOURCE
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "host_params.h"

#define SF21_PI 3.1415926535897932385E0 /* Input_variables.h:10 */

const char *sf21_strerror(int code) {
  switch (code) {
    case SF21_OK: return "ok";
    case SF21_ERR_ARG: return "invalid argument or unsupported size";
    case SF21_ERR_ALLOC: return "allocation failed";
    case SF21_ERR_HIP: return "HIP runtime error";
    case SF21_ERR_IO: return "file missing, unreadable or short";
    case SF21_ERR_FORMAT: return "malformed parameter file";
    default: return "unknown error";
  }
}

static void set_msg(char *msg, int cap, const char *text) {
  if (msg && cap > 0) {
    strncpy(msg, text, (size_t)cap - 1);
    msg[cap - 1] = 0;
  }
}

/* Input_variables.c:16-141 for the keys get_HIIbubbles reads.
 * - lines whose first character is '#' or '\n' are skipped (:39);
 * - any other line must contain '=' (:40), which becomes a blank, and must
 *   yield two whitespace-separated tokens (:42-43) -- so text after the
 *   value (a trailing comment) is ignored;
 * - unknown keys are ignored; T/F flags accept exactly "T" or "F";
 * - derived values as :121-133. */
int sf21_params_read(const char *base_dir, sf21_params *p, char *msg, int msg_cap) {
  char path[4096], line[256], key[256], val[256], *eq;
  FILE *f;
  if (!base_dir || !p) return SF21_ERR_ARG;
  memset(p, 0, sizeof(*p));
  snprintf(path, sizeof(path), "%s/simfast21.ini", base_dir);
  f = fopen(path, "r");
  if (!f) {
    set_msg(msg, msg_cap, "\nThe parameter file simfast21.ini cannot be open. Exit...\n");
    return SF21_ERR_IO;
  }
  while (fgets(line, sizeof(line), f) != NULL) {
    int nt;
    if (line[0] == '#' || line[0] == '\n') continue;
    eq = strchr(line, '=');
    if (eq) *eq = ' ';
    nt = eq ? sscanf(line, "%255s %255s", key, val) : 0;
    if (!eq || nt != 2) {
      char buf[400];
      snprintf(buf, sizeof(buf), "Wrong format! Exiting...\n%s\n", line);
      set_msg(msg, msg_cap, buf);
      fclose(f);
      return SF21_ERR_FORMAT;
    }
    if (!strcmp(key, "nthreads")) p->nthreads = atoi(val);
    else if (!strcmp(key, "dz")) p->dz = atof(val);
    else if (!strcmp(key, "zmax")) p->zmax = atof(val);
    else if (!strcmp(key, "zmin")) p->zmin = atof(val);
    else if (!strcmp(key, "sim_length")) p->box_len = atof(val);
    else if (!strcmp(key, "N_halo")) p->n_halo = atoi(val);
    else if (!strcmp(key, "N_smoothed")) p->n = atoi(val);
    else if (!strcmp(key, "hubble")) p->hubble = atof(val);
    else if (!strcmp(key, "fesc")) p->fesc = atof(val);
    else if (!strcmp(key, "Ion_cutoff")) p->ion_cutoff = atof(val);
    else if (!strcmp(key, "bubble_Rmax")) p->bubble_rmax = atof(val);
    else if (!strcmp(key, "bubble_Nbins")) p->bubble_nbins = atoi(val);
    else if (!strcmp(key, "use_SFR")) {
      if (!strcmp(val, "T")) p->use_sfr = 1;
      if (!strcmp(val, "F")) p->use_sfr = 0;
    }
    else if (!strcmp(key, "Vel_comp")) p->vel_comp = atoi(val);
    else if (!strcmp(key, "omega_matter")) p->omega_m = atof(val);
    else if (!strcmp(key, "omega_baryon")) p->omega_b = atof(val);
    else if (!strcmp(key, "omega_lambda")) p->omega_lambda = atof(val);
    else if (!strcmp(key, "Zminsfr")) p->zmin_sfr = atof(val);
    else if (!strcmp(key, "use_Lya_xrays")) {
      if (!strcmp(val, "T")) p->use_lya_xrays = 1;
      if (!strcmp(val, "F")) p->use_lya_xrays = 0;
    }
    else if (!strcmp(key, "Original_nldensity_box")) {
      if (!strcmp(val, "T")) p->save_original_nl = 1;
      if (!strcmp(val, "F")) p->save_original_nl = 0;
    }
  }
  fclose(f);
  p->box_len = p->box_len * p->hubble;
  p->bubble_rmax = p->bubble_rmax * p->hubble;
  if (p->bubble_rmax > p->box_len / 2.) p->bubble_rmax = p->box_len / 2.;
  p->dk = 2 * SF21_PI / p->box_len;
  p->dx_halo = p->n_halo ? p->box_len / p->n_halo : 0.0;
  p->dx = p->n ? p->box_len / p->n : 0.0;
  if (p->dz != 0.0) {
    p->zmin = p->zmax - p->dz * (double)ceil((p->zmax - p->zmin) / p->dz);
    /* Input_variables.c:137-139 */
    p->zmin_sfr = p->zmax - p->dz * (double)ceil((p->zmax - p->zmin_sfr) / p->dz);
    if (p->zmin_sfr < p->zmin) p->zmin_sfr = p->zmin;
  }
  set_msg(msg, msg_cap, "");
  return SF21_OK;
}

/* ---- background cosmology (auxiliary.c:224-303) ----
 * H(z) = h H0 sqrt(Om (1+z)^3 + OL) in 1/s, H0 = 3.24078e-18 h/s
 * (Input_variables.h:108); the growth factor is H(z)/H(0) I(z)/I(0) with
 * I(z) the midpoint sum of (1+z')/(H(z')/H(0))^3 over [z, z + 100) in steps
 * of 1e-3 (the loop variable accumulated in FP64 as the reference does);
 * dD/dt the central difference of step 1e-3 in z times dz/dt = -H(z)(1+z). */
#define SF21_H0 3.24078e-18

double sf21_hubble_z(const sf21_params *p, double z) {
  return p->hubble * SF21_H0 * sqrt(p->omega_m * (1. + z) * (1. + z) * (1. + z) + p->omega_lambda);
}

/* Midpoints z, z + dz, ... below end, each the rounded sum of the one before
 * and dz.  Inside a binade the spacing of the doubles is constant, so every
 * addition of dz advances by the same multiple d of it (once two steps in a row
 * agree: a tie, dz half way between two multiples, goes by the parity, which
 * then no longer changes) and z + m d is exact: runs of values without the
 * chain of additions. */
#define GROWTH_DZ 0.001
#define GROWTH_BLOCK 256
typedef struct {
  double z, end, d;
  long left; /* values left in the run */
} growth_seq;

static int growth_fill(growth_seq *q, double *zs) {
  int n = 0;
  while (n < GROWTH_BLOCK && q->z < q->end) {
    if (q->left == 0) {
      const double z = q->z, d = (z + GROWTH_DZ) - z, z1 = z + d;
      if (z1 == z) { /* dz below the spacing at z */
        q->z = q->end;
        break;
      }
      q->left = 1;
      if (z >= 0x1p-6 && (z1 + GROWTH_DZ) - z1 == d) {
        const double top = ldexp(1.0, ilogb(z) + 1), lim = top < q->end ? top : q->end;
        long c = (long)((lim - z) / d);
        while (c > 1 && !(z + (c - 1) * d < lim)) c--;
        while (z + c * d < lim) c++;
        if (c > 1) q->left = c;
      }
      q->d = d;
    }
    const int c = q->left < GROWTH_BLOCK - n ? (int)q->left : GROWTH_BLOCK - n;
    for (int m = 0; m < c; m++) zs[n + m] = q->z + m * q->d;
    n += c;
    q->left -= c;
    q->z = q->left ? q->z + c * q->d : zs[n - 1] + GROWTH_DZ;
  }
  return n;
}

/* (1+z)/(H(z)/H(0))^3 of a block, zero behind its n values: one square root
 * and four divisions a term, in vector units where the CPU has wide ones.
 * Every operation rounds by itself, as in a loop over single values. */
static inline __attribute__((always_inline)) void growth_terms_body(const sf21_params *p, double h0,
                                                                    int n, double *zt) {
  const double om = p->omega_m, ol = p->omega_lambda, a = p->hubble * SF21_H0;
  for (int m = n; m < GROWTH_BLOCK; m++) zt[m] = 0.;
  for (int m = 0; m < GROWTH_BLOCK; m++) {
    const double z = zt[m], z1 = 1. + z;
    const double e = a * sqrt(om * z1 * z1 * z1 + ol) / h0;
    zt[m] = z1 / e / e / e;
  }
  for (int m = n; m < GROWTH_BLOCK; m++) zt[m] = 0.;
}
static void growth_terms_base(const sf21_params *p, double h0, int n, double *zt) {
  growth_terms_body(p, h0, n, zt);
}
#ifdef __x86_64__
__attribute__((target("avx2"))) static void growth_terms_avx2(const sf21_params *p, double h0, int n,
                                                              double *zt) {
  growth_terms_body(p, h0, n, zt);
}
__attribute__((target("avx512f,prefer-vector-width=512"))) static void growth_terms_avx512(
    const sf21_params *p, double h0, int n, double *zt) {
  growth_terms_body(p, h0, n, zt);
}
#endif

/* D(z[k]), k < nz <= 3, in one sweep together with the integral at 0: the
 * sums, chains of dependent additions in ascending z, run side by side.  Bound
 * by the divider: an integral of 1e5 terms 0.085 ms with 512-bit vectors, 0.145
 * with 256-bit ones, 0.48 one value at a time (EPYC). */
void sf21_growth_many(const sf21_params *p, int nz, const double *z, double *growth) {
  void (*terms)(const sf21_params *, double, int, double *) = growth_terms_base;
  const double h0 = sf21_hubble_z(p, 0.);
  double s[4] = {0., 0., 0., 0.};
  double buf[4][GROWTH_BLOCK];
  growth_seq q[4];
  int more = 1;
#ifdef __x86_64__
  if (__builtin_cpu_supports("avx512f")) terms = growth_terms_avx512;
  else if (__builtin_cpu_supports("avx2")) terms = growth_terms_avx2;
#endif
  memset(buf, 0, sizeof(buf));
  for (int k = 0; k <= nz; k++) {
    const double zz = k < nz ? z[k] : 0.;
    q[k] = (growth_seq){zz + GROWTH_DZ / 2., zz + 100., 0., 0};
  }
  while (more) {
    more = 0;
    for (int k = 0; k <= nz; k++) {
      const int n = growth_fill(&q[k], buf[k]);
      terms(p, h0, n, buf[k]);
      if (n) more = 1;
    }
    if (more)
      for (int m = 0; m < GROWTH_BLOCK; m++)
        for (int k = 0; k < 4; k++) s[k] += buf[k][m];
  }
  for (int k = 0; k < nz; k++)
    growth[k] = sf21_hubble_z(p, z[k]) / h0 * (s[k] * GROWTH_DZ) / (s[nz] * GROWTH_DZ);
}

double sf21_growth(const sf21_params *p, double z) {
  double d;
  sf21_growth_many(p, 1, &z, &d);
  return d;
}

/* from D(z + dz/2) and D(z - dz/2) */
double sf21_dgrowth_of(const sf21_params *p, double z, double hi, double lo) {
  return (hi - lo) / GROWTH_DZ * (-sf21_hubble_z(p, z) * (1. + z));
}

double sf21_dgrowth_dt(const sf21_params *p, double z) {
  const double zs[2] = {z + GROWTH_DZ / 2., z - GROWTH_DZ / 2.};
  double d[2];
  sf21_growth_many(p, 2, zs, d);
  return sf21_dgrowth_of(p, z, d[0], d[1]);
}

int sf21_ladder(double rmax, double dx, int nbins, double *radii, int cap, int *n_main) {
  double bfactor, R;
  int k = 0, m;
  if (!(dx > 0) || nbins <= 0 || cap < 0) return SF21_ERR_ARG;
  bfactor = pow(10.0, log10(rmax / dx) / nbins);
  if (!(bfactor > 1.0)) return SF21_ERR_ARG;
  R = rmax;
  while (R >= 2 * dx) {
    if (k >= cap) return SF21_ERR_ARG;
    if (radii) radii[k] = R;
    k++;
    R /= bfactor;
  }
  m = k;
  while (R >= dx) {
    if (k >= cap) return SF21_ERR_ARG;
    if (radii) radii[k] = R;
    k++;
    R /= bfactor;
  }
  if (n_main) *n_main = m;
  return k;
}

long sf21_ball_d2max(double R, double dx) {
  long m;
  if (!(R >= 0) || !(dx > 0)) return -1;
  m = (long)floor((R / dx) * (R / dx));
  while (m > 0 && !(sqrt((double)m) * dx <= R)) m--;
  while (sqrt((double)(m + 1)) * dx <= R) m++;
  return m;
}
