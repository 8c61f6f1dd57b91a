// Fused finder on box sides without a register transform plan: whole-line
// mixed-radix Stockham transforms (first and last stage in HBM, the others
// through LDS), the cell pre-pass packing, and their launchers.
#include "fft_core.h"
#include "kernels.h"
#include "cells.h"

namespace sf21 {

// ------------------------------------------------------------------------
// Generic sizes (box sides with no register plan, e.g. 600 = 8*3*5*5):
// whole-line mixed-radix Stockham transforms, 8 lines per 256-thread block.
// Stage of radix R and span NS (the product of the earlier radices),
// butterfly j < L/R with k = j mod NS: a_r = x[j + r L/R] w^(k r), w =
// exp(-+2 pi i / (NS R)); DFT_R; y[(j/NS) NS R + k + r NS] = a_r -- the
// self-sorting stages of the register transforms.  The first stage reads its
// inputs from HBM and the last writes its outputs there (positions j + r L/R
// in both, so runs of consecutive j stay coalesced); the stages in between
// exchange through one padded LDS line per line (a thread's butterflies are
// read into registers, barrier, written, barrier).  Lanes: rows (axis 0)
// take 32 consecutive butterflies of one line per half wave; the column
// passes (axes 1, 2) take the 8 lines -- adjacent p columns, 64 B runs --
// fastest.  32-bit indices (L^3 <= 2^30).
// ------------------------------------------------------------------------
constexpr int kGenLines = 8;
constexpr int kGenMaxL = 768;

// floor(a / d) for 0 <= a, d <= 2^11 from rd = 1/d rounded to float:
// (a + 1/2)/d lies at least 1/(2d) >= 2^-12 inside an integer interval and
// the product's rounding error is below 2^-12.
__device__ __forceinline__ int gen_div(int a, float rd) {
  return (int)(((float)a + 0.5f) * rd);
}

// twiddles w^(k r), r = 1..R-1, of a stage's butterfly
template <int R, int SIGN>
__device__ __forceinline__ void gen_twiddle(float2* a, int k, int tstep,
                                            const float2* __restrict__ tw) {
#pragma unroll
  for (int r = 1; r < R; ++r) {
    float2 w = tw[k * r * tstep];
    if (SIGN > 0) w.y = -w.y;
    a[r] = cmul(a[r], w);
  }
}

// First stage (radix 8, NS = 1): inputs from HBM.
// Output position o = 8 j + r is kept transposed, at slot r L/8 + j, so that
// the stores of consecutive butterflies are consecutive (a stride-8 store
// pattern conflicts in the LDS banks); the next stage reads position o at
// gen_t1_slot(o).
__device__ __forceinline__ int gen_t1_slot(int o, int lr0) { return (o & 7) * lr0 + (o >> 3); }

// LC (and NSC): the side (and the stage span) as compile-time constants for
// the specialised sides, 0 for the runtime plan.
template <int R, int SIGN, int LC>
__device__ __forceinline__ void gen_first(const GenPlan& P, int jj, float2* line,
                                          const float2* src, unsigned base, unsigned stride) {
  const int L = LC ? LC : P.L, Lr = L / R;
#pragma unroll 2
  for (int j = jj; j < Lr; j += 32) {
    float2 a[R];
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = src[base + (unsigned)(j + r * Lr) * stride];
    Dft<R, SIGN>::run(a);
#pragma unroll
    for (int r = 0; r < R; ++r) line[r * Lr + j] = a[r];
  }
  lds_pin();
  __syncthreads();
}

// Filtered first stage (mode 1) of the i-axis pass: the W of the block's 8
// lines depends on |k|^2 = msq_l + fold(e)^2, so it is evaluated once per
// (line, |fold(e)|) -- 8 (L/2 + 1) values instead of 8 L -- into a table in
// the line buffers, which the stage's stores overwrite only after every
// thread has multiplied its inputs.  The first radix is 8, so a
// thread holds at most (768/8 + 31)/32 = 3 butterflies.
template <int SIGN, int LC>
__device__ __forceinline__ void gen_first_wtab(const GenPlan& P, float2* gsm, float2* line,
                                               int l, int jj, const float2* src, unsigned base,
                                               unsigned stride, int mfix, int p0, float2 kappa) {
  constexpr int R = 8, MAXIT = ((LC ? LC : kGenMaxL) / R + 31) / 32;
  const int L = LC ? LC : P.L, Lr = L / R, H = L / 2 + 1;
  float* wt = reinterpret_cast<float*>(gsm);
  for (int t = threadIdx.x; t < kGenLines * H; t += blockDim.x) {
    const int ll = t / H, f = t - ll * H;
    wt[t] = w_tophat_k(kappa, mfix + fold_sq(p0 + ll, L) + f * f);
  }
  lds_pin();
  __syncthreads();
  float2 a[MAXIT][R];
#pragma unroll
  for (int it = 0; it < MAXIT; ++it) {
    const int j = jj + 32 * it;
    if (j < Lr) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = j + r * Lr;
        const float2 v = src[base + (unsigned)e * stride];
        const float w = wt[l * H + (e <= L / 2 ? e : L - e)];
        a[it][r] = make_float2(v.x * w, v.y * w);
      }
    }
  }
  lds_pin();
  __syncthreads();
#pragma unroll
  for (int it = 0; it < MAXIT; ++it) {
    const int j = jj + 32 * it;
    if (j < Lr) {
      Dft<R, SIGN>::run(a[it]);
#pragma unroll
      for (int r = 0; r < R; ++r) line[r * Lr + j] = a[it][r];
    }
  }
  lds_pin();
  __syncthreads();
}

// Middle stage: all of a thread's butterflies are read before the barrier,
// then written back into the same line.  T1: the stage after the first
// (inputs in the transposed slots).
template <int R, int SIGN, bool T1, int LC, int NSC>
__device__ __forceinline__ void gen_mid(const GenPlan& P, int st, int jj, float2* line,
                                        const float2* __restrict__ tw) {
  constexpr int MAXIT = ((LC ? LC : kGenMaxL) / R + 31) / 32;
  const int L = LC ? LC : P.L, NS = LC ? NSC : P.ns[st], Lr = L / R, tstep = L / (NS * R);
  const float rns = P.rns[st];
  auto quot = [&](int j) { return LC ? (int)((unsigned)j / (unsigned)NSC) : gen_div(j, rns); };
  float2 a[MAXIT][R];
#pragma unroll
  for (int it = 0; it < MAXIT; ++it) {
    const int j = jj + 32 * it;
    if (j < Lr) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int o = j + r * Lr;
        a[it][r] = line[T1 ? gen_t1_slot(o, L >> 3) : o];
      }
      gen_twiddle<R, SIGN>(a[it], j - quot(j) * NS, tstep, tw);
      Dft<R, SIGN>::run(a[it]);
    }
  }
  lds_pin();
  __syncthreads();
#pragma unroll
  for (int it = 0; it < MAXIT; ++it) {
    const int j = jj + 32 * it;
    if (j < Lr) {
      const int q = quot(j), k = j - q * NS;
      float2* y = line + q * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) y[r * NS] = a[it][r];
    }
  }
  lds_pin();
  __syncthreads();
}

// Last stage (NS R = L, k = j): outputs at j + r L/R to HBM.
template <int R, int SIGN, bool T1, int LC, int NSC>
__device__ __forceinline__ void gen_last(const GenPlan& P, int st, int jj, const float2* line,
                                         float2* dst, unsigned base, unsigned stride,
                                         const float2* __restrict__ tw) {
  const int L = LC ? LC : P.L, NS = LC ? NSC : P.ns[st], Lr = L / R, tstep = L / (NS * R);
#pragma unroll 2
  for (int j = jj; j < Lr; j += 32) {
    float2 a[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int o = j + r * Lr;
      a[r] = line[T1 ? gen_t1_slot(o, L >> 3) : o];
    }
    gen_twiddle<R, SIGN>(a, j, tstep, tw);
    Dft<R, SIGN>::run(a);
#pragma unroll
    for (int r = 0; r < R; ++r) dst[base + (unsigned)(j + r * Lr) * stride] = a[r];
  }
}

// 4 waves per SIMD (128 VGPRs): the LDS line buffers allow 4 blocks per CU
// at 600, and the bound (a few spilled registers in the column variants) ran
// 5% faster than 130 VGPRs at 3 waves
// LC = 600: the sample configuration's side with its plan 8, 3, 5, 5 (spans
// 1, 8, 24, 120) and LDS line stride 616 as constants; 0: the runtime plan.
template <int SIGN, int MODE, bool ROWS, int LC>
__global__ __launch_bounds__(256, 4) void k_gen_pass(const float2* src, float2* dst, GenPlan plan,
                                                  int axis, const float2* __restrict__ tw,
                                                  float2 kappa) {
  extern __shared__ float2 gsm[];
  const unsigned L = LC ? (unsigned)LC : (unsigned)plan.L, L2 = L * L;
  // column passes with bit `axis` of plan.xcd: consecutive tiles (which
  // share 128 B lines) on one XCD -- workgroups are dealt round-robin over
  // the 8 XCDs, and the grid (L^2/8 blocks, L a multiple of 8) is a multiple
  // of 8, so the remap is a permutation.  Measured at 600: the filtered i
  // pass 1.30 -> 1.15 ms, the j pass 0.80 -> 0.81 ms (default: i passes
  // only; the autotuner searches the four masks).
  const unsigned blk = (!ROWS && ((plan.xcd >> axis) & 1))
                           ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)
                           : blockIdx.x;
  const int l = ROWS ? (int)(threadIdx.x >> 5) : (int)(threadIdx.x & 7);
  const int jj = ROWS ? (int)(threadIdx.x & 31) : (int)(threadIdx.x >> 3);
  unsigned base, stride;
  if (ROWS) {
    const unsigned row = blk * kGenLines + l;
    base = row * L;
    stride = 1;
  } else {
    const unsigned ntile = L / kGenLines;
    const unsigned outer = blk / ntile;
    const unsigned p = (blk % ntile) * kGenLines + l;
    base = axis == 1 ? outer * L2 + p : outer * L + p;
    stride = axis == 1 ? L : L2;
  }
  float2* line = gsm + l * (LC == 600 ? 616 : plan.lp);
  // the first radix is 8 on every generic side (multiples of 8)
  if constexpr (MODE == 1 && !ROWS) {
    // the filtered pass runs along i only (axis 2: outer = j)
    const unsigned ntile = L / kGenLines;
    gen_first_wtab<SIGN, LC>(plan, gsm, line, l, jj, src, base, stride,
                             fold_sq((int)(blk / ntile), (int)L),
                             (int)((blk % ntile) * kGenLines), kappa);
  } else {
    gen_first<8, SIGN, LC>(plan, jj, line, src, base, stride);
  }
  if constexpr (LC == 600) {
    gen_mid<3, SIGN, true, 600, 8>(plan, 1, jj, line, tw);
    gen_mid<5, SIGN, false, 600, 24>(plan, 2, jj, line, tw);
    gen_last<5, SIGN, false, 600, 120>(plan, 3, jj, line, dst, base, stride, tw);
    return;
  }
  const int last = plan.nst - 1;
#define GMS(R, T) gen_mid<R, SIGN, T, 0, 0>(plan, st, jj, line, tw)
#define GLS(R, T) \
  gen_last<R, SIGN, T, 0, 0>(plan, last, jj, line, dst, base, stride, tw)
  if (last == 1) {
    switch (plan.radix[1]) {
      case 8: GLS(8, true); break;
      case 4: GLS(4, true); break;
      case 2: GLS(2, true); break;
      case 3: GLS(3, true); break;
      default: GLS(5, true); break;
    }
    return;
  }
  {
    const int st = 1;
    switch (plan.radix[1]) {
      case 8: GMS(8, true); break;
      case 4: GMS(4, true); break;
      case 2: GMS(2, true); break;
      case 3: GMS(3, true); break;
      default: GMS(5, true); break;
    }
  }
  for (int st = 2; st < last; ++st) {
    switch (plan.radix[st]) {
      case 8: GMS(8, false); break;
      case 4: GMS(4, false); break;
      case 2: GMS(2, false); break;
      case 3: GMS(3, false); break;
      default: GMS(5, false); break;
    }
  }
  switch (plan.radix[last]) {
    case 8: GLS(8, false); break;
    case 4: GLS(4, false); break;
    case 2: GLS(2, false); break;
    case 3: GLS(3, false); break;
    default: GLS(5, false); break;
  }
#undef GMS
#undef GLS
}

__global__ void k_gen_pack(long n3, const float* __restrict__ a, const float* __restrict__ b,
                           const float* __restrict__ c, CellConsts k,
                           const float* __restrict__ bal, float2* __restrict__ spec) {
  const float sc = bal[0];
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n3;
       i += (long)gridDim.x * blockDim.x) {
    float rec, ion, fr;
    cell_fields(k, a, b, c, i, rec, ion, fr);
    spec[i] = make_float2(rec, ion * sc);
  }
}

// ------------------------------------------------------------------------
// The finder's per-radius passes on these sides, specialised per side: plan,
// spans and iteration counts are compile-time constants (66-112 VGPRs; the
// runtime plan above holds every stage at the largest side's count, 128 with
// spills).  Inverse transforms with the stages of k_gen_pass; the twiddle
// products in the fixed form the compiler gives those.
//
// Per-radius buffer: tiles of G adjacent p columns (G = 16, or 8 on the sides
// that are an odd multiple of 8), element (i, j, p) at ((p/G) n + i) G n + G j
// + p%G, as the register-plan sides' t16 layout.  A piece of 8 columns is half
// a cache line, so at G = 8 up to 512 a line holds the pieces of two i planes:
// ((p/8) n/2 + i/2) 16 n + 16 j + 8 (i%2) + p%8.  All three passes per slice,
// lines shared by two planes against half lines: 360^3 14.0 ms against 15.7,
// 200^3 2.20 against 2.45; at 600^3 the j pass's blocks of 16 lines (75 KiB)
// lose more than the filter pass gains (28.2 + 40.0 + 25.4 ms against 35.1 +
// 32.2 + 23.4).  Tried and slower: neighbouring tiles behind each other along
// i in at most 40 groups (600^3 p pass 30.0 ms against 25.0); j blocks over
// half the columns of a line (600^3 41.0 ms), or over its halves in turn with
// both loaded first (43.9: 155 registers).
// ------------------------------------------------------------------------
#define SF21_GEN_SIDES(X)                                                                  \
  X(16) X(24) X(40) X(48) X(72) X(80) X(120) X(144) X(160) X(200) X(216) X(240) X(288) X(320) \
  X(360) X(384) X(400) X(432) X(480) X(576) X(600) X(640) X(720) X(768)

struct GPlanC {
  int nst = 0;
  int radix[8] = {};
  int ns[8] = {};
};
constexpr GPlanC gplan(int n) {
  GPlanC p;
  int m = n, ns = 1;
  while (m > 1) {
    const int r = m % 8 == 0 ? 8 : m % 4 == 0 ? 4 : m % 2 == 0 ? 2 : m % 3 == 0 ? 3 : 5;
    p.radix[p.nst] = r;
    p.ns[p.nst] = ns;
    ns *= r;
    m /= r;
    ++p.nst;
  }
  return p;
}
constexpr int gen_group(int n) { return n % 16 == 0 ? 16 : 8; }
// Half lines of two planes side by side; columns of a tile's rows.
constexpr bool gen_pair(int n) { return gen_group(n) == 8 && n <= 512; }
constexpr int gen_row(int n) { return gen_pair(n) ? 16 : gen_group(n); }
// Offset of (i, tile) in the per-radius buffer.
template <int L>
__device__ __forceinline__ unsigned gen_tile(unsigned i, unsigned tile) {
  if constexpr (gen_pair(L)) return (tile * (L / 2) + i / 2) * (16 * L) + i % 2 * 8;
  else return (tile * L + i) * (gen_group(L) * L);
}
// Sides whose planes fit the LDS of one block.
constexpr bool gen_plane(int n) { return n < 144; }

// Threads per line of the passes with g lines per block: the count T (T g a
// multiple of 64) with at most 16 values of the first stage per thread, fewest
// idle slots.
constexpr int gen_threads(int n, int g) {
  const GPlanC p = gplan(n);
  int best = 0;
  long cost = 0;
  for (int t = 64 / g; t * g <= 1024; t += 64 / g) {
    if ((n / 8 + t - 1) / t > 2) continue;
    long c = 0;  // slots of all stages
    for (int s = 0; s < p.nst; ++s) c += (long)((n / p.radix[s] + t - 1) / t) * t * p.radix[s];
    if (!best || c < cost) {
      best = t;
      cost = c;
    }
  }
  return best;
}
// The same for rows, whose threads sit in one wave (a power of two up to 64).
constexpr int gen_row_threads(int n) {
  const GPlanC p = gplan(n);
  int best = 64;
  long cost = 0;
  for (int t = 8; t <= 64; t *= 2) {
    if ((n / 8 + t - 1) / t > 2) continue;
    long c = 0;
    for (int s = 0; s < p.nst; ++s) c += (long)((n / p.radix[s] + t - 1) / t) * t * p.radix[s];
    if (!cost || c < cost) {
      best = t;
      cost = c;
    }
  }
  return best;
}
// Rows per block: 256 threads, or 512 where a row's piece of a tile is half a
// cache line (600^3 23.4 ms against 25.1; 480^3, whole lines, 8.5 against 7.6).
constexpr int gen_block_rows(int n) {
  const int r = (gen_row(n) == 8 ? 512 : 256) / gen_row_threads(n);
  return n % r == 0 ? r : 8;
}
constexpr int gen_col_threads(int n) { return gen_threads(n, gen_group(n)); }

// Butterfly of a thread's iteration; where the last iteration is partly idle
// its spare threads repeat the last butterfly and store nothing, so that the
// stages stay straight-line code.
template <int Lr, int T>
__device__ __forceinline__ unsigned gs_index(int t, int it) {
  const unsigned j = t + T * it;
  return T * (it + 1) <= Lr || j < Lr ? j : Lr - 1;
}

// Inputs of stage ST (>= 1) of the butterflies j = t + T it from ld(position),
// twiddled and transformed.  T1: the stage after the first reads positions
// that the first stage stored transposed (position 8 j + r at slot r n/8 + j).
template <int L, int ST, int T, bool T1, bool ROUND, int N, int R, class Ld>
__device__ __forceinline__ void gs_load(float2 (&a)[N][R], int t, const float2* tw, Ld&& ld) {
  constexpr int NS = gplan(L).ns[ST], Lr = L / R, tstep = L / (NS * R);
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const unsigned j = gs_index<Lr, T>(t, it);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned o = j + r * Lr;
      a[it][r] = ld(T1 && ST == 1 ? (o & 7) * (L / 8) + (o >> 3) : o);
    }
    const unsigned k = j % NS;
#pragma unroll
    for (int r = 1; r < R; ++r) {
      float2 w = tw[k * r * tstep];
      w.y = -w.y;
      a[it][r] = cmul_fixed(a[it][r], w);
    }
    Dft<R, +1, ROUND>::run(a[it]);
  }
}
template <int L, int ST, int T, bool T1, int N, int R, class St>
__device__ __forceinline__ void gs_store(const float2 (&a)[N][R], int t, St&& st) {
  constexpr int NS = gplan(L).ns[ST], Lr = L / R;
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const unsigned j = t + T * it;
    if (T * (it + 1) <= Lr || j < Lr) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        st(T1 && ST == 0 ? r * Lr + j : j / NS * (NS * R) + j % NS + r * NS, a[it][r]);
    }
  }
}
// Stages ST .. last - 1 (each: load, sync, store, sync); the last stage's
// butterflies then go to last(it, r, position, value).
template <int L, int ST, int T, bool T1, bool ROUND, bool WAVE, class Ld, class St, class Last>
__device__ __forceinline__ void gs_rest(int t, const float2* tw, Ld&& ld, St&& st, Last&& last) {
  constexpr GPlanC P = gplan(L);
  constexpr int R = P.radix[ST], N = (L / R + T - 1) / T;
  constexpr bool LAST = ST == P.nst - 1;
  float2 a[N][R];
  gs_load<L, ST, T, T1, ROUND && LAST>(a, t, tw, ld);
  if constexpr (LAST) {
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const unsigned j = t + T * it;
      if (T * (it + 1) <= L / R || j < L / R) {
#pragma unroll
        for (int r = 0; r < R; ++r) last(it, r, j, a[it][r]);
      }
    }
  } else {
    exchange_sync<WAVE>();
    gs_store<L, ST, T, T1>(a, t, st);
    exchange_sync<WAVE>();
    gs_rest<L, ST + 1, T, T1, ROUND, WAVE>(t, tw, ld, st, last);
  }
}

// Filtered inverse along i, a batch of radii: the block's G lines of the full
// spectrum stay in registers, each radius multiplies them by the weight table
// (launch_w_table; products rounded), transforms and writes the tile layout.
// Column order: mirror lines kj, n - kj behind each other -- they read the
// same weights, from one L2 when bit 2 of plan.xcd deals runs of blocks to
// one XCD.  blockIdx.y: groups of rper radii.
// Writes the per-radius buffer and reads the weights once per mirror pair: 480^3,
// 46 radii 10.8 ms (41 GB + 5 GB, 4.2 TB/s), 360^3 4.1 ms, 600^3 35 ms (half lines,
// 2.7 TB/s); evaluating the weights per radius from the spectrum in memory took
// 53.8 ms at 600^3.
template <int L>
__global__ __launch_bounds__(gen_col_threads(L)* gen_group(L)) void k_gen_filter(
    const float2* __restrict__ spec, float2* __restrict__ u, int nrad, int rper,
    const float* __restrict__ wt, const float2* __restrict__ tw, int xcd) {
  constexpr int G = gen_group(L), T = gen_col_threads(L), H = L / 2 + 1, Lr = L / 8;
  constexpr int N0 = (Lr + T - 1) / T, RL = gplan(L).radix[gplan(L).nst - 1];
  constexpr bool kT1 = false;
  __shared__ float2 buf[L * G];
  __shared__ float2 twl[L];
  const unsigned blk = ((xcd >> 2) & 1) ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)
                                        : blockIdx.x;
  const int tile = blk / L, s = blk % L;
  const int kj = s == 0 ? 0 : (s & 1) ? (s + 1) / 2 : L - s / 2;
  const int l = threadIdx.x % G, t = threadIdx.x / G;
  for (int q = threadIdx.x; q < L; q += T * G) twl[q] = tw[q];
  float2 z[N0][8];
  const float2* __restrict__ src = spec + (long)kj * L + tile * G;
#pragma unroll
  for (int it = 0; it < N0; ++it)
#pragma unroll
    for (int r = 0; r < 8; ++r)
      z[it][r] = uniform_ptr(src + (long)(r * Lr) * (L * L))[gs_index<Lr, T>(t, it) * (L * L) + l];
  constexpr long kWRadius = (long)H * (L / G) * (H * G);
  const int r0 = blockIdx.y * rper, r1 = min(r0 + rper, nrad);
  const float* __restrict__ wr =
      wt + r0 * kWRadius + ((long)(kj <= L / 2 ? kj : L - kj) * (L / G) + tile) * (H * G);
  float wv[N0][8];
  auto weights = [&]() {
#pragma unroll
    for (int it = 0; it < N0; ++it)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        // position j + r L/8, j < L/8: its frequency, or its mirror's from L/2 up
        const unsigned j = gs_index<Lr, T>(t, it);
        wv[it][r] = r < 4 ? uniform_ptr(wr + r * Lr * G)[j * G + l]
                          : uniform_ptr(wr + (L - (r + 1) * Lr) * G)[(Lr - j) * G + l];
      }
  };
  weights();
  __syncthreads();
#pragma unroll 1
  for (int rad = r0; rad < r1; ++rad) {
    const int tl = opaque_lane(t);
    float2 a[N0][8];
#pragma unroll
    for (int it = 0; it < N0; ++it) {
#pragma unroll
      for (int r = 0; r < 8; ++r)
        a[it][r] = make_float2(mul_rounded(z[it][r].x, wv[it][r]), mul_rounded(z[it][r].y, wv[it][r]));
      Dft<8, +1>::run(a[it]);
    }
    gs_store<L, 0, T, kT1>(a, tl, [&](unsigned o, float2 v) { buf[o * G + l] = v; });
    wr += kWRadius;
    if (rad + 1 < r1) weights();  // in flight during the transform
    exchange_sync<false>();
    float2* __restrict__ dst = u + (long)rad * ((long)L * L * L) + kj * gen_row(L);
    gs_rest<L, 1, T, kT1, false, false>(
        tl, twl, [&](unsigned o) { return buf[o * G + l]; },
        [&](unsigned o, float2 v) { buf[o * G + l] = v; },
        [&](int it, int r, unsigned, float2 v) {
          // t + (even constant): the offsets add
          st_stream(uniform_ptr(dst + gen_tile<L>(T * it + r * (L / RL), tile)) + gen_tile<L>(tl, 0) + l, v);
        });
    exchange_sync<false>();  // the buffer is read before the next radius lands in it
  }
}

// Inverse along j in place over the tile layout: a block per contiguous piece
// of n rows ((i, tile), or two planes of a tile of 8); blockIdx.y: radius.
// Memory-bound: 600^3, 48 radii 32.2 ms (5.2 TB/s read and written; 40.8 ms from
// strided lines), 480^3 15.1 ms.
template <int L>
__global__ __launch_bounds__(gen_threads(L, gen_row(L)) * gen_row(L)) void k_gen_inv_j(
    float2* __restrict__ u, const float2* __restrict__ tw, int xcd) {
  constexpr int C = gen_row(L), T = gen_threads(L, C), Lr = L / 8;
  constexpr int N0 = (Lr + T - 1) / T, RL = gplan(L).radix[gplan(L).nst - 1];
  __shared__ float2 buf[L * C];
  // the remainder of a grid that is no multiple of 8 (two planes a piece) keeps its place
  const unsigned blk = ((xcd >> 1) & 1) && blockIdx.x < (gridDim.x & ~7u)
                           ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)
                           : blockIdx.x;
  const int l = threadIdx.x % C, t = threadIdx.x / C;
  float2* __restrict__ line = u + (long)blockIdx.y * ((long)L * L * L) + (long)blk * (L * C);
  float2 a[N0][8];
#pragma unroll
  for (int it = 0; it < N0; ++it)
#pragma unroll
    for (int r = 0; r < 8; ++r)
      a[it][r] = ld_stream(uniform_ptr(line + r * Lr * C) + gs_index<Lr, T>(t, it) * C + l);
#pragma unroll
  for (int it = 0; it < N0; ++it) Dft<8, +1>::run(a[it]);
  gs_store<L, 0, T, false>(a, t, [&](unsigned o, float2 v) { buf[o * C + l] = v; });
  exchange_sync<false>();
  gs_rest<L, 1, T, false, false, false>(
      t, tw, [&](unsigned o) { return buf[o * C + l]; }, [&](unsigned o, float2 v) { buf[o * C + l] = v; },
      [&](int, int r, unsigned j, float2 v) { st_stream(line + (j + r * (L / RL)) * C + l, v); });
}

// Inverse along p and the centre test of a batch of radii, smallest radius
// first (the last centre found has the largest bound), the next radius loaded
// during the transform.  A row's T threads sit in one wave: no block barriers
// in the loop.  Blocks of 512 threads are held to 128 registers (two per CU; the
// smaller ones take 142-153, and spill at 128: 480^3 11.3 ms against 7.7).
// dbg (one radius): the unscaled pairs in natural order, the values the test
// saw.
// Bound by VALU issue, 81% busy, and the lines it reads: 600^3, 48 radii 23-23.5 ms
// for 83 GB, 3.5 TB/s (one radius per launch, no prefetch: 28.7), where half lines
// make it fetch 1.6 times that, 5.1 TB/s; 480^3, whole lines, 7.7 ms (5.3 TB/s).
template <int L>
__global__ __launch_bounds__(gen_row_threads(L)* gen_block_rows(L),
                             gen_row_threads(L) * gen_block_rows(L) > 256 ? 4 : 1) void k_gen_crit(
    const float2* __restrict__ u, int nrad, const int* __restrict__ d2max,
    const float* __restrict__ bal, int* __restrict__ wmap, float2* __restrict__ dbg,
    const float2* __restrict__ tw) {
  constexpr int G = gen_group(L), T = gen_row_threads(L), RPB = gen_block_rows(L), Lr = L / 8;
  constexpr int N0 = (Lr + T - 1) / T, RL = gplan(L).radix[gplan(L).nst - 1];
  constexpr int LrL = L / RL, NL = (LrL + T - 1) / T;
  // rows an odd multiple of 8 apart: neighbouring rows in other banks
  constexpr int SR = (L + 8) % 16 == 0 ? L : L + 8;
  __shared__ float2 buf[RPB * SR];
  __shared__ float2 twl[L];
  const int lw = threadIdx.x / T, t = threadIdx.x % T;
  for (int q = threadIdx.x; q < L; q += T * RPB) twl[q] = tw[q];
  // rows of one plane, or of the two that share the cache lines
  constexpr int PI = gen_pair(L) ? 2 : 1, RJ = RPB / PI;
  const unsigned i = blockIdx.x / (L / RJ) * PI + lw % PI, j = blockIdx.x % (L / RJ) * RJ + lw / PI;
  const long row = (long)i * L + j;
  float2* line = buf + lw * SR;
  const float sc = bal[0];
  int wbest[NL][RL];
#pragma unroll
  for (int it = 0; it < NL; ++it)
#pragma unroll
    for (int r = 0; r < RL; ++r) wbest[it][r] = -1;
  float2 nx[N0][8];
  auto fetch = [&](int rad) {
    const float2* __restrict__ src = u + (long)rad * ((long)L * L * L) + gen_tile<L>(i, 0) + gen_row(L) * j;
#pragma unroll
    for (int it = 0; it < N0; ++it)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const unsigned p = gs_index<Lr, T>(t, it) + r * Lr;
        nx[it][r] = ld_stream(src + (gen_tile<L>(0, p / G) + p % G));
      }
  };
  fetch(nrad - 1);
  __syncthreads();
#pragma unroll 1
  for (int rad = nrad - 1; rad >= 0; --rad) {
    const int tl = opaque_lane(t);
    float2 a[N0][8];
#pragma unroll
    for (int it = 0; it < N0; ++it) {
#pragma unroll
      for (int r = 0; r < 8; ++r) a[it][r] = nx[it][r];
      Dft<8, +1>::run(a[it]);
    }
    if (rad > 0) fetch(rad - 1);
    gs_store<L, 0, T, true>(a, tl, [&](unsigned o, float2 v) { line[o] = v; });
    exchange_sync<true>();
    const int w = d2max[rad];
    gs_rest<L, 1, T, true, true, true>(
        tl, twl, [&](unsigned o) { return line[o]; }, [&](unsigned o, float2 v) { line[o] = v; },
        [&](int it, int r, unsigned jb, float2 v) {
          wbest[it][r] = is_centre(v.x * sc, v.y) ? w : wbest[it][r];
          if (dbg) dbg[row * L + jb + r * LrL] = make_float2(v.x, v.y / sc);
        });
    exchange_sync<true>();
  }
  if (dbg) return;
#pragma unroll
  for (int it = 0; it < NL; ++it)
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const unsigned jb = t + T * it;
      if ((T * (it + 1) <= LrL || jb < LrL) && wbest[it][r] >= 0)
        wmap[row * L + jb + r * LrL] = wbest[it][r];
    }
}

// Sides below 144: j and p inverses and the centre test of one (i, radius)
// plane in one block, 8 threads per line, the plane in LDS between the stages
// (element (j, p) at j SR + p).  blockIdx.y: groups of rper radii (wmap by
// atomic maximum when there are several).  Reads the buffer once instead of
// three accesses: 120^3, 33 radii 0.28 ms, one launch, bound by the barriers of its
// exchanges, one block of 15 waves per CU (VALU 34%, LDS 10% busy, 1.8 TB/s); with the separate passes of one radius each 0.9 ms and 66 launches.
template <int L>
struct GenPlaneCfg {
  static constexpr int T = 8;
  static constexpr int kThreads = (L * T + 63) / 64 * 64;
  static constexpr int SR = (L + 8) % 16 == 0 ? L : L + 8;
  static constexpr int kLds = (L * SR + L) * (int)sizeof(float2);
};
template <int L>
__global__ __launch_bounds__(GenPlaneCfg<L>::kThreads) void k_gen_plane(
    const float2* __restrict__ u, int nrad, int rper, const int* __restrict__ d2max,
    const float* __restrict__ bal, int* __restrict__ wmap, float2* __restrict__ dbg,
    const float2* __restrict__ tw) {
  using C = GenPlaneCfg<L>;
  constexpr int G = gen_group(L), T = C::T, Lr = L / 8, SR = C::SR;
  constexpr int N0 = (Lr + T - 1) / T, RL = gplan(L).radix[gplan(L).nst - 1];
  constexpr int LrL = L / RL, NL = (LrL + T - 1) / T;
  extern __shared__ float2 gpl[];
  float2* twl = gpl + L * SR;
  // planes 2m, 2m + 1 (which share cache lines where G = 8) eight blocks
  // apart: on one XCD
  const int b = blockIdx.x, i = G == 8 && b < L / 16 * 16 ? b / 16 * 16 + (b & 7) * 2 + (b >> 3 & 1) : b;
  const int tid = threadIdx.x;
  for (int q = tid; q < L; q += C::kThreads) twl[q] = tw[q];
  const bool ok = tid < L * T;  // the last wave may be partly idle
  // columns: c = p, tc its thread; rows: j, t
  const int c = ok ? tid % L : 0, tc = ok ? tid / L : 0;
  const int j = ok ? tid / T : 0, t = ok ? tid % T : 0;
  const float sc = bal[0];
  const int r0 = blockIdx.y * rper, r1 = min(r0 + rper, nrad);
  int wbest[NL][RL];
#pragma unroll
  for (int it = 0; it < NL; ++it)
#pragma unroll
    for (int r = 0; r < RL; ++r) wbest[it][r] = -1;
  const unsigned off = gen_tile<L>(i, c / G) + c % G;
  __syncthreads();
#pragma unroll 1
  for (int rad = r1 - 1; rad >= r0; --rad) {
    const int tcl = opaque_lane(tc), tl = opaque_lane(t);
    float2* col = gpl + c;
    float2* line = gpl + j * SR;
    {
      const float2* __restrict__ src = u + (long)rad * ((long)L * L * L);
      float2 a[N0][8];
#pragma unroll
      for (int it = 0; it < N0; ++it)
#pragma unroll
        for (int r = 0; r < 8; ++r)
          a[it][r] = ld_stream(uniform_ptr(src + r * Lr * gen_row(L)) + off + gs_index<Lr, T>(tcl, it) * gen_row(L));
#pragma unroll
      for (int it = 0; it < N0; ++it) Dft<8, +1>::run(a[it]);
      if (ok) gs_store<L, 0, T, false>(a, tcl, [&](unsigned o, float2 v) { col[o * SR] = v; });
    }
    exchange_sync<false>();
    float2 y[NL][RL];
    gs_rest<L, 1, T, false, false, false>(
        tcl, twl, [&](unsigned o) { return col[o * SR]; },
        [&](unsigned o, float2 v) {
          if (ok) col[o * SR] = v;
        },
        [&](int it, int r, unsigned, float2 v) { y[it][r] = v; });
    exchange_sync<false>();
    if (ok) {
#pragma unroll
      for (int it = 0; it < NL; ++it)
#pragma unroll
        for (int r = 0; r < RL; ++r)
          if (T * (it + 1) <= LrL || tcl + T * it < LrL) col[(tcl + T * it + r * LrL) * SR] = y[it][r];
    }
    exchange_sync<false>();
    {
      float2 a[N0][8];
#pragma unroll
      for (int it = 0; it < N0; ++it) {
#pragma unroll
        for (int r = 0; r < 8; ++r) a[it][r] = line[gs_index<Lr, T>(tl, it) + r * Lr];
        Dft<8, +1>::run(a[it]);
      }
      exchange_sync<true>();
      if (ok) gs_store<L, 0, T, true>(a, tl, [&](unsigned o, float2 v) { line[o] = v; });
    }
    exchange_sync<true>();
    const int w = d2max[rad];
    gs_rest<L, 1, T, true, true, true>(
        tl, twl, [&](unsigned o) { return line[o]; },
        [&](unsigned o, float2 v) {
          if (ok) line[o] = v;
        },
        [&](int it, int r, unsigned jb, float2 v) {
          wbest[it][r] = is_centre(v.x * sc, v.y) ? w : wbest[it][r];
          if (dbg && ok) dbg[((long)i * L + j) * L + jb + r * LrL] = make_float2(v.x, v.y / sc);
        });
    exchange_sync<false>();  // the rows are read before the next columns land in them
  }
  if (!ok || dbg) return;
#pragma unroll
  for (int it = 0; it < NL; ++it)
#pragma unroll
    for (int r = 0; r < RL; ++r) {
      const unsigned jb = t + T * it;
      if ((T * (it + 1) <= LrL || jb < LrL) && wbest[it][r] >= 0) {
        int* w = wmap + ((long)i * L + j) * L + jb + r * LrL;
        if (gridDim.y > 1) atomicMax(w, wbest[it][r]);
        else *w = wbest[it][r];
      }
    }
}

bool gen_plan_make(int n, GenPlan* p) {
  if (n < 16 || n > kGenMaxL || n % kGenLines != 0) return false;
  int m = n, ns = 1, st = 0;
  while (m > 1) {
    int r;
    if (m % 8 == 0) r = 8;
    else if (m % 4 == 0) r = 4;
    else if (m % 2 == 0) r = 2;
    else if (m % 3 == 0) r = 3;
    else if (m % 5 == 0) r = 5;
    else return false;
    if (st >= 16) return false;
    p->radix[st] = r;
    p->ns[st] = ns;
    p->rns[st] = 1.0f / (float)ns;
    ns *= r;
    m /= r;
    ++st;
  }
  p->L = n;
  p->nst = st;
  p->xcd = 1 << 2;
  if (p->radix[0] != 8 || st < 2) return false;  // the kernels' first stage is radix 8
  // line stride = 8 (mod 32) float2: the 8 lines of a column-pass wave
  // start in different bank groups
  p->lp = n + ((8 - n % 32) + 32) % 32;
  return true;
}

size_t gen_pass_lds(const GenPlan& p) { return sizeof(float2) * kGenLines * (size_t)p.lp; }

#define GEN_KERNELS_L(X, LC)                                                               \
  X(-1, 0, true, LC) X(-1, 0, false, LC) X(+1, 0, true, LC) X(+1, 0, false, LC)             \
  X(+1, 1, false, LC)
#define GEN_KERNELS(X) GEN_KERNELS_L(X, 0) GEN_KERNELS_L(X, 600)

bool gen_prepare(const GenPlan& p) {
  // LDS of the transform blocks above 64 KiB is requested per kernel
  const size_t lds = gen_pass_lds(p);
  if (lds <= 65536) return true;
  const int v = (int)lds;
  const hipFuncAttribute at = hipFuncAttributeMaxDynamicSharedMemorySize;
  bool ok = true;
#define GA(SG, MD, RW, LC) \
  ok = ok && hipFuncSetAttribute((const void*)k_gen_pass<SG, MD, RW, LC>, at, v) == hipSuccess;
  GEN_KERNELS(GA)
#undef GA
  return ok;
}

bool gen_finder_prepare(int n) {
  bool ok = false;
#define X(L)                                                                               \
  if (n == L) {                                                                            \
    ok = true;                                                                             \
    if constexpr (gen_plane(L))                                                            \
      ok = hipFuncSetAttribute((const void*)k_gen_plane<L>,                                \
                               hipFuncAttributeMaxDynamicSharedMemorySize,                 \
                               GenPlaneCfg<L>::kLds) == hipSuccess;                        \
  }
  SF21_GEN_SIDES(X)
#undef X
  return ok;
}

bool gen_plane_side(int n) { return gen_plane(n); }

// Groups of radii per launch: about 16 waves per CU.
static int gen_groups(long waves, int nrad) {
  const long want = (4096 + waves - 1) / waves;
  return (int)(want > nrad ? nrad : want);
}

void launch_gen_filter(const GenPlan& plan, const float2* spec, float2* u, int nrad, const float* wt,
                       const float2* tw, hipStream_t s) {
  const int side = plan.L;
#define X(L)                                                                               \
  if (side == L) {                                                                          \
    constexpr int G = gen_group(L), NT = gen_col_threads(L) * G, NB = L * (L / G);         \
    const int g = gen_groups((long)NB * ((NT + 63) / 64), nrad), per = (nrad + g - 1) / g; \
    hipLaunchKernelGGL(k_gen_filter<L>, dim3(NB, (nrad + per - 1) / per), dim3(NT), 0, s, spec, u, \
                       nrad, per, wt, tw, plan.xcd);                                       \
  }
  SF21_GEN_SIDES(X)
#undef X
}

void launch_gen_inv_j(const GenPlan& plan, float2* u, int nrad, const float2* tw, hipStream_t s) {
  const int side = plan.L;
#define X(L)                                                                               \
  if (side == L) {                                                                          \
    if constexpr (!gen_plane(L))                                                           \
      {                                                                \
      constexpr int C = gen_row(L);                                                        \
      hipLaunchKernelGGL(k_gen_inv_j<L>, dim3(L * L / C, nrad), dim3(gen_threads(L, C) * C), 0, s, \
                         u, tw, plan.xcd);                                                 \
    }                                                                                      \
  }
  SF21_GEN_SIDES(X)
#undef X
}

void launch_gen_crit(const GenPlan& plan, const float2* u, int nrad, const int* d2max,
                     const float* bal, int* wmap, float2* dbg, const float2* tw, hipStream_t s) {
  const int side = plan.L;
#define X(L)                                                                               \
  if (side == L) {                                                                          \
    if constexpr (gen_plane(L)) {                                                          \
      using C = GenPlaneCfg<L>;                                                            \
      const int g = gen_groups((long)L * (C::kThreads / 64), nrad), per = (nrad + g - 1) / g; \
      hipLaunchKernelGGL(k_gen_plane<L>, dim3(L, (nrad + per - 1) / per), dim3(C::kThreads), \
                         C::kLds, s, u, nrad, per, d2max, bal, wmap, dbg, tw);             \
    } else {                                                                               \
      hipLaunchKernelGGL(k_gen_crit<L>, dim3(L * (L / gen_block_rows(L))),                 \
                         dim3(gen_row_threads(L) * gen_block_rows(L)), 0, s, u,            \
                         nrad, d2max, bal, wmap, dbg, tw);                                 \
    }                                                                                      \
  }
  SF21_GEN_SIDES(X)
#undef X
}

void launch_gen_pass(const GenPlan& plan, int axis, int sign, int mode, const float2* src,
                     float2* dst, const float2* tw, float2 kappa, hipStream_t s) {
  const unsigned L = (unsigned)plan.L;
  const dim3 g(L * L / kGenLines), b(256);
  const size_t lds = gen_pass_lds(plan);
  const bool rows = axis == 0;
  const int sg = sign < 0 ? -1 : +1, md = sign < 0 ? 0 : mode;
  // the specialised side's plan is the one gen_plan_make builds for it
  const int lc = (plan.L == 600 && plan.nst == 4 && plan.lp == 616) ? 600 : 0;
#define GL(SG, MD, RW, LC)                                                                     \
  if (sg == SG && md == MD && rows == RW && lc == LC)                                          \
    hipLaunchKernelGGL((k_gen_pass<SG, MD, RW, LC>), g, b, lds, s, src, dst, plan, axis, tw, kappa);
  GEN_KERNELS(GL)
#undef GL
}

void launch_gen_pack(long n3, const float* a, const float* b, const float* c, CellConsts k,
                     const float* bal, float2* spec, hipStream_t s) {
  long blocks = (n3 + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_gen_pack, dim3((unsigned)blocks), dim3(256), 0, s, n3, a, b, c, k, bal, spec);
}

}  // namespace sf21
