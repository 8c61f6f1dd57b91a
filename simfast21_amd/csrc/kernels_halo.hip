// Halo-catalog emissivity (use_SFR = F, get_HIIbubbles.c:229-259): cloud-in-
// cell deposit of each halo's ionising rate Rion(M, z) (user_functions.c:40-47)
// on the N_halo^3 grid (auxiliary.c:761-808), the block average down to
// N_smoothed^3 (smooth_box, auxiliary.c:643-682) times (dx_s/dx_h)^3 fesc; and
// the non-linear density's displacement deposit on the N_halo^3 grid.
#include <hip/hip_runtime.h>

#include <climits>

#include "kernels.h"

namespace sf21 {

// Cloud in cell along one axis (auxiliary.c:764-784): position x in grid-cell
// units to the lower cell and the far cell's weight -- truncation toward zero
// and, for a negative remainder, one cell down with |remainder| as the far
// weight.
__device__ __forceinline__ void cic_axis(float x, int& cell, float& far) {
  cell = (int)x;
  far = x - (float)cell;
  if (far < 0.0f) {
    cell -= 1;
    far = -far;
  }
}

__device__ __forceinline__ int wrap_cell(int q, int ng) {
  q %= ng;
  return q < 0 ? q + ng : q;
}

// Deposit of v at (x1, y1, z1) (auxiliary.c:785-808); the 8 cells wrap
// periodically.  FP32 atomics.
__device__ __forceinline__ void cic_deposit(float x1, float y1, float z1, float v, int ng,
                                            float* __restrict__ grid) {
  int x, y, z;
  float fx, fy, fz;
  cic_axis(x1, x, fx);
  cic_axis(y1, y, fy);
  cic_axis(z1, z, fz);
  for (int a = 0; a < 2; ++a) {
    const int xi = wrap_cell(x + a, ng);
    const float wx = a ? fx : 1.0f - fx;
    for (int b = 0; b < 2; ++b) {
      const int yi = wrap_cell(y + b, ng);
      const float wy = b ? fy : 1.0f - fy;
      for (int c = 0; c < 2; ++c) {
        const int zi = wrap_cell(z + c, ng);
        const float wz = c ? fz : 1.0f - fz;
        atomicAdd(&grid[((long)xi * ng + yi) * ng + zi], wx * wy * wz * v);
      }
    }
  }
}

// Weights of a halo's two cells along one axis on the block-averaged grid:
// block of either cell; both in one block: the sum there (w1 = 0).
__device__ __forceinline__ void cic_block_axis(float x, int ng, int sm, int& b0, int& b1, float& w0,
                                               float& w1) {
  int c;
  float far;
  cic_axis(x, c, far);
  b0 = wrap_cell(c, ng) / sm;
  b1 = wrap_cell(c + 1, ng) / sm;
  w0 = 1.0f - far;
  w1 = far;
  if (b0 == b1) {
    w0 += w1;
    w1 = 0.0f;
  }
}

// One thread per halo: the deposited value is Rion(M, z)
// (user_functions.c:40-47, k_rion = c1 (1+z)^c4 / V_norm, or that over Qion(z)
// for the SFR of user_functions.c:71-74) times f = scale / sm^3.  The block
// average of the deposit is linear in it, so each halo goes straight to the
// at most 8 blocks of the n^3 box that hold its 8 cells; cells past the last
// whole block are dropped, as smooth_box drops them.  T = double: more halos
// meet in a block than in a fine cell, and the averaging was compensated.
// 512^3 to 256^3, 10^6 halos, against zeroing, filling and averaging the fine
// grid (1 GB of traffic): 0.67 -> 0.21 ms (FP32 sums: 0.19).  Bound: the atomics' scattered lines.
template <class T>
__global__ void k_cic_rion(long nhalos, const float* __restrict__ halos, int ng, int ns, int sm,
                           float k_rion, float c2, float c3, float f, T* __restrict__ out) {
  for (long h = (long)blockIdx.x * blockDim.x + threadIdx.x; h < nhalos;
       h += (long)gridDim.x * blockDim.x) {
    const float m = halos[4 * h], x1 = halos[4 * h + 1], y1 = halos[4 * h + 2],
                z1 = halos[4 * h + 3];
    // Rion = c1 M (1+z)^c4 (M/c2)^c3 exp(-(c2/M)^3) / V_norm
    const float q = c2 / m;
    const float v = k_rion * m * powf(m / c2, c3) * expf(-(q * q * q)) * f;
    int bx[2], by[2], bz[2];
    float wx[2], wy[2], wz[2];
    cic_block_axis(x1, ng, sm, bx[0], bx[1], wx[0], wx[1]);
    cic_block_axis(y1, ng, sm, by[0], by[1], wy[0], wy[1]);
    cic_block_axis(z1, ng, sm, bz[0], bz[1], wz[0], wz[1]);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const bool merged = (a && bx[0] == bx[1]) || (b && by[0] == by[1]) || (c && bz[0] == bz[1]);
          if (merged || bx[a] >= ns || by[b] >= ns || bz[c] >= ns) continue;
          atomicAdd(&out[((long)bx[a] * ns + by[b]) * ns + bz[c]], (T)(wx[a] * wy[b] * wz[c] * v));
        }
  }
}

// Non-linear density (get_nldensity.c:140-166): every cell (i, j, p) of the
// N_halo^3 grid moves its mass 1 + delta0 D_in to (i, j, p) + v s (D(z) -
// D_in) and deposits it by CIC on a grid that starts at -1.  v: the z = 0
// velocity boxes (Mpc), s = N_halo h / L_h turns them into cells.
__global__ void k_fill_value(float* __restrict__ p, float value, long count) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (long)gridDim.x * blockDim.x)
    p[i] = value;
}

// A block takes a tile of source cells.  Neighbouring cells move together, so
// the tile lands in a box little larger than itself: where that box fits the
// block's LDS the deposits are added there and every touched cell then takes
// one global atomic, in rows of consecutive addresses -- about 3 per source
// cell instead of 8.  The LDS sums are FP64: an FP32 LDS atomic takes 193
// cycles a wave here, an FP64 one 9.  A tile whose cells scatter farther
// deposits directly (a NaN position truncates to cell 0, with NaN weights, on
// either way).  Blocks stay and take one tile after another,
// the next one's velocities loaded while this one is added up.  512^3,
// displacements of 1.1 cells rms: 24.7 ms direct, 6.1 with FP32 sums in tiles of
// 16 x 16 x 32, 2.1 this way (2.5 with a block per tile).  Tried and slower: tiles by
// parity in 8 launches with plain additions to the grid, 2.8 ms.  Bound: the
// global atomics, 2e11 a second, and the phases of one block per CU.
constexpr int kDepTX = 16, kDepTY = 16, kDepTZ = 16, kDepThreads = 1024;
constexpr int kDepCells = kDepTX * kDepTY * kDepTZ / kDepThreads;  // of a thread, in registers
constexpr int kDepCap = 19968;  // doubles: one block per CU
constexpr long kDepBlocks = 256;  // one per CU

__global__ __launch_bounds__(kDepThreads) void k_displace_deposit(
    int ng, int tiles, const float* __restrict__ vx, const float* __restrict__ vy,
    const float* __restrict__ vz, const float* __restrict__ delta0, float vscale, float growth_in,
    float growth, float* __restrict__ grid) {
  extern __shared__ double box[];
  __shared__ int lo[3], hi[3];
  const int nty = (ng + kDepTY - 1) / kDepTY, ntz = (ng + kDepTZ - 1) / kDepTZ;
  const int tid = threadIdx.x;
  // the thread's cells of a tile, p fastest over the threads
  auto cell = [&](int tile, int u, int& i, int& j, int& p) {
    const int e = tid + u * kDepThreads;
    i = tile / (nty * ntz) * kDepTX + e / (kDepTY * kDepTZ);
    j = tile / ntz % nty * kDepTY + e / kDepTZ % kDepTY;
    p = tile % ntz * kDepTZ + e % kDepTZ;
    return i < ng && j < ng && p < ng;
  };
  float v[kDepCells][4] = {};
  auto load = [&](int tile) {
#pragma unroll
    for (int u = 0; u < kDepCells; ++u) {
      int i, j, p;
      if (!cell(tile, u, i, j, p)) continue;
      const long ind = ((long)i * ng + j) * ng + p;
      v[u][0] = vx[ind];
      v[u][1] = vy[ind];
      v[u][2] = vz[ind];
      v[u][3] = delta0[ind];
    }
  };
  if ((int)blockIdx.x < tiles) load(blockIdx.x);
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    if (tid < 3) {
      lo[tid] = INT_MAX;
      hi[tid] = INT_MIN;
    }
    __syncthreads();
    float r[kDepCells][3], m[kDepCells];  // displaced positions, masses
    bool in[kDepCells];
    int mn[3] = {INT_MAX, INT_MAX, INT_MAX}, mx[3] = {INT_MIN, INT_MIN, INT_MIN};
#pragma unroll
    for (int u = 0; u < kDepCells; ++u) {
      int c[3];
      in[u] = cell(tile, u, c[0], c[1], c[2]);
      m[u] = fmaf(v[u][3], growth_in, 1.0f);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        r[u][a] = fmaf(v[u][a] * vscale, growth, (float)c[a]);
        int q;
        float far;
        cic_axis(r[u][a], q, far);
        if (in[u]) {
          mn[a] = min(mn[a], q);
          mx[a] = max(mx[a], q);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        mn[a] = min(mn[a], __shfl_xor(mn[a], o, 64));
        mx[a] = max(mx[a], __shfl_xor(mx[a], o, 64));
      }
      if ((tid & 63) == 0) {
        atomicMin(&lo[a], mn[a]);
        atomicMax(&hi[a], mx[a]);
      }
    }
    if (tile + (int)gridDim.x < tiles) load(tile + gridDim.x);  // before this tile's atomics
    __syncthreads();
    const int x0 = lo[0], y0 = lo[1], z0 = lo[2];
    // cells lo .. hi + 1 along each axis; 64-bit: positions may be anything
    const long ex = (long)hi[0] - x0 + 2, ey = (long)hi[1] - y0 + 2, ez = (long)hi[2] - z0 + 2;
    // a full edge first: the product of the three stays below 2^62
    const bool fits = ex <= kDepCap && ey <= kDepCap && ez <= kDepCap && ex * ey * ez <= kDepCap;
    if (!fits) {
#pragma unroll
      for (int u = 0; u < kDepCells; ++u)
        if (in[u]) cic_deposit(r[u][0], r[u][1], r[u][2], m[u], ng, grid);
      __syncthreads();  // lo and hi are read before the next tile resets them
      continue;
    }
    const int dy = (int)ey, dz = (int)ez, vol = (int)(ex * ey * ez);
    for (int e = tid; e < vol; e += kDepThreads) box[e] = 0.0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kDepCells; ++u) {
      if (!in[u]) continue;
      int x, y, z;
      float fx, fy, fz;
      cic_axis(r[u][0], x, fx);
      cic_axis(r[u][1], y, fy);
      cic_axis(r[u][2], z, fz);
      double* b = box + ((x - x0) * dy + (y - y0)) * dz + (z - z0);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float w = (a ? fx : 1.0f - fx) * (c ? fy : 1.0f - fy);
          double* q = b + (a * dy + c) * dz;
          atomicAdd(q, (double)(w * (1.0f - fz) * m[u]));
          atomicAdd(q + 1, (double)(w * fz * m[u]));
        }
    }
    __syncthreads();
    // offsets past a wrapped start: one subtraction unless the box is wider
    // than the grid
    const int xw = wrap_cell(x0, ng), yw = wrap_cell(y0, ng), zw = wrap_cell(z0, ng);
    auto past = [ng](int w, int k) {
      w += k;
      if (w >= ng) w -= ng;
      return w < ng ? w : w % ng;
    };
    // floor(e / n) for e < 2^15: (e + 1/2) / n lies 1/(2 n) or more inside an
    // integer interval, the product's error is below 2^-7 / n
    const float rdz = 1.0f / (float)dz, rdy = 1.0f / (float)dy;
    for (int e = tid; e < vol; e += kDepThreads) {
      const float s = (float)box[e];
      const int q = (int)(((float)e + 0.5f) * rdz), a = (int)(((float)q + 0.5f) * rdy);
      // 0: nothing landed there, or nothing to add
      if (s != 0.0f)
        atomicAdd(&grid[((long)past(xw, a) * ng + past(yw, q - a * dy)) * ng + past(zw, e - q * dz)], s);
    }
    __syncthreads();  // the box is read before the next tile clears it
  }
}

// Block average of sm^3 cells (compensated FP32 sum in the cells' order).  A
// row of 64 lanes per row of blocks; PAIR: blocks of 2 on an even, aligned
// grid, whose four pairs are loaded together.  Bound: the read of the grid.
// 512^3 to 256^3: 0.157 ms with a 64-bit division per block and single loads,
// 0.113 ms this way.
template <bool PAIR>
__global__ __launch_bounds__(256) void k_smooth_scale(int ng, int ns, int sm,
                                                      const float* __restrict__ grid,
                                                      float* __restrict__ out) {
  const float inv = 1.0f / ((float)sm * sm * sm);
  for (int row = blockIdx.x * 4 + threadIdx.y; row < ns * ns; row += gridDim.x * 4) {
    const int a = row / ns, b = row % ns;
    const float* __restrict__ first = grid + ((long)a * sm * ng + (long)b * sm) * ng;
    for (int c = threadIdx.x; c < ns; c += 64) {
      float s = 0.0f, comp = 0.0f;
      auto add = [&](float x) {
        const float yv = x - comp;
        const float t = s + yv;
        comp = (t - s) - yv;
        s = t;
      };
      if constexpr (PAIR) {
        float2 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          x[q] = reinterpret_cast<const float2*>(first + ((long)(q >> 1) * ng + (q & 1)) * ng)[c];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          add(x[q].x);
          add(x[q].y);
        }
      } else {
        for (int u = 0; u < sm; ++u)
          for (int v = 0; v < sm; ++v) {
            const float* __restrict__ line = first + ((long)u * ng + v) * ng + (long)c * sm;
            for (int w = 0; w < sm; ++w) add(line[w]);
          }
      }
      out[(long)row * ns + c] = s * inv;
    }
  }
}


template <class T>
__global__ void k_zero(T* __restrict__ p, long count) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (long)gridDim.x * blockDim.x)
    p[i] = T(0);
}

__global__ void k_to_f32(long count, const double* __restrict__ in, float* __restrict__ out) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (long)gridDim.x * blockDim.x)
    out[i] = (float)in[i];
}

static unsigned blocks_for(long count) {
  long b = (count + 255) / 256;
  if (b > 8192) b = 8192;
  if (b < 1) b = 1;
  return (unsigned)b;
}

// FP64 sum of a float box: block partials, then one block.
__global__ __launch_bounds__(256) void k_sum_f32(long count, const float* __restrict__ x,
                                                 double* __restrict__ part) {
  __shared__ double r[256];
  double a = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (long)gridDim.x * blockDim.x)
    a += (double)x[i];
  r[threadIdx.x] = a;
  __syncthreads();
  for (int st = blockDim.x / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) r[threadIdx.x] += r[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = r[0];
}

__global__ __launch_bounds__(256) void k_sum_final(const double* __restrict__ part, int np,
                                                   double* __restrict__ out) {
  __shared__ double r[256];
  double a = 0.0;
  for (int i = threadIdx.x; i < np; i += blockDim.x) a += part[i];
  r[threadIdx.x] = a;
  __syncthreads();
  for (int st = blockDim.x / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) r[threadIdx.x] += r[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = r[0];
}

int sum_partials_count(long count) { return (int)blocks_for(count); }

void launch_sum_f32(long count, const float* x, double* part, double* out, hipStream_t s) {
  const unsigned nb = blocks_for(count);
  hipLaunchKernelGGL(k_sum_f32, dim3(nb), dim3(256), 0, s, count, x, part);
  hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(256), 0, s, part, (int)nb, out);
}

bool deposit_prepare() {
  // LDS above 64 KiB is requested per kernel
  return hipFuncSetAttribute((const void*)k_displace_deposit,
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)sizeof(double) * kDepCap) == hipSuccess;
}

void launch_nldensity_start(int ng, float* grid, hipStream_t s) {
  const long g3 = (long)ng * ng * ng;
  hipLaunchKernelGGL(k_fill_value, dim3(blocks_for(g3)), dim3(256), 0, s, grid, -1.0f, g3);
}

void launch_nldensity(int ng, int ns, int sm, const float* vx, const float* vy, const float* vz,
                      const float* delta0, float vscale, float growth_in, float growth,
                      float* grid, float* out, hipStream_t s) {
  const long tiles = (long)((ng + kDepTX - 1) / kDepTX) * ((ng + kDepTY - 1) / kDepTY) *
                     ((ng + kDepTZ - 1) / kDepTZ);
  hipLaunchKernelGGL(k_displace_deposit, dim3((unsigned)(tiles < kDepBlocks ? tiles : kDepBlocks)),
                     dim3(kDepThreads), sizeof(double) * kDepCap, s, ng, (int)tiles, vx, vy, vz,
                     delta0, vscale, growth_in, growth, grid);
  if (!out) return;
  const dim3 g(blocks_for((long)ns * ns * 64)), b(64, 4);
  if (sm == 2 && ng % 2 == 0 && reinterpret_cast<uintptr_t>(grid) % sizeof(float2) == 0)
    hipLaunchKernelGGL(k_smooth_scale<true>, g, b, 0, s, ng, ns, sm, grid, out);
  else
    hipLaunchKernelGGL(k_smooth_scale<false>, g, b, 0, s, ng, ns, sm, grid, out);
}

void launch_halo_emissivity(long nhalos, const float* halos, int ng, int ns, int sm, float k_rion,
                            float c2, float c3, float scale, double* acc, float* out,
                            hipStream_t s) {
  const long n3 = (long)ns * ns * ns;
  const float f = (float)((double)scale / ((double)sm * sm * sm));
  const dim3 g(blocks_for(n3)), gh(blocks_for(nhalos)), b(256);
  if (sm == 1) {  // a block is one cell: the deposit's own FP32 sums
    hipLaunchKernelGGL(k_zero<float>, g, b, 0, s, out, n3);
    if (nhalos > 0)
      hipLaunchKernelGGL(k_cic_rion<float>, gh, b, 0, s, nhalos, halos, ng, ns, sm, k_rion, c2, c3,
                         f, out);
    return;
  }
  hipLaunchKernelGGL(k_zero<double>, g, b, 0, s, acc, n3);
  if (nhalos > 0)
    hipLaunchKernelGGL(k_cic_rion<double>, gh, b, 0, s, nhalos, halos, ng, ns, sm, k_rion, c2, c3, f,
                       acc);
  hipLaunchKernelGGL(k_to_f32, g, b, 0, s, n3, acc, out);
}

}  // namespace sf21
