// Bandwidth-bound and small-matrix kernels of the HF/GW path (gfx950).
#include "kernels.hpp"

#include <algorithm>
#include <cmath>

namespace ggpu {
namespace {

constexpr int TILE = 32;

__device__ inline z64 cmul(z64 a, z64 b) { return z64{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ inline z64 csub(z64 a, z64 b) { return z64{a.x - b.x, a.y - b.y}; }

template <class T> __device__ inline c32 narrow(T v) { return c32{(float)v.x, (float)v.y}; }
template <class T> __device__ inline T cjt(T a) { return T{a.x, -a.y}; }
template <class T> __device__ inline T scl(T a, double f) {
  using R = decltype(a.x);
  return T{(R)(f * a.x), (R)(f * a.y)};
}

// 32 x 32 tiles through LDS; block = 32 x 8 threads.
template <class TI, class TO>
__global__ __launch_bounds__(256) void block_copy_kernel(const BlockCopy a) {
  __shared__ TO tile[TILE][TILE + 1];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int c0 = blockIdx.x * TILE, r0 = blockIdx.y * TILE;
  const int outer = blockIdx.z / a.n_inner, inner = blockIdx.z - outer * a.n_inner;
  const TI* in = static_cast<const TI*>(a.in) + (a.in_off ? a.in_off[outer] : 0) + inner * a.in_bs;
  TO* out = static_cast<TO*>(a.out) + (a.out_off ? a.out_off[outer] : 0) + inner * a.out_bs;
  const bool tr = a.trans ? a.trans[outer] != 0 : a.trans_all != 0;
  const bool cg = a.conj ? a.conj[outer] != 0 : a.conj_all != 0;
  if (tr) {
    // in is cols x rows: element (r, c) of the output is in[c][r].
#pragma unroll
    for (int j = 0; j < TILE; j += 8) {
      const int c = c0 + ty + j, r = r0 + tx;
      if (c < a.cols && r < a.rows) {
        if constexpr (sizeof(TI) == sizeof(TO)) tile[ty + j][tx] = in[c * a.in_ld + r];
        else tile[ty + j][tx] = narrow(in[c * a.in_ld + r]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TILE; j += 8) {
      const int r = r0 + ty + j, c = c0 + tx;
      if (r < a.rows && c < a.cols) {
        TO v = tile[tx][ty + j];
        if (a.scale != 1.0) v = scl(v, a.scale);
        out[r * a.out_ld + c] = cg ? cjt(v) : v;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < TILE; j += 8) {
      const int r = r0 + ty + j, c = c0 + tx;
      if (r < a.rows && c < a.cols) {
        TO v;
        if constexpr (sizeof(TI) == sizeof(TO)) v = in[r * a.in_ld + c];
        else v = narrow(in[r * a.in_ld + c]);
        if (a.scale != 1.0) v = scl(v, a.scale);
        out[r * a.out_ld + c] = cg ? cjt(v) : v;
      }
    }
  }
}

__global__ void to_c32_kernel(const z64* in, c32* out, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = c32{(float)in[i].x, (float)in[i].y};
}

__global__ void slab_gather_kernel(const z64* in, const int64_t* src_off, z64* out,
                                   const int64_t* dst_off, int n_slabs, int64_t len, double scale) {
  const int64_t total = (int64_t)n_slabs * len;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t o = e / len, i = e - o * len;
    const z64 v = in[src_off[o] + i];
    out[dst_off[o] + i] = z64{scale * v.x, scale * v.y};
  }
}

__global__ __launch_bounds__(256) void herm_one_minus_kernel(z64* M, z64* A, int n) {
  __shared__ z64 t1[TILE][TILE + 1];
  __shared__ z64 t2[TILE][TILE + 1];
  // lower-triangular tile pair index -> (bi, bj), bi >= bj
  const int x = blockIdx.x;
  int bi = (int)((sqrt(8.0 * x + 1.0) - 1.0) * 0.5);
  while ((bi + 1) * (bi + 2) / 2 <= x) ++bi;
  while (bi * (bi + 1) / 2 > x) --bi;
  const int bj = x - bi * (bi + 1) / 2;
  const int64_t w = blockIdx.y;
  z64* Mw = M + w * (int64_t)n * n;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int ri = bi * TILE, rj = bj * TILE;
#pragma unroll
  for (int j = 0; j < TILE; j += 8) {
    const int r = ty + j;
    if (ri + r < n && rj + tx < n) t1[r][tx] = Mw[(int64_t)(ri + r) * n + rj + tx];   // tile (bi, bj)
    if (rj + r < n && ri + tx < n) t2[r][tx] = Mw[(int64_t)(rj + r) * n + ri + tx];   // tile (bj, bi)
  }
  __syncthreads();
  z64* Aw = A ? A + w * (int64_t)n * n : nullptr;
#pragma unroll
  for (int j = 0; j < TILE; j += 8) {
    const int r = ty + j;
    // element (ri + r, rj + tx) of H = (M + M^dagger)/2
    if (ri + r < n && rj + tx < n) {
      const z64 a = t1[r][tx], b = t2[tx][r];
      z64 h = z64{0.5 * (a.x + b.x), 0.5 * (a.y - b.y)};
      const int64_t idx = (int64_t)(ri + r) * n + rj + tx;
      Mw[idx] = h;
      if (Aw) Aw[idx] = z64{(ri + r == rj + tx ? 1.0 : 0.0) - h.x, -h.y};
    }
    // element (rj + r, ri + tx)
    if (bi != bj && rj + r < n && ri + tx < n) {
      const z64 a = t2[r][tx], b = t1[tx][r];
      z64 h = z64{0.5 * (a.x + b.x), 0.5 * (a.y - b.y)};
      const int64_t idx = (int64_t)(rj + r) * n + ri + tx;
      Mw[idx] = h;
      if (Aw) Aw[idx] = z64{-h.x, -h.y};
    }
  }
}

__global__ void zero_kernel(z64* p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = z64{0.0, 0.0};
}
__global__ void zero_int_kernel(int* p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0;
}
constexpr int NBMAX = 32;

// The small factorisation and solve kernels below are serial chains of nb
// steps; what bounds them is the latency of one step.  Step s makes one element
// of every row (or column) final and the others are updated with it, so the
// nb elements are dealt to G groups of lanes, element e to group e mod G, local
// index e / G: in registers, because the local index is unrolled, with code
// small enough to stay in the instruction cache, because the group is not.
// (Whole rows per lane, unrolled 32 x 32, ran at the speed of instruction
// fetch: 24 us per triangular solve, no faster than the chains through LDS.)  A
// step costs one exchange through LDS and one barrier; the two buffers of the
// exchange take turns, so one barrier is enough.
// Measured at NQ = 154, 70 frequencies (in brackets the same steps as one chain
// through LDS or global memory per row): LU panel 37-47 us (65-91), forward
// solve of 32 rows 12-15 us (28-38), Cholesky diagonal block 16 us (40), panel
// 15 us (25).
//
// Which product of a complex product is fused with the other is written out:
// left to the compiler it follows its order of the operands, and a kernel that
// is only rearranged would round differently.
__device__ inline z64 mul(z64 a, z64 b) {    // a b
  return z64{__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.y, b.x, a.x * b.y)};
}
__device__ inline z64 mulc(z64 a, z64 b) {   // a conj(b)
  return z64{__builtin_fma(a.x, b.x, a.y * b.y), __builtin_fma(a.y, b.x, -(a.x * b.y))};
}

constexpr int SG = 4;              // groups = waves of a triangular solve
constexpr int SL = NBMAX / SG;     // elements per lane

// Solve T y = y for 64 right-hand sides, one per lane; group g (a wave) holds
// elements 4 j + g.  T: 32 x 32 lower triangle in LDS.  Every element's sum runs
// over ascending s, as a solve row by row sums it.
// KIND: kTriLower  T non-unit (Cholesky L, forward)
//       kTriUnitLower  T unit lower (LU L, forward)
//       kTriConjLower  conj(T), non-unit (Cholesky panel)
enum { kTriLower, kTriUnitLower, kTriConjLower };

template <int KIND>
__device__ inline void solve_lower(const z64 (&T)[NBMAX][NBMAX], z64 (&ex)[2][64], double (&rd)[NBMAX], z64 (&y)[SL],
                                   int nb) {
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  // reciprocals of the diagonal, out of the chain
  if (KIND != kTriUnitLower) {
    if (threadIdx.x < nb) rd[threadIdx.x] = 1.0 / T[threadIdx.x][threadIdx.x].x;
    __syncthreads();
  }
  auto term = [&](int r, int s, z64 ys) {
    return KIND == kTriConjLower ? mulc(ys, T[r][s]) : mul(T[r][s], ys);
  };
#pragma unroll
  for (int k = 0; k < SL; ++k) {
#pragma unroll 1
    for (int gg = 0; gg < SG; ++gg) {
      const int s = SG * k + gg;
      if (s >= nb) break;
      if (g == gg) {
        if (KIND != kTriUnitLower) y[k] = z64{y[k].x * rd[s], y[k].y * rd[s]};
        ex[s & 1][lane] = y[k];
      }
      __syncthreads();
      const z64 ys = ex[s & 1][lane];
      // the group's element of the same local index first: the next step needs it
      if (g > gg) y[k] = csub(y[k], term(SG * k + g, s, ys));
#pragma unroll
      for (int j = k + 1; j < SL; ++j) y[j] = csub(y[j], term(SG * j + g, s, ys));
    }
  }
}

// The nb x nb triangle at (i0, i0) of A into LDS, zero past nb.
__device__ inline void load_triangle(z64 (&T)[NBMAX][NBMAX], const z64* Aw, int64_t lda, int i0, int nb) {
  for (int e = threadIdx.x; e < NBMAX * NBMAX; e += blockDim.x) {
    const int r = e / NBMAX, c = e % NBMAX;
    T[r][c] = (r < nb && c < nb) ? Aw[(int64_t)(i0 + r) * lda + i0 + c] : z64{0.0, 0.0};
  }
}

// Cholesky of the nb x nb diagonal block, one workgroup per matrix: lane r of
// group g (32 lanes) holds elements 8 j + g of row r.
constexpr int DG = 8, DL = NBMAX / DG;
__global__ __launch_bounds__(32 * DG) void chol_diag_kernel(z64* A, int n, int j0, int nb, int* info) {
  __shared__ z64 col[2][NBMAX];
  const int64_t w = blockIdx.x;
  const int r = threadIdx.x & 31, g = threadIdx.x >> 5;
  z64* Ar = A + w * (int64_t)n * n + (int64_t)(j0 + min(r, nb - 1)) * n + j0;
  z64 x[DL];
#pragma unroll
  for (int j = 0; j < DL; ++j) x[j] = (DG * j + g <= r && r < nb) ? Ar[DG * j + g] : z64{0.0, 0.0};
#pragma unroll
  for (int k = 0; k < DL; ++k) {
#pragma unroll 1
    for (int gg = 0; gg < DG; ++gg) {
      const int c = DG * k + gg;
      if (c >= nb) break;
      if (g == gg) {
        double d = __shfl(x[k].x, c, 32);
        if (!(d > 0.0)) {                  // not positive definite (or NaN)
          if (r == 0 && info[w] == 0) info[w] = j0 + c + 1;
          d = 1.0;
        } else {
          d = sqrt(d);
        }
        const double inv = 1.0 / d;
        if (r > c) x[k] = z64{x[k].x * inv, x[k].y * inv};
        else if (r == c) x[k] = z64{d, 0.0};
        col[c & 1][r] = x[k];
      }
      __syncthreads();
      const z64 l = col[c & 1][r];
#pragma unroll
      for (int j = 0; j < DL; ++j) {
        const int s = DG * j + g;
        if (j >= k && s > c && s <= r) x[j] = csub(x[j], mulc(l, col[c & 1][s]));
      }
    }
  }
#pragma unroll
  for (int j = 0; j < DL; ++j)
    if (DG * j + g <= r && r < nb) Ar[DG * j + g] = x[j];
}

// Rows below the diagonal block: x L11^dagger = a.  64 rows per workgroup, one
// per lane; rows pass through LDS so that memory is read along them.
__global__ __launch_bounds__(64 * SG) void chol_panel_kernel(z64* A, int n, int j0, int nb) {
  __shared__ z64 T[NBMAX][NBMAX], ex[2][64];
  __shared__ z64 X[64][NBMAX + 1];
  __shared__ double rd[NBMAX];
  z64* Aw = A + blockIdx.y * (int64_t)n * n;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int r0 = j0 + nb + blockIdx.x * 64;
  load_triangle(T, Aw, n, j0, nb);
  for (int e = threadIdx.x; e < 64 * NBMAX; e += 64 * SG) {
    const int r = e / NBMAX, c = e % NBMAX;
    X[r][c] = (c < nb && r0 + r < n) ? Aw[(int64_t)(r0 + r) * n + j0 + c] : z64{0.0, 0.0};
  }
  __syncthreads();
  z64 y[SL];
#pragma unroll
  for (int j = 0; j < SL; ++j) y[j] = X[lane][SG * j + g];
  solve_lower<kTriConjLower>(T, ex, rd, y, nb);
#pragma unroll
  for (int j = 0; j < SL; ++j) X[lane][SG * j + g] = y[j];
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * NBMAX; e += 64 * SG) {
    const int r = e / NBMAX, c = e % NBMAX;
    if (c < nb && r0 + r < n) Aw[(int64_t)(r0 + r) * n + j0 + c] = X[r][c];
  }
}

// Triangular solve with the nb x nb diagonal block T at (i0, i0) of the
// matrix A (row stride lda) on rows i0 .. i0+nb of B, columns bcol0 ..
// bcol0+ncols; 64 right-hand-side columns per workgroup, one per lane.
template <int KIND>
__global__ __launch_bounds__(64 * SG) void trsm_lower_kernel(const z64* A, int lda, int64_t a_ms, z64* B, int ldb,
                                                             int64_t b_ms, int bcol0, int ncols, int i0, int nb) {
  __shared__ z64 T[NBMAX][NBMAX], ex[2][64];
  __shared__ double rd[NBMAX];
  const int64_t w = blockIdx.y;
  const int g = threadIdx.x >> 6, col = blockIdx.x * 64 + (threadIdx.x & 63);
  z64* Bc = B + w * b_ms + (int64_t)i0 * ldb + bcol0 + min(col, ncols - 1);
  load_triangle(T, A + w * a_ms, lda, i0, nb);
  z64 y[SL];
#pragma unroll
  for (int j = 0; j < SL; ++j) y[j] = SG * j + g < nb ? Bc[(int64_t)(SG * j + g) * ldb] : z64{0.0, 0.0};
  __syncthreads();
  solve_lower<KIND>(T, ex, rd, y, nb);
  if (col >= ncols) return;
#pragma unroll
  for (int j = 0; j < SL; ++j)
    if (SG * j + g < nb) Bc[(int64_t)(SG * j + g) * ldb] = y[j];
}

// The backward solves: T^dagger of the lower L (HERM, Cholesky) or T upper
// non-unit (LU).  A row's sum runs over ascending s, so it starts with the
// element just solved and cannot run ahead; one wave per 64 columns, eight terms
// at a time so that their reads are in flight together.  Terms past nb are
// zeros.  25-32 us at the size above (28-38 one term at a time).
template <bool HERM>
__global__ __launch_bounds__(64) void trsm_back_kernel(const z64* A, int lda, int64_t a_ms, z64* B, int ldb,
                                                       int64_t b_ms, int bcol0, int ncols, int i0, int nb) {
  constexpr int CH = 8;
  __shared__ z64 U[NBMAX][NBMAX + CH];   // U[r][s]: L[s][r] or T[r][s], raw
  __shared__ z64 Y[NBMAX + CH][64];
  __shared__ double rd[NBMAX];
  const int64_t w = blockIdx.y;
  const z64* Aw = A + w * a_ms;
  const int lane = threadIdx.x, col = blockIdx.x * 64 + lane;
  z64* Bc = B + w * b_ms + (int64_t)i0 * ldb + bcol0 + min(col, ncols - 1);
  for (int e = lane; e < NBMAX * NBMAX; e += 64) {
    const int r = e / NBMAX, c = e % NBMAX;
    const z64 v = (r < nb && c < nb) ? Aw[(int64_t)(i0 + r) * lda + i0 + c] : z64{0.0, 0.0};
    if (HERM) U[c][r] = v;
    else U[r][c] = v;
  }
  for (int e = lane; e < NBMAX * CH; e += 64) U[e / CH][NBMAX + e % CH] = z64{0.0, 0.0};
#pragma unroll 8
  for (int r = 0; r < NBMAX + CH; ++r) Y[r][lane] = r < nb ? Bc[(int64_t)min(r, nb - 1) * ldb] : z64{0.0, 0.0};
  __syncthreads();
  if (lane < nb) {
    const z64 d = U[lane][lane];
    rd[lane] = 1.0 / (HERM ? d.x : __builtin_fma(d.x, d.x, d.y * d.y));
  }
  __syncthreads();
  for (int r = nb - 1; r >= 0; --r) {
    z64 acc = Y[r][lane];
    for (int s0 = r + 1; s0 < nb; s0 += CH) {
      z64 u[CH], y[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        u[i] = U[r][s0 + i];
        y[i] = Y[s0 + i][lane];
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) acc = csub(acc, HERM ? mulc(y[i], u[i]) : mul(u[i], y[i]));
    }
    if (!HERM) acc = mulc(acc, U[r][r]);
    acc = z64{acc.x * rd[r], acc.y * rd[r]};
    Y[r][lane] = acc;
    if (col < ncols) Bc[(int64_t)r * ldb] = acc;
  }
}

// One step of a maximum over 16 lanes (larger value, then smaller index) with
// the lane that the data-parallel primitive DPP exchanges with.
template <int DPP>
__device__ inline void max_step(double& v, int& i) {
  const long long b = __double_as_longlong(v);
  const int lo = (int)b, hi = (int)(b >> 32);
  const uint32_t lo2 = __builtin_amdgcn_update_dpp(lo, lo, DPP, 0xF, 0xF, false);
  const uint32_t hi2 = __builtin_amdgcn_update_dpp(hi, hi, DPP, 0xF, 0xF, false);
  const int i2 = __builtin_amdgcn_update_dpp(i, i, DPP, 0xF, 0xF, false);
  const double v2 = __longlong_as_double((long long)(((uint64_t)hi2 << 32) | lo2));
  if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
}
__device__ inline void max_16_lanes(double& v, int& i) {
  max_step<0xB1>(v, i);    // quad_perm 1 0 3 2
  max_step<0x4E>(v, i);    // quad_perm 2 3 0 1
  max_step<0x141>(v, i);   // row_half_mirror
  max_step<0x140>(v, i);   // row_mirror
}

// LU with partial pivoting of the panel of columns j0 .. j0+nb, rows j0 .. n
// (LAPACK zgetf2 semantics on the panel): one workgroup per matrix, the panel
// in registers: wave (b, g) of SG x ceil(rows / (64 RB)) holds columns 4 j + g
// of rows 64 RB b + 64 i + lane (at most LU_ROWS rows; lu_panel_global_kernel
// takes longer panels).  Pivot = first row of largest |re| + |im| (izamax); the
// row swaps are applied inside the panel only (lu_row_swaps applies them to
// the other columns).  ipiv[w * n + c] = pivot row of column c (0-based);
// info[w] = column + 1 of the first exactly zero pivot (0 = none).
constexpr int LU_ROWS = 512;

template <int RB>
__global__ __launch_bounds__(1024) void lu_panel_kernel(z64* A, int n, int j0, int nb, int* ipiv, int* info) {
  __shared__ double sval[1024 / 64];
  __shared__ int sidx[1024 / 64];
  // the column of the step before the swap (buffers take turns: a wave may read
  // one step's while the next step's is written)
  __shared__ z64 colv[2][64 * RB * (1024 / 64 / SG)];
  __shared__ z64 prow[NBMAX], crow[NBMAX];   // the pivot row and the row it replaces
  const int64_t w = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = wave % SG, b = wave / SG, nwb = (blockDim.x >> 6) / SG;
  const int rows = n - j0;
  z64* Aw = A + w * (int64_t)n * n + (int64_t)j0 * n + j0;
  int row[RB];
  z64 a[RB][SL];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    row[i] = (b * RB + i) * 64 + lane;
#pragma unroll
    for (int j = 0; j < SL; ++j)
      a[i][j] = (row[i] < rows && SG * j + g < nb) ? Aw[(int64_t)row[i] * n + SG * j + g] : z64{0.0, 0.0};
  }
#pragma unroll
  for (int k = 0; k < SL; ++k) {
#pragma unroll 1
    for (int gg = 0; gg < SG; ++gg) {
      const int c = SG * k + gg;
      if (c >= nb) break;
      if (g == gg) {
        // a NaN never wins; with nothing but NaN the pivot is the diagonal
        double best = -1.0;
        int p = c;
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          colv[c & 1][row[i]] = a[i][k];
          const double m = fabs(a[i][k].x) + fabs(a[i][k].y);
          if (row[i] >= c && row[i] < rows && m > best) { best = m; p = row[i]; }
        }
        max_16_lanes(best, p);
        if ((lane & 15) == 0) { sval[4 * b + lane / 16] = best; sidx[4 * b + lane / 16] = p; }
      }
      __syncthreads();
      // the 4 nwb <= 16 partial maxima, one per lane
      double best = -2.0;
      int p = c;
      if ((lane & 15) < 4 * nwb) { best = sval[lane & 15]; p = sidx[lane & 15]; }
      max_16_lanes(best, p);
      p = __builtin_amdgcn_readfirstlane(p);
      if (threadIdx.x == 0) ipiv[w * n + j0 + c] = j0 + p;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if (row[i] == p)
#pragma unroll
          for (int j = 0; j < SL; ++j) prow[SG * j + g] = a[i][j];
        if (row[i] == c && p != c)
#pragma unroll
          for (int j = 0; j < SL; ++j) crow[SG * j + g] = a[i][j];
      }
      const z64 piv = colv[c & 1][p];
      const bool zero_piv = piv.x == 0.0 && piv.y == 0.0;
      if (zero_piv && threadIdx.x == 0 && info[w] == 0) info[w] = j0 + c + 1;
      const double d = 1.0 / __builtin_fma(piv.x, piv.x, piv.y * piv.y);
      const z64 inv = z64{piv.x * d, -piv.y * d};
      z64 l[RB];   // the multiplier of the row that stands here after the swap
#pragma unroll
      for (int i = 0; i < RB; ++i) l[i] = mul(inv, colv[c & 1][row[i] == p ? c : row[i]]);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        if (p != c && (row[i] == c || row[i] == p))
#pragma unroll
          for (int j = 0; j < SL; ++j) a[i][j] = row[i] == c ? prow[SG * j + g] : crow[SG * j + g];
        if (row[i] > c && !zero_piv) {
          if (g == gg) a[i][k] = l[i];
          if (g > gg) a[i][k] = csub(a[i][k], mul(l[i], prow[SG * k + g]));
#pragma unroll
          for (int j = k + 1; j < SL; ++j) a[i][j] = csub(a[i][j], mul(l[i], prow[SG * j + g]));
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < SL; ++j)
      if (row[i] < rows && SG * j + g < nb) Aw[(int64_t)row[i] * n + SG * j + g] = a[i][j];
}

// The same for panels of more than LU_ROWS rows, the panel in global memory.
constexpr int LU_THREADS = 256;

__global__ __launch_bounds__(LU_THREADS) void lu_panel_global_kernel(z64* A, int n, int j0, int nb, int* ipiv, int* info) {
  __shared__ double sval[LU_THREADS];
  __shared__ int sidx[LU_THREADS];
  __shared__ z64 srow[NBMAX];
  const int64_t w = blockIdx.x;
  z64* Aw = A + w * (int64_t)n * n;
  const int tid = threadIdx.x;
  for (int c = j0; c < j0 + nb; ++c) {
    double best = -1.0;
    int bi = c;                                // also the pivot if every entry is NaN
    for (int r = c + tid; r < n; r += LU_THREADS) {
      const z64 v = Aw[(int64_t)r * n + c];
      const double a = fabs(v.x) + fabs(v.y);
      if (a > best) { best = a; bi = r; }      // rows visited in increasing order: ties keep the first
    }
    sval[tid] = best;
    sidx[tid] = bi;
    __syncthreads();
    for (int h = LU_THREADS / 2; h > 0; h >>= 1) {
      if (tid < h) {
        const double o = sval[tid + h];
        const int oi = sidx[tid + h];
        if (o > sval[tid] || (o == sval[tid] && oi < sidx[tid])) { sval[tid] = o; sidx[tid] = oi; }
      }
      __syncthreads();
    }
    const int p = sidx[0];
    if (tid == 0) ipiv[w * n + c] = p;
    // swap rows c and p inside the panel
    if (p != c && tid < nb) {
      const int64_t a = (int64_t)c * n + j0 + tid, b = (int64_t)p * n + j0 + tid;
      const z64 t = Aw[a];
      Aw[a] = Aw[b];
      Aw[b] = t;
    }
    __syncthreads();
    const z64 piv = Aw[(int64_t)c * n + c];
    const bool zero_piv = piv.x == 0.0 && piv.y == 0.0;
    if (zero_piv) {
      if (tid == 0 && info[w] == 0) info[w] = c + 1;
    } else {
      const double m = 1.0 / (piv.x * piv.x + piv.y * piv.y);
      const z64 inv = z64{piv.x * m, -piv.y * m};
      for (int r = c + 1 + tid; r < n; r += LU_THREADS) {
        const int64_t a = (int64_t)r * n + c;
        Aw[a] = cmul(Aw[a], inv);
      }
    }
    if (tid < j0 + nb - c - 1) srow[tid] = Aw[(int64_t)c * n + c + 1 + tid];
    __syncthreads();
    // rank-1 update of the panel's remaining columns
    const int m = j0 + nb - c - 1;
    if (m > 0 && !zero_piv) {
      const int rows = n - c - 1;
      for (int e = tid; e < rows * m; e += LU_THREADS) {
        const int r = c + 1 + e / m, cc = e - (e / m) * m;
        const int64_t a = (int64_t)r * n + c + 1 + cc;
        Aw[a] = csub(Aw[a], cmul(Aw[(int64_t)r * n + c], srow[cc]));
      }
    }
    __syncthreads();
  }
}

// Apply the row interchanges ipiv[w * ldp + i], i = i_begin .. i_end (in
// order), to the columns of B outside [skip_lo, skip_hi): one thread per
// column.  B: nw matrices of ldb columns, row stride ldb, matrix stride b_ms.
__global__ __launch_bounds__(256) void lu_row_swaps_kernel(z64* B, int ldb, int64_t b_ms, int ncols,
                                                           const int* ipiv, int ldp, int i_begin, int i_end,
                                                           int skip_lo, int skip_hi) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= ncols || (c >= skip_lo && c < skip_hi)) return;
  const int64_t w = blockIdx.y;
  z64* Bw = B + w * b_ms;
  const int* pw = ipiv + w * ldp;
  for (int i = i_begin; i < i_end; ++i) {
    const int p = pw[i];
    if (p != i) {
      const z64 t = Bw[(int64_t)i * ldb + c];
      Bw[(int64_t)i * ldb + c] = Bw[(int64_t)p * ldb + c];
      Bw[(int64_t)p * ldb + c] = t;
    }
  }
}

__device__ inline uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Complex Gaussian sample for counter e (two uniforms from one hash chain,
// Box-Muller).  The host generator of the test suite uses the same formulas.
__device__ inline z64 gauss_c(uint64_t seed, uint64_t e, double sigma) {
  const uint64_t h1 = splitmix64(seed * 0xD1B54A32D192ED03ull + e);
  const uint64_t h2 = splitmix64(h1);
  const double u1 = ((double)(h1 >> 11) + 0.5) * 0x1.0p-53;
  const double u2 = (double)(h2 >> 11) * 0x1.0p-53;
  const double rad = sigma * sqrt(-2.0 * log(u1));
  const double ang = 6.283185307179586 * u2;
  double sn, cs;
  sincos(ang, &sn, &cs);
  return z64{rad * cs, rad * sn};
}

// One pair per grid row (blockIdx.y), the pair's NQ * nao^2 elements along
// x: no 64-bit index division per element (they cost more than the Gaussian
// itself).  Counter of element (Q, i, j) of stored pair p:
// (p * NQ + Q) * nao^2 + i * nao + j.
__global__ void synth_integrals_kernel(z64* V, int64_t p0, const int* diag, int NQ, int nao, uint64_t seed,
                                       double sigma) {
  const int nn = nao * nao;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;   // element of the pair
  if (e >= NQ * nn) return;
  const int64_t lp = blockIdx.y;
  const int Q = e / nn, ij = e - Q * nn;
  const uint64_t base = ((uint64_t)(p0 + lp) * NQ + Q) * nn;
  z64 v = gauss_c(seed, base + ij, sigma);
  if (diag[lp]) {
    const int i = ij / nao, j = ij - i * nao;
    const z64 t = gauss_c(seed, base + j * nao + i, sigma);
    v = z64{0.5 * (v.x + t.x), 0.5 * (v.y - t.y)};
  }
  V[lp * NQ * nn + e] = v;
}

inline int grid_for(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

void block_copy(const BlockCopy& a, hipStream_t s) {
  if (a.rows <= 0 || a.cols <= 0 || a.n_outer <= 0 || a.n_inner <= 0) return;
  require(a.n_inner <= 65535, "block_copy: inner batch above 65535");
  require(!(a.in_f32 && !a.out_f32), "block_copy: complex64 -> complex128 not supported");
  // grid.z is limited to 65535: launch the outer batches in chunks
  const int per = 65535 / a.n_inner;
  for (int o0 = 0; o0 < a.n_outer; o0 += per) {
    BlockCopy c = a;
    c.n_outer = std::min(per, a.n_outer - o0);
    if (c.in_off) c.in_off += o0;
    if (c.out_off) c.out_off += o0;
    if (c.trans) c.trans += o0;
    if (c.conj) c.conj += o0;
    dim3 grid((c.cols + TILE - 1) / TILE, (c.rows + TILE - 1) / TILE, c.n_outer * c.n_inner);
    if (!c.in_f32 && !c.out_f32) hipLaunchKernelGGL((block_copy_kernel<z64, z64>), grid, dim3(256), 0, s, c);
    else if (!c.in_f32) hipLaunchKernelGGL((block_copy_kernel<z64, c32>), grid, dim3(256), 0, s, c);
    else hipLaunchKernelGGL((block_copy_kernel<c32, c32>), grid, dim3(256), 0, s, c);
    GGPU_HIP(hipGetLastError());
  }
}

void slab_gather(const z64* in, const int64_t* src_off, z64* out, const int64_t* dst_off, int n_slabs,
                 int64_t len, double scale, hipStream_t s) {
  if (n_slabs <= 0 || len <= 0) return;
  hipLaunchKernelGGL(slab_gather_kernel, dim3(grid_for(n_slabs * len, 256)), dim3(256), 0, s, in, src_off,
                     out, dst_off, n_slabs, len, scale);
  GGPU_HIP(hipGetLastError());
}

void herm_one_minus(z64* M, z64* A, int n, int nw, hipStream_t s) {
  if (n <= 0 || nw <= 0) return;
  const int T = (n + TILE - 1) / TILE;
  require(nw <= 65535, "herm_one_minus: too many matrices");
  hipLaunchKernelGGL(herm_one_minus_kernel, dim3(T * (T + 1) / 2, nw), dim3(256), 0, s, M, A, n);
  GGPU_HIP(hipGetLastError());
}

void to_c32(const z64* in, c32* out, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(to_c32_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, in, out, n);
  GGPU_HIP(hipGetLastError());
}

void zero(z64* p, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(zero_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n);
  GGPU_HIP(hipGetLastError());
}

void zero_int(int* p, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(zero_int_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, p, n);
  GGPU_HIP(hipGetLastError());
}

void chol_diag_block(z64* A, int n, int nw, int j0, int nb, int* info, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && j0 >= 0 && j0 + nb <= n, "chol_diag_block: bad block");
  require(nw <= 2147483647, "chol_diag_block: nw");
  hipLaunchKernelGGL(chol_diag_kernel, dim3(nw), dim3(32 * DG), 0, s, A, n, j0, nb, info);
  GGPU_HIP(hipGetLastError());
}

void chol_panel(z64* A, int n, int nw, int j0, int nb, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && j0 >= 0 && j0 + nb <= n, "chol_panel: bad block");
  const int rows = n - j0 - nb;
  if (rows <= 0) return;
  require(nw <= 65535, "chol_panel: nw");
  hipLaunchKernelGGL(chol_panel_kernel, dim3((rows + 63) / 64, nw), dim3(64 * SG), 0, s, A, n, j0, nb);
  GGPU_HIP(hipGetLastError());
}

void trsm_lower_block(const z64* L, z64* B, int n, int nrhs, int nw, int i0, int nb, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && i0 >= 0 && i0 + nb <= n && nw <= 65535, "trsm_lower_block: bad block");
  if (nrhs <= 0) return;
  hipLaunchKernelGGL((trsm_lower_kernel<kTriLower>), dim3((nrhs + 63) / 64, nw), dim3(64 * SG), 0, s, L, n,
                     (int64_t)n * n, B, nrhs, (int64_t)n * nrhs, 0, nrhs, i0, nb);
  GGPU_HIP(hipGetLastError());
}

void trsm_upper_h_block(const z64* L, z64* B, int n, int nrhs, int nw, int i0, int nb, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && i0 >= 0 && i0 + nb <= n && nw <= 65535, "trsm_upper_h_block: bad block");
  if (nrhs <= 0) return;
  hipLaunchKernelGGL((trsm_back_kernel<true>), dim3((nrhs + 63) / 64, nw), dim3(64), 0, s, L, n, (int64_t)n * n, B,
                     nrhs, (int64_t)n * nrhs, 0, nrhs, i0, nb);
  GGPU_HIP(hipGetLastError());
}

void lu_panel(z64* A, int n, int nw, int j0, int nb, int* ipiv, int* info, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && j0 >= 0 && j0 + nb <= n, "lu_panel: bad block");
  const int rows = n - j0;
  if (rows <= LU_ROWS / 2)
    hipLaunchKernelGGL((lu_panel_kernel<1>), dim3(nw), dim3((rows + 63) / 64 * 64 * SG), 0, s, A, n, j0, nb, ipiv, info);
  else if (rows <= LU_ROWS)
    hipLaunchKernelGGL((lu_panel_kernel<2>), dim3(nw), dim3((rows + 127) / 128 * 64 * SG), 0, s, A, n, j0, nb, ipiv,
                       info);
  else
    hipLaunchKernelGGL(lu_panel_global_kernel, dim3(nw), dim3(LU_THREADS), 0, s, A, n, j0, nb, ipiv, info);
  GGPU_HIP(hipGetLastError());
}

void lu_row_swaps(z64* B, int ldb, int ncols, int nw, const int* ipiv, int ldp, int i_begin, int i_end, int skip_lo,
                  int skip_hi, hipStream_t s) {
  require(i_begin >= 0 && i_end <= ldp && nw <= 65535 && ncols <= ldb, "lu_row_swaps: bad range");
  if (ncols <= 0 || i_end <= i_begin) return;
  hipLaunchKernelGGL(lu_row_swaps_kernel, dim3((ncols + 255) / 256, nw), dim3(256), 0, s, B, ldb,
                     (int64_t)ldp * ldb, ncols, ipiv, ldp, i_begin, i_end, skip_lo, skip_hi);
  GGPU_HIP(hipGetLastError());
}

void trsm_unit_lower_cols(const z64* A, z64* B, int n, int nw, int i0, int nb, int bcol0, int ncols, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && i0 >= 0 && i0 + nb <= n && nw <= 65535 && bcol0 >= 0 && bcol0 + ncols <= n,
          "trsm_unit_lower_cols: bad block");
  if (ncols <= 0) return;
  hipLaunchKernelGGL((trsm_lower_kernel<kTriUnitLower>), dim3((ncols + 63) / 64, nw), dim3(64 * SG), 0, s, A, n,
                     (int64_t)n * n, B, n, (int64_t)n * n, bcol0, ncols, i0, nb);
  GGPU_HIP(hipGetLastError());
}

void trsm_upper_cols(const z64* A, z64* B, int n, int nw, int i0, int nb, int bcol0, int ncols, hipStream_t s) {
  require(nb >= 1 && nb <= NBMAX && i0 >= 0 && i0 + nb <= n && nw <= 65535 && bcol0 >= 0 && bcol0 + ncols <= n,
          "trsm_upper_cols: bad block");
  if (ncols <= 0) return;
  hipLaunchKernelGGL((trsm_back_kernel<false>), dim3((ncols + 63) / 64, nw), dim3(64), 0, s, A, n, (int64_t)n * n, B,
                     n, (int64_t)n * n, bcol0, ncols, i0, nb);
  GGPU_HIP(hipGetLastError());
}

void synth_integrals(z64* V, int64_t p0, int64_t np, const int* pair_is_diag, int NQ, int nao, uint64_t seed,
                     double sigma, hipStream_t s) {
  if (np <= 0) return;
  const int64_t per_pair = (int64_t)NQ * nao * nao;
  require(per_pair < ((int64_t)1 << 31), "synth_integrals: NQ * nao^2 above 2^31");
  const unsigned bx = (unsigned)((per_pair + 255) / 256);
  // grid.y is limited to 65535: launch the pairs in chunks
  for (int64_t c = 0; c < np; c += 65535) {
    const int64_t n = std::min<int64_t>(65535, np - c);
    hipLaunchKernelGGL(synth_integrals_kernel, dim3(bx, (unsigned)n), dim3(256), 0, s, V + c * per_pair, p0 + c,
                       pair_is_diag + c, NQ, nao, seed, sigma);
    GGPU_HIP(hipGetLastError());
  }
}

}  // namespace ggpu
