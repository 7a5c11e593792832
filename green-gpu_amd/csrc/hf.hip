// Kernels of the Hartree term, the Fock assembly and the HF energy.
//
// All are reductions over the integrals or over small matrices, bound by HBM
// reads when the system is large and by the latency of one load chain when it
// is small, so each splits its sum over as many lanes as the sum has terms
// and reads the stored pair blocks where they lie (no unfolded copy).  As
// matrix products with one row or column they kept one lane of 64 busy:
// nk = 64, nao = 52, NQ = 300, ns = 2: Hartree vector 24.6 ms -> 0.4 ms,
// traces 0.32 ms -> 5 us; partial sums of K one slice after the other 12.5 ms.
#include "hf.hpp"

#include <algorithm>

namespace ggpu {
namespace {

__device__ inline z64 cfma(z64 a, z64 b, z64 c) {
  return z64{c.x + a.x * b.x - a.y * b.y, c.y + a.x * b.y + a.y * b.x};
}

// Sum over the 256 threads of a workgroup; valid in thread 0.
__device__ inline z64 block_sum(z64 v) {
  __shared__ z64 part[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    v.x += __shfl_down(v.x, o);
    v.y += __shfl_down(v.y, o);
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  z64 t = part[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) { t.x += part[w].x; t.y += part[w].y; }
  return t;
}

// One workgroup per (Q, pair); lanes run along the stored block.
__global__ __launch_bounds__(256) void hartree_vector_kernel(const PairBlocks v, int NQ, int nao, const z64* D, int nps,
                                                             int nj, double scale, z64* part) {
  const int Q = blockIdx.x, b = blockIdx.y, n2 = nao * nao;
  const z64* S = v.base + v.off[b] + (int64_t)Q * n2;
  const z64* Db = D + (int64_t)b * nps * n2;
  const bool tr = v.trans[b] != 0, cg = v.conj[b] != 0;
  z64 acc{0.0, 0.0};
  for (int e = threadIdx.x; e < n2; e += 256) {
    z64 x = S[e];
    if (cg) x.y = -x.y;
    // element (r, c) of the stored block is V[r][c], or V[c][r] if transposed,
    // and meets D[c][r] or D[r][c]
    const int r = e / nao, c = e - r * nao, m = tr ? e : c * nao + r;
    for (int s = 0; s < nj; ++s) acc = cfma(x, Db[(int64_t)s * n2 + m], acc);
  }
  const z64 t = block_sum(acc);
  if (threadIdx.x == 0) part[(int64_t)b * NQ + Q] = z64{scale * t.x, scale * t.y};
}

// 64 elements of the stored block x 8 groups of Q per workgroup.
constexpr int JG = 8;
__global__ __launch_bounds__(64 * JG) void hartree_fock_kernel(const PairBlocks v, int NQ, int nao, const z64* jvec,
                                                               z64* F, int nps, int nj) {
  __shared__ z64 red[JG][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6, b = blockIdx.y, n2 = nao * nao;
  const int e = blockIdx.x * 64 + lane;
  const z64* S = v.base + v.off[b] + min(e, n2 - 1);
  const double sg = v.conj[b] != 0 ? -1.0 : 1.0;
  z64 acc{0.0, 0.0};
#pragma unroll 4
  for (int Q = g; Q < NQ; Q += JG) {
    z64 x = S[(int64_t)Q * n2];
    x.y *= sg;
    acc = cfma(x, jvec[Q], acc);
  }
  red[g][lane] = acc;
  __syncthreads();
  if (g != 0 || e >= n2) return;
#pragma unroll
  for (int w = 1; w < JG; ++w) { acc.x += red[w][lane].x; acc.y += red[w][lane].y; }
  const int r = e / nao, c = e - r * nao, m = v.trans[b] != 0 ? c * nao + r : e;
  for (int s = 0; s < nj; ++s) {
    z64* p = F + ((int64_t)b * nps + s) * n2 + m;
    *p = z64{p->x + acc.x, p->y + acc.y};
  }
}

__global__ __launch_bounds__(256) void density_traces_kernel(const z64* D, const z64* F, int64_t f_k, int64_t f_s,
                                                             int n, int nk, z64* tr) {
  const int k = blockIdx.x, s = blockIdx.y, n2 = n * n;
  const z64* Dk = D + ((int64_t)s * nk + k) * n2;
  const z64* Fk = F + k * f_k + s * f_s;
  z64 acc{0.0, 0.0};
  for (int e = threadIdx.x; e < n2; e += 256) {
    const int r = e / n, c = e - r * n;
    acc = cfma(Dk[e], Fk[c * n + r], acc);
  }
  const z64 t = block_sum(acc);
  if (threadIdx.x == 0) tr[(int64_t)s * nk + k] = t;
}

// 64 elements x 8 groups of slices per workgroup.
__global__ __launch_bounds__(64 * JG) void sum_slices_kernel(const z64* in, int64_t in_bs, int64_t stride, int np,
                                                             z64* out, int64_t out_bs, int64_t n) {
  __shared__ z64 red[JG][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const z64* p = in + blockIdx.y * in_bs + (i < n ? i : n - 1);
  z64 acc{0.0, 0.0};
#pragma unroll 8
  for (int k = g; k < np; k += JG) {
    const z64 x = p[k * stride];
    acc.x += x.x;
    acc.y += x.y;
  }
  red[g][lane] = acc;
  __syncthreads();
  if (g != 0 || i >= n) return;
#pragma unroll
  for (int w = 1; w < JG; ++w) { acc.x += red[w][lane].x; acc.y += red[w][lane].y; }
  out[blockIdx.y * out_bs + i] = acc;
}

}  // namespace

void hartree_vector(const PairBlocks& v, int n, int NQ, int nao, const z64* D, int nps, int nj, double scale,
                    z64* part, hipStream_t s) {
  require(nj >= 1 && nj <= nps && (int64_t)nao * nao < ((int64_t)1 << 31), "hartree_vector: bad sizes");
  // grid.y is limited to 65535: launch the pairs in chunks
  for (int b0 = 0; b0 < n; b0 += 65535) {
    const int m = std::min(n - b0, 65535);
    PairBlocks c{v.base, v.off + b0, v.trans + b0, v.conj + b0};
    hipLaunchKernelGGL(hartree_vector_kernel, dim3(NQ, m), dim3(256), 0, s, c, NQ, nao,
                       D + (int64_t)b0 * nps * nao * nao, nps, nj, scale, part + (int64_t)b0 * NQ);
    GGPU_HIP(hipGetLastError());
  }
}

void hartree_fock(const PairBlocks& v, int n, int NQ, int nao, const z64* jvec, z64* F, int nps, int nj,
                  hipStream_t s) {
  require(nj >= 1 && nj <= nps && (int64_t)nao * nao < ((int64_t)1 << 31), "hartree_fock: bad sizes");
  const int64_t n2 = (int64_t)nao * nao;
  for (int b0 = 0; b0 < n; b0 += 65535) {
    const int m = std::min(n - b0, 65535);
    PairBlocks c{v.base, v.off + b0, v.trans + b0, v.conj + b0};
    hipLaunchKernelGGL(hartree_fock_kernel, dim3((unsigned)((n2 + 63) / 64), m), dim3(64 * JG), 0, s, c, NQ, nao, jvec,
                       F + (int64_t)b0 * nps * n2, nps, nj);
    GGPU_HIP(hipGetLastError());
  }
}

void density_traces(const z64* D, const z64* F, int64_t f_k, int64_t f_s, int n, int nsp, int nk, z64* tr,
                    hipStream_t s) {
  require((int64_t)n * n < ((int64_t)1 << 31) && nsp <= 65535, "density_traces: bad sizes");
  hipLaunchKernelGGL(density_traces_kernel, dim3(nk, nsp), dim3(256), 0, s, D, F, f_k, f_s, n, nk, tr);
  GGPU_HIP(hipGetLastError());
}

void sum_slices(const z64* in, int64_t in_bs, int64_t stride, int np, z64* out, int64_t out_bs, int64_t n, int nb,
                hipStream_t s) {
  if (n <= 0 || nb <= 0) return;
  require(np >= 0 && nb <= 65535 && (n + 63) / 64 < ((int64_t)1 << 31), "sum_slices: bad sizes");
  hipLaunchKernelGGL(sum_slices_kernel, dim3((unsigned)((n + 63) / 64), nb), dim3(64 * JG), 0, s, in, in_bs, stride,
                     np, out, out_bs, n);
  GGPU_HIP(hipGetLastError());
}

}  // namespace ggpu
