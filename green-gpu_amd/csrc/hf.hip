// Kernels of the HF exchange (FP64, small nao), the Hartree term, the Fock
// assembly and the HF energy.
//
// The reductions (Hartree vector, Fock update, traces, partial sums) are bound
// by HBM reads when the system is large and by the latency of one load chain
// when it is small, so each splits its sum over as many lanes as the sum has
// terms and reads the stored pair blocks where they lie (no unfolded copy).
// As matrix products with one row or column, and K's partial slices summed one
// after the other, they took 45 of the 181 ms of a Fock build at nk = 64,
// nao = 52, NQ = 300, ns = 2, and 1.5 of 1.85 ms at nk = 8, nao = 26, NQ = 100.
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

// ---------------------------------------------------------------------------
// Exchange: K_s(k) += f sum_{k2, Q} V^Q D_s(k2) V^Q dagger for nao <= 57
// ---------------------------------------------------------------------------
// A workgroup sums its chunk of the (k2, Q) entries of one k and one density
// block.  V^Q (double-buffered) and D_s(k2) lie in LDS, rows copied there by
// load-to-LDS straight from the stored pair, whatever its order.  Wave
// (cs, ib) owns the 16 rows i of block ib and the 16-wide blocks c of X = V D
// with c / 16 = cs mod CS:
//
//   (X^T)[c][i] = sum_a D[a][c] V[i][a],   K[i][j] += sum_c X[i][c] conj(V[j][c])
//
// The MFMA output of the first product (lane l, register r: row c = l / 16 +
// 4 r, column i = l % 16) is the A operand of the second (row i = l % 16,
// k = c = l / 16 of step r), so X never leaves the registers and K stays in
// accumulators for the whole chunk.
//
// Bound: the FP64 matrix pipe (both products with three real products per
// complex one, extents padded to 16 rows and 4 k).  V is read once per
// density block, nothing is written but the partial K of the chunk; as two
// GEMM launches per k, X went to memory and back and V was unfolded and read
// three times.  Fock builds before and after: nk = 64, nao = 52, NQ = 300,
// ns = 2 136 -> 111 ms; nk = 27 (time reversal), nao = 41 6.3 -> 4.5 ms;
// nk = 8, nao = 26 0.39 -> 0.17 ms; X2C nk = 8, nao = 30 0.71 -> 0.39 ms.
constexpr int kExMaxNao = 57;   // 3 (nao | 1) nao 16-byte elements within 160 KiB

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

struct ExchangeArgs {
  PairBlocks v;            // pair of (k group entry g, k2 = b): index g * pairs_ld + b
  int pairs_ld;
  const z64* D;            // (k2 = k2_0 + b, nps, nao, nao)
  z64* part;               // (group, slices, nps, nao, nao)
  int nao, NQ, nps;
  int npairs;              // pairs b < npairs of every k in this launch
  int per_chunk, split;    // pairs per chunk (split == 1), or split chunks per pair
  int chunk0, slices;      // first chunk of this launch; slices per k in `part`
  double scale;
};

template <int IB, int CS>
__global__ __launch_bounds__(64 * IB * CS) __attribute__((amdgpu_waves_per_eu(2))) void exchange_kernel(
    const ExchangeArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  constexpr int NW = IB * CS;
  const int nao = a.nao, n2 = nao * nao, np = nao | 1;   // odd row stride in LDS: no bank conflicts either way
  const int buf = nao * np * 16;                         // V stage 0, V stage 1, D
  const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ib = w % IB, cs = w / IB;
  const int chunk = blockIdx.x, s = blockIdx.y, g = blockIdx.z;
  int b0, b1, q0, q1;   // pairs [b0, b1), auxiliary functions [q0, q1) of each
  if (a.split > 1) {
    b0 = chunk / a.split;
    b1 = b0 + 1;
    const int j = chunk - b0 * a.split, len = (a.NQ + a.split - 1) / a.split;
    q0 = min(j * len, a.NQ);
    q1 = min(q0 + len, a.NQ);
  } else {
    b0 = chunk * a.per_chunk;
    b1 = min(b0 + a.per_chunk, a.npairs);
    q0 = 0;
    q1 = a.NQ;
  }
  const int nq = q1 - q0;

  auto copy_rows = [&](const z64* src, int8_t* dst) {
    if (lane < nao)
      for (int r = w; r < nao; r += NW)
        __builtin_amdgcn_global_load_lds((const void*)(src + r * nao + lane),
                                         (__attribute__((address_space(3))) void*)(dst + r * np * 16), 16, 0, 0);
  };
  auto wait_own = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); };
  auto barrier = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  struct Pair {
    const z64* src;   // V^{q0} of the pair
    int tr, cg;
  };
  auto pair = [&](int b) {   // uniform, into scalar registers
    const int64_t i = (int64_t)g * a.pairs_ld + b, off = a.v.off[i];
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)off), hi = __builtin_amdgcn_readfirstlane((int)(off >> 32));
    Pair p;
    p.src = a.v.base + (int64_t)(((uint64_t)hi << 32) | lo) + (int64_t)q0 * n2;
    p.tr = __builtin_amdgcn_readfirstlane(a.v.trans[i]);
    p.cg = __builtin_amdgcn_readfirstlane(a.v.conj[i]);
    return p;
  };
  auto read = [&](int byte) { return *reinterpret_cast<const v2d*>(lds + byte); };
  auto flip = [](v2d& x, uint32_t sign) {   // x.y times +-1, off the FP64 pipe
    x.y = __longlong_as_double(__double_as_longlong(x.y) ^ ((long long)sign << 32));
  };

  v4d k1[IB], k2[IB], k3[IB];
#pragma unroll
  for (int j = 0; j < IB; ++j) k1[j] = k2[j] = k3[j] = v4d{0, 0, 0, 0};
  const int full = nao / 4, left = nao - 4 * full;   // whole and partial k steps of the first product

  int stage = 0;
  Pair cur = {nullptr, 0, 0}, next = cur;
  if (nq > 0 && b1 > b0) {
    cur = pair(b0);
    copy_rows(cur.src, lds);
  } else {
    b1 = b0;
  }
  for (int b = b0; b < b1; ++b) {
    // V[r][k] is element r rs + k ks of a stage; rows past the end repeat the
    // last one and are not stored
    const int rs = cur.tr ? 16 : np * 16, ks = cur.tr ? np * 16 : 16;
    const uint32_t s1 = cur.cg ? 0x80000000u : 0u, s2 = s1 ^ 0x80000000u;   // V, conj(V)
    const int vi = min(ib * 16 + lr, nao - 1) * rs + lk * ks;
    int vj[IB];
#pragma unroll
    for (int j = 0; j < IB; ++j) vj[j] = min(j * 16 + lr, nao - 1) * rs;
    for (int q = 0; q < nq; ++q) {
      wait_own();
      barrier();   // V has landed, and every wave is done with the other stage and with D
      if (q == 0) {
        copy_rows(a.D + ((int64_t)b * a.nps + s) * n2, lds + 2 * buf);
        if (b + 1 < b1) next = pair(b + 1);
        wait_own();
        barrier();
      }
      if (q + 1 < nq) copy_rows(cur.src + (int64_t)(q + 1) * n2, lds + (stage ^ 1) * buf);
      else if (b + 1 < b1) copy_rows(next.src, lds + (stage ^ 1) * buf);
      const int sV = stage * buf;
      stage ^= 1;
#pragma unroll
      for (int cc = 0; cc < (IB + CS - 1) / CS; ++cc) {
        const int c0 = (cs + cc * CS) * 16;
        if (c0 >= nao) break;
        v4d x1 = {0, 0, 0, 0}, x2 = {0, 0, 0, 0}, x3 = {0, 0, 0, 0};
        int pd = 2 * buf + (lk * np + min(c0 + lr, nao - 1)) * 16, pv = sV + vi;
        auto step = [&](v2d d, v2d v) {
          flip(v, s1);
          x1 = __builtin_amdgcn_mfma_f64_16x16x4f64(d.x, v.x, x1, 0, 0, 0);
          x2 = __builtin_amdgcn_mfma_f64_16x16x4f64(d.y, v.y, x2, 0, 0, 0);
          x3 = __builtin_amdgcn_mfma_f64_16x16x4f64(d.x + d.y, v.x + v.y, x3, 0, 0, 0);
        };
        // whole steps in groups of four: eight reads in flight, twelve MFMAs
        int t = 0;
        for (; t + 4 <= full; t += 4) {
          v2d d[4], v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            d[u] = read(pd);
            v[u] = read(pv);
            pd += 64 * np;
            pv += 4 * ks;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) step(d[u], v[u]);
        }
        for (; t < full; ++t) {
          step(read(pd), read(pv));
          pd += 64 * np;
          pv += 4 * ks;
        }
        if (left > 0) {   // the lanes past the end of k read the last one and drop it
          const int over = max(lk - (left - 1), 0);
          v2d d = read(pd - over * np * 16), v = read(pv - over * ks);
          if (over) d = v = v2d{0.0, 0.0};
          step(d, v);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (c0 + 4 * r >= nao) break;
          const int c = c0 + 4 * r + lk, pk = sV + min(c, nao - 1) * ks;
          const bool out = c >= nao;
          const double xr = out ? 0.0 : x1[r] - x2[r], xi = out ? 0.0 : x3[r] - x1[r] - x2[r], xs = xr + xi;
          v2d v[IB];
#pragma unroll
          for (int j = 0; j < IB; ++j) v[j] = read(pk + vj[j]);
#pragma unroll
          for (int j = 0; j < IB; ++j) {
            flip(v[j], s2);
            if (out) v[j] = v2d{0.0, 0.0};
            k1[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xr, v[j].x, k1[j], 0, 0, 0);
            k2[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi, v[j].y, k2[j], 0, 0, 0);
            k3[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, v[j].x + v[j].y, k3[j], 0, 0, 0);
          }
        }
      }
    }
    cur = next;
  }
  z64* out = a.part + (((int64_t)g * a.slices + (int64_t)(a.chunk0 + chunk) * CS + cs) * a.nps + s) * n2;
#pragma unroll
  for (int j = 0; j < IB; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = ib * 16 + lk + 4 * r, col = j * 16 + lr;
      if (row < nao && col < nao)
        out[row * nao + col] =
            z64{a.scale * (k1[j][r] - k2[j][r]), a.scale * (k3[j][r] - k1[j][r] - k2[j][r])};
    }
}

template <int IB, int CS>
void exchange_launch(const ExchangeArgs& a, dim3 grid, hipStream_t s) {
  const size_t bytes = (size_t)3 * a.nao * (a.nao | 1) * 16;
  const void* f = reinterpret_cast<const void*>(&exchange_kernel<IB, CS>);
  GGPU_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  hipLaunchKernelGGL((exchange_kernel<IB, CS>), grid, dim3(64 * IB * CS), bytes, s, a);
  GGPU_HIP(hipGetLastError());
}

// c-split of the waves for each number of 16-row blocks: enough waves for two
// per SIMD where one workgroup fills the LDS of a CU.
int exchange_csplit(int nao) {
  const int ib = (nao + 15) / 16;
  return ib == 1 ? 1 : ib == 3 ? 3 : 2;
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

bool exchange_fits(int nao) { return nao <= kExMaxNao; }

ExchangePlan exchange_plan(int nao, int NQ, int nps, int nk, int ink, int kb) {
  ExchangePlan p;
  // workgroups a CU holds at once by LDS and by registers
  static const int by_registers[5] = {0, 16, 4, 1, 1};
  const int64_t lds = (int64_t)3 * nao * (nao | 1) * 16;
  const int occ = (int)std::max<int64_t>(1, std::min<int64_t>((160 << 10) / lds, by_registers[(nao + 15) / 16]));
  // chunks per k: three rounds of workgroups over the 256 CUs when every k is
  // in the launch, and at least 32 so that a rank's share of the k fills the
  // chip too.  A chunk is whole pairs, or a part of one pair with four
  // auxiliary functions or more, whatever the share and the residence: the
  // sums are the same in all.
  const int64_t want = std::max<int64_t>(32, (3LL * 256 * occ + (int64_t)nps * ink - 1) / ((int64_t)nps * ink));
  if (want > nk) {
    p.split = (int)std::max<int64_t>(1, std::min<int64_t>((want + nk - 1) / nk, NQ / 4));
    p.per_chunk = 1;
  } else {
    p.split = 1;
    p.per_chunk = std::max(1, std::min((int)(nk / want), kb));
  }
  p.chunks = p.split > 1 ? nk * p.split : (nk + p.per_chunk - 1) / p.per_chunk;
  p.slices = p.chunks * exchange_csplit(nao);
  return p;
}

void exchange_f64(const ExchangePlan& p, const PairBlocks& v, int pairs_ld, int ngroup, int b0, int npairs, int nao,
                  int NQ, const z64* D, int nps, double scale, z64* part, hipStream_t s) {
  require(exchange_fits(nao) && b0 % p.per_chunk == 0 && ngroup >= 1 && npairs >= 1, "exchange: bad launch");
  ExchangeArgs a;
  a.v = v;
  a.pairs_ld = pairs_ld;
  a.D = D + (int64_t)b0 * nps * nao * nao;
  a.part = part;
  a.nao = nao; a.NQ = NQ; a.nps = nps;
  a.npairs = npairs;
  a.per_chunk = p.per_chunk; a.split = p.split;
  a.chunk0 = p.split > 1 ? b0 * p.split : b0 / p.per_chunk;
  a.slices = p.slices;
  a.scale = scale;
  const int chunks = p.split > 1 ? npairs * p.split : (npairs + p.per_chunk - 1) / p.per_chunk;
  require(ngroup <= 65535 && nps <= 65535, "exchange: grid too large");
  const dim3 grid(chunks, nps, ngroup);
  switch ((nao + 15) / 16) {
    case 1: return exchange_launch<1, 1>(a, grid, s);
    case 2: return exchange_launch<2, 2>(a, grid, s);
    case 3: return exchange_launch<3, 3>(a, grid, s);
    default: return exchange_launch<4, 2>(a, grid, s);
  }
}

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
