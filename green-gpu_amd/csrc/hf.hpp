// Kernels of the HF exchange (FP64), the Hartree term, the Fock assembly and the
// HF energy (hf.hip).
#pragma once

#include "common.hpp"

namespace ggpu {

// Stored pairs as a kernel reads them: the block of pair b starts at
// base + off[b] (NQ x nao x nao) and is transposed / conjugated per Q where
// trans[b] / conj[b] say so.
struct PairBlocks {
  const z64* base = nullptr;
  const int64_t* off = nullptr;   // device, one entry per pair
  const int* trans = nullptr;     // device
  const int* conj = nullptr;      // device
};

// The fused FP64 exchange (nao that fits LDS): K_s(k) as `slices` partial
// matrices, each summed over one chunk of the (k2, Q) entries.
bool exchange_fits(int nao);
struct ExchangePlan {
  int per_chunk = 1;   // pairs per chunk (split == 1)
  int split = 1;       // chunks per pair
  int chunks = 0;      // of one k
  int slices = 0;      // partial matrices of one k and density block
};
// kb: pairs a staged batch may hold (chunks never span batches of whole chunks).
ExchangePlan exchange_plan(int nao, int NQ, int nps, int nk, int ink, int kb);
// The chunks of pairs [b0, b0 + npairs) of `ngroup` k: pair b0 + b of group
// entry g is v's entry g * pairs_ld + b.  b0 is a multiple of p.per_chunk, and
// so is npairs unless the pairs end there.  D: (nk, nps, nao, nao);
// part: (ngroup, p.slices, nps, nao, nao).
void exchange_f64(const ExchangePlan& p, const PairBlocks& v, int pairs_ld, int ngroup, int b0, int npairs, int nao,
                  int NQ, const z64* D, int nps, double scale, z64* part, hipStream_t s);

// part[b * NQ + Q] = scale sum_{a,c} V_b^Q[a][c] sum_{s < nj} D[b][s][c][a]
// for the n pairs b; D: (n, nps, nao, nao).
void hartree_vector(const PairBlocks& v, int n, int NQ, int nao, const z64* D, int nps, int nj, double scale,
                    z64* part, hipStream_t s);

// F[b][s] += sum_Q jvec[Q] V_b^Q for every pair b < n and block s < nj; F: (n, nps, nao, nao).
void hartree_fock(const PairBlocks& v, int n, int NQ, int nao, const z64* jvec, z64* F, int nps, int nj,
                  hipStream_t s);

// tr[s * nk + k] = sum_{a,b} D[s][k][a][b] F[k f_k + s f_s][b][a]; D: (nsp, nk, n, n),
// f_k, f_s in elements.
void density_traces(const z64* D, const z64* F, int64_t f_k, int64_t f_s, int n, int nsp, int nk, z64* tr,
                    hipStream_t s);

// out[b * out_bs + i] = sum_p in[b * in_bs + p * stride + i] for i < n, b < nb.
void sum_slices(const z64* in, int64_t in_bs, int64_t stride, int np, z64* out, int64_t out_bs, int64_t n, int nb,
                hipStream_t s);

}  // namespace ggpu
