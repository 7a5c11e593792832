// Kernels of the Hartree term, the Fock assembly and the HF energy (hf.hip).
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
