// FP64 batched complex GEMM on v_mfma_f64_16x16x4_f64.
//
// A workgroup of WM x WN waves computes a (16 WM MB) x (16 WN NB) tile of C,
// each wave MB x NB blocks of the 16 x 16 MFMA output, with the 3-product
// (Gauss) complex scheme: t1 = ar br, t2 = ai bi, t3 = (ar + ai)(br + bi);
// re = t1 - t2, im = t3 - t1 - t2.
//
// What bounds it: the FP64 matrix pipe (78 TFLOP/s of real products measured
// on registers alone, 74 with the two sums per fragment that share the FP64
// pipe; x 4/3 for the Gauss scheme: 99 TFLOP/s of complex products), so every
// cycle that a wave spends waiting for operands and every padded row counts:
//
// * Operands go HBM -> LDS by load-to-LDS copies of 16 bytes (one complex
//   element) per lane, two stages of 8 k each: no staging registers, no
//   address arithmetic beyond one 32-bit offset per copy, and a whole k tile
//   of MFMAs between issue and use.  (Staged through registers instead, one
//   k tile ahead: 71 against 84-87 TFLOP/s at M = 600, N = 10816, K = 600.)
//   The stages are bytes to the compiler: of a typed array it believes that
//   every read may touch the copy in flight and waits for it.
// * An LDS slot is one element; reading a fragment is one conflict-free
//   ds_read_b128 per lane.  Row-contiguous operands: 16 rows x 4 k per copy,
//   in fragment order.  k-contiguous operands: 8 rows x 8 k per copy (whole
//   128-byte lines), k exchanged by the low row bits so that the 8 lanes a
//   read serves at a time fall into different banks.
// * Conjugation is a sign in the sums and in the epilogue.
// * Edge tiles read clamped rows (never stored) and clamped k; the wave that
//   copied a k past the end overwrites it with zero before the barrier.
// * Small wave tiles (3 to 6 waves per SIMD) beat large ones at the same
//   padding: 128 x 64 with two waves per SIMD gains nothing at the largest
//   shapes, so the menu of tiles is there for padding and for filling the
//   chip (choose_tile).
#include "tiling.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace ggpu {
namespace {

constexpr int BK = 8;        // k per LDS stage
constexpr int KG = BK / 4;   // MFMA k steps per stage

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

// Waits for this wave's copies and LDS accesses.
__device__ inline void wait_own() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

// AKC / BKC: the operand's k index is copied as the contiguous one (a matter
// of speed only).  WIDE: 64-bit element offsets within a tile.  WPE: waves per
// SIMD the registers must allow.
template <int WM, int WN, int MB, int NB, int WPE, bool AKC, bool BKC, int SITE, bool WIDE = false>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm_f64_kernel(
    const GemmDesc d) {
  using Off = std::conditional_t<WIDE, int64_t, uint32_t>;
  constexpr int TM = 16 * WM * MB, TN = 16 * WN * NB, NW = WM * WN;
  constexpr int FA = TM / 16 * KG, FB = TN / 16 * KG;               // 1 KiB slots groups per stage
  constexpr int LA = (FA + NW - 1) / NW, LB = (FB + NW - 1) / NW;   // copies per wave
  constexpr int STAGE = (FA + FB) * 1024;
  __shared__ __attribute__((aligned(1024))) int8_t lds[2 * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TileCoord tc = tile_coord(d, (d.M + TM - 1) / TM, (d.N + TN - 1) / TN);
  const int m0 = tc.mt * TM, n0 = tc.nt * TN;
  const z64* A = static_cast<const z64*>(d.A.ptr) + tc.b0 * d.A.bs0 +
                 (d.A.off1 ? d.A.off1[tc.b1] : tc.b1 * d.A.bs1) + (int64_t)m0 * d.A.rs;
  const z64* B = static_cast<const z64*>(d.B.ptr) + tc.b0 * d.B.bs0 +
                 (d.B.off1 ? d.B.off1[tc.b1] : tc.b1 * d.B.bs1) + (int64_t)n0 * d.B.cs;
  z64* C = static_cast<z64*>(d.C.ptr) + tc.b0 * d.C.bs0 + (d.C.off1 ? d.C.off1[tc.b1] : tc.b1 * d.C.bs1);

  // Copy j of this wave fills the slot group f = min(w + NW j, F - 1) (waves
  // without a group of their own repeat the last one): row and k of a lane.
  auto group = [&](int j, int F) { return min(w + NW * j, F - 1); };
  auto slot_row = [&](int f, bool kc) { return kc ? f * (64 / BK) + lane / BK : (f / KG) * 16 + (lane & 15); };
  auto slot_k = [&](int f, bool kc) {
    return kc ? (lane % BK) ^ (slot_row(f, true) & 7) : (f % KG) * 4 + (lane >> 4);
  };
  const Off a_rs = (Off)(d.A.rs * 16), a_ks = (Off)(d.A.cs * 16), b_rs = (Off)(d.B.cs * 16),
            b_ks = (Off)(d.B.rs * 16);
  Off av[LA], bv[LB];   // byte offset of the lane's element in a full k tile
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int f = group(j, FA);
    av[j] = (Off)min(slot_row(f, AKC), d.M - 1 - m0) * a_rs + (Off)slot_k(f, AKC) * a_ks;
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int f = group(j, FB);
    bv[j] = (Off)min(slot_row(f, BKC), d.N - 1 - n0) * b_rs + (Off)slot_k(f, BKC) * b_ks;
  }
  const char *Ab = reinterpret_cast<const char*>(A), *Bb = reinterpret_cast<const char*>(B);   // of a K-batch entry
  const int64_t a_kb = d.A.kbs * 16, b_kb = d.B.kbs * 16, a_kt = d.A.cs * (16 * BK), b_kt = d.B.rs * (16 * BK);
  const int nkb = d.kb_total > 0 ? min(d.KB, d.kb_total - (int)tc.b0 * d.KB) : d.KB;
  const int ktiles = (d.K + BK - 1) / BK, niter = nkb * ktiles;
  const int tail = d.K - (ktiles - 1) * BK;   // k extent of a K-batch entry's last tile
  const char *pa = Ab, *pb = Bb;
  int ikt = 0;                                // tile (pa, pb) point at
  auto issue = [&](int st) {
    int8_t* dst = lds + st * STAGE;
    const int rem = ikt + 1 == ktiles ? tail : BK;
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int f = group(j, FA);
      Off o = av[j];
      if (rem < BK) o -= (Off)max(slot_k(f, AKC) - (rem - 1), 0) * a_ks;   // clamp k
      __builtin_amdgcn_global_load_lds((const void*)(pa + o), (__attribute__((address_space(3))) void*)(dst + f * 1024),
                                       16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int f = group(j, FB);
      Off o = bv[j];
      if (rem < BK) o -= (Off)max(slot_k(f, BKC) - (rem - 1), 0) * b_ks;
      __builtin_amdgcn_global_load_lds((const void*)(pb + o),
                                       (__attribute__((address_space(3))) void*)(dst + (FA + f) * 1024), 16, 0, 0);
    }
    pa += a_kt;
    pb += b_kt;
    if (++ikt == ktiles) {
      ikt = 0;
      pa = Ab += a_kb;
      pb = Bb += b_kb;
    }
  };
  // zero the k past the end of K in what this wave copied
  auto clear_tail = [&](int st) {
    int8_t* dst = lds + st * STAGE + 16 * lane;
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      const int f = group(j, FA);
      if (slot_k(f, AKC) >= tail) *reinterpret_cast<v2d*>(dst + f * 1024) = v2d{0.0, 0.0};
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int f = group(j, FB);
      if (slot_k(f, BKC) >= tail) *reinterpret_cast<v2d*>(dst + (FA + f) * 1024) = v2d{0.0, 0.0};
    }
  };

  const int wm = (w / WN) * MB, wn = (w % WN) * NB;   // the wave's first 16-row block of A / B
  const int lr = lane & 15, lk = lane >> 4;
  const double sA = d.A.conj ? -1.0 : 1.0, sB = d.B.conj ? -1.0 : 1.0;
  v4d acc[3][MB][NB];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[a][i][j] = v4d{0, 0, 0, 0};
  auto frag = [&](const int8_t* base, bool kc, int rb, int g) {
    return *reinterpret_cast<const v2d*>(
        base + (kc ? ((rb * 16 + lr) * BK + ((4 * g + lk) ^ (lr & 7))) * 16 : (rb * KG + g) * 1024 + 16 * lane));
  };
  auto kstep = [&](int st, int g) {
    const int8_t *pA = lds + st * STAGE, *pB = pA + FA * 1024;
    v2d a[MB], b[NB];
    double as[MB], bs[NB];
#pragma unroll
    for (int i = 0; i < MB; ++i) a[i] = frag(pA, AKC, wm + i, g);
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = frag(pB, BKC, wn + j, g);
#pragma unroll
    for (int i = 0; i < MB; ++i) as[i] = __builtin_fma(sA, a[i].y, a[i].x);
#pragma unroll
    for (int j = 0; j < NB; ++j) bs[j] = __builtin_fma(sB, b[j].y, b[j].x);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, acc[0][i][j], 0, 0, 0);
        acc[1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].y, acc[1][i][j], 0, 0, 0);
        acc[2][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], acc[2][i][j], 0, 0, 0);
      }
  };

  if (niter > 0) issue(0);
  int kt = 0;
  for (int it = 0; it < niter; ++it) {
    const int rem = kt + 1 == ktiles ? tail : BK;
    wait_own();
    if (rem < BK) {
      clear_tail(it & 1);
      wait_own();
    }
    // this tile has landed for every wave, and every wave is done with the
    // stage that the next copies overwrite
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (it + 1 < niter) issue((it & 1) ^ 1);
#pragma unroll
    for (int g = 0; g < KG; ++g)
      if (g == 0 || 4 * g < rem) kstep(it & 1, g);   // uniform: skip steps past the end of K
    if (++kt == ktiles) kt = 0;
  }

  // v_mfma_f64_16x16x4_f64 (measured on gfx950): lane l, register r holds row
  // l / 16 + 4 r, column l % 16
  const bool use_beta = (d.beta_re != 0.0 || d.beta_im != 0.0);
  const double s2 = sA * sB;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + (wm + i) * 16 + lk + 4 * r;
        const int col = n0 + (wn + j) * 16 + lr;
        if (row < d.M && col < d.N) {
          const double t1 = acc[0][i][j][r], t2 = s2 * acc[1][i][j][r], t3 = acc[2][i][j][r];
          const double xr = t1 - t2, xi = t3 - t1 - t2;
          double vr = d.alpha_re * xr - d.alpha_im * xi;
          double vi = d.alpha_re * xi + d.alpha_im * xr;
          z64* p = C + row * d.C.rs + col * d.C.cs;
          if (use_beta) {
            const z64 o = *p;
            vr += d.beta_re * o.x - d.beta_im * o.y;
            vi += d.beta_re * o.y + d.beta_im * o.x;
          }
          *p = z64{vr, vi};
        }
      }
}

// The menu of workgroup tiles: rows, columns, waves per SIMD that the
// registers (24 accumulator registers per 16 x 16 block and wave) and LDS
// leave, and the tile's own time per area against the others'.  All give the
// same sums.
enum Tile { k64x64, k48x64, k64x32, k64x48, k64x80, k64x96, k64x112, k80x64, k32x64, k64x16, k32x32, kTiles };
struct TileShape { int m, n, waves; double time; };
constexpr TileShape kTileShape[kTiles] = {
    {64, 64, 3, 0.95}, {48, 64, 4, 1.0},  {64, 32, 5, 0.95}, {64, 48, 4, 1.05}, {64, 80, 3, 1.0}, {64, 96, 2, 1.0},
    {64, 112, 2, 1.0}, {80, 64, 3, 1.0}, {32, 64, 5, 0.95}, {64, 16, 6, 1.1},  {32, 32, 6, 1.0}};

// Expected time of a launch in units of matrix-pipe work per CU: the padded
// tile area each of the 256 CUs gets through (whole rounds while the grid
// fills the chip only a few times), slower by 1 + 0.3 / n with n waves per
// SIMD to hide latencies, plus the tile's operand traffic (rows + columns).
// Fitted to 60 shapes of the HF / GW contractions (nao 10 to 104, NQ 64 to
// 600) timed with every tile: the choice is within 1 % of the fastest tile on
// (geometric) average over all sites.  At sig_contract alone (four entries, NQ =
// 4 nao, nts = 62) it is within 3 % at nao = 64, 75, 80, but takes 64 x 16 at
// nao = 41, 100 and 104 and then has 34, 37, 45 TFLOP/s where 64 x 48 or 64 x 112
// have 48, 51, 55.  Against a 64 x 64 tile everywhere it is 1.3 - 2.2x
// faster where an extent is just above a multiple of 64 (nao = 72: p0_gvh
// 46 -> 69 TFLOP/s) or the grid is small (nao = 26, NQ = 100: p0_contract
// 20 -> 33, sig_vg 20 -> 36).
double tile_cost(const GemmDesc& d, const TileShape& t) {
  const double tiles = (double)((d.M + t.m - 1) / t.m) * ((d.N + t.n - 1) / t.n) * d.nb0 * d.nb1;
  double rounds = tiles / 256.0;
  if (rounds <= 8.0 * t.waves) rounds = std::ceil(rounds);
  const double n = std::min<double>(t.waves, std::max(1.0, std::ceil(tiles / 256.0)));
  return t.time * rounds * ((double)t.m * t.n * (1.0 + 0.3 / n) + 3.0 * (t.m + t.n));
}

Tile choose_tile(const GemmDesc& d) {
  int best = 0;
  double cost = 0;
  for (int t = 0; t < kTiles; ++t) {
    const double c = tile_cost(d, kTileShape[t]);
    if (t == 0 || c < cost) { best = t; cost = c; }
  }
  return (Tile)best;
}

template <int WM, int WN, int MB, int NB, int WPE, bool AKC, bool BKC, int SITE, bool WIDE = false>
void launch_one(const GemmDesc& d, hipStream_t stream) {
  constexpr int TM = 16 * WM * MB, TN = 16 * WN * NB;
  const int64_t tiles = (int64_t)((d.M + TM - 1) / TM) * ((d.N + TN - 1) / TN);
  const int64_t total = tiles * d.nb0 * d.nb1;
  require(total < (int64_t)1 << 31, "gemm: grid too large");
  hipLaunchKernelGGL((gemm_f64_kernel<WM, WN, MB, NB, WPE, AKC, BKC, SITE, WIDE>), dim3((unsigned)total),
                     dim3(64 * WM * WN), 0, stream, d);
  GGPU_HIP(hipGetLastError());
}

template <bool AKC, bool BKC, int SITE>
void launch_tile(const GemmDesc& d, hipStream_t stream, Tile t) {
  switch (t) {
    case k48x64: return launch_one<1, 4, 3, 1, 4, AKC, BKC, SITE>(d, stream);
    case k64x32: return launch_one<2, 2, 2, 1, 5, AKC, BKC, SITE>(d, stream);
    case k64x48: return launch_one<4, 1, 1, 3, 4, AKC, BKC, SITE>(d, stream);
    case k64x80: return launch_one<4, 1, 1, 5, 3, AKC, BKC, SITE>(d, stream);
    case k64x96: return launch_one<4, 1, 1, 6, 2, AKC, BKC, SITE>(d, stream);
    case k64x112: return launch_one<4, 1, 1, 7, 2, AKC, BKC, SITE>(d, stream);
    case k80x64: return launch_one<1, 4, 5, 1, 3, AKC, BKC, SITE>(d, stream);
    case k32x64: return launch_one<1, 4, 2, 1, 5, AKC, BKC, SITE>(d, stream);
    case k64x16: return launch_one<4, 1, 1, 1, 6, AKC, BKC, SITE>(d, stream);
    case k32x32: return launch_one<2, 2, 1, 1, 6, AKC, BKC, SITE>(d, stream);
    default: return launch_one<2, 2, 2, 2, 3, AKC, BKC, SITE>(d, stream);
  }
}

}  // namespace

void launch_f64(const GemmDesc& d, hipStream_t stream, int variant) {
  const bool akc = (d.A.cs == 1) || (d.A.rs != 1), bkc = (d.B.rs == 1) || (d.B.cs != 1);
  // lane offsets within a tile are 32 bits wide: at most 112 rows and 8 k
  auto span = [](int64_t rs, int64_t ks) { return 16.0 * (112.0 * (double)std::abs(rs) + BK * (double)std::abs(ks)); };
  const bool wide = d.A.rs < 0 || d.A.cs < 0 || d.B.rs < 0 || d.B.cs < 0 || span(d.A.rs, d.A.cs) >= 4294967296.0 ||
                    span(d.B.cs, d.B.rs) >= 4294967296.0;
  if (wide) {
    if (akc && bkc) return launch_one<2, 2, 2, 2, 2, true, true, kSiteOther, true>(d, stream);
    if (akc) return launch_one<2, 2, 2, 2, 2, true, false, kSiteOther, true>(d, stream);
    if (bkc) return launch_one<2, 2, 2, 2, 2, false, true, kSiteOther, true>(d, stream);
    return launch_one<2, 2, 2, 2, 2, false, false, kSiteOther, true>(d, stream);
  }
  const Tile t = variant == 8 ? k64x64 : variant == 16 ? k48x64 : choose_tile(d);
  // each contraction site has its own symbol, compiled for its one layout
  switch (d.site) {
    case kSiteP0X1: return launch_tile<true, false, kSiteP0X1>(d, stream, t);
    case kSiteP0X2: return launch_tile<true, true, kSiteP0X2>(d, stream, t);
    case kSiteP0: return launch_tile<false, true, kSiteP0>(d, stream, t);
    case kSiteSigY1: return launch_tile<true, false, kSiteSigY1>(d, stream, t);
    case kSiteSigY2: return launch_tile<false, false, kSiteSigY2>(d, stream, t);
    case kSiteSigma: return launch_tile<true, true, kSiteSigma>(d, stream, t);
    default: break;
  }
  if (akc && bkc) return launch_tile<true, true, kSiteOther>(d, stream, t);
  if (akc) return launch_tile<true, false, kSiteOther>(d, stream, t);
  if (bkc) return launch_tile<false, true, kSiteOther>(d, stream, t);
  return launch_tile<false, false, kSiteOther>(d, stream, t);
}

}  // namespace ggpu
