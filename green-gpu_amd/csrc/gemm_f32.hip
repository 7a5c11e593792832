// FP32 batched complex GEMM on v_mfma_f32_16x16x4_f32.
//
// A workgroup of WM x WN waves computes a (16 WM MB) x (16 WN NB) tile of C,
// each wave MB x NB blocks of the 16 x 16 MFMA output with separate real and
// imaginary accumulators, 4 real products per complex one:
// re += ar br - ai bi, im += ar bi + ai br.
//
// What bounds it: the FP32 matrix pipe (157 TFLOP/s at 2.4 GHz; one complex block
// and k step of 4 holds it for 128 cycles), and in the small shapes padding and
// idle CUs, so the tile follows the shape (choose_tile).
//
// * Complex elements stay interleaved in LDS, [k][row]: a fragment is one
//   ds_read_b64 per lane.
// * Two stages of 8 k, the next one loaded into registers while this one is
//   multiplied.  The loader has nothing per element but the load: a 32-bit offset per
//   element and one uniform pointer per stage; rows past the edge are clamped
//   (never stored), k past the end clamped in an entry's last stage only, and
//   zeroed there before they reach LDS.  With bounds and 64-bit addresses for
//   each element and 64 x 64 tiles throughout it took, TFLOP/s then -> now:
//   nao = 104, NQ = 600 sig_py 106 -> 124, p0_contract 99 -> 115, sig_vg 85 ->
//   107; nao = 41, NQ = 177 sig_py 89 -> 97, sig_contract 30 -> 45, p0_gvh 46 ->
//   61.
#include "tiling.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace ggpu {
namespace {

constexpr int BK = 8;        // k per LDS stage

typedef float v4f __attribute__((ext_vector_type(4)));

// Row stride of an LDS stage in elements.  Operands written with 8 consecutive
// k per 8 lanes: 4 elements (8 banks) between the k; written along the rows:
// half the banks between the k, so that the four k of a fragment read meet in
// no bank.
constexpr int lds_stride(int rows, bool kc) { return kc ? rows + 4 : rows + (48 - rows % 32) % 32; }

// TO: complex element type of C.  AKC / BKC: the operand's k index is loaded as
// the contiguous one (a matter of speed only).  WIDE: 64-bit offsets within a
// tile.  WPE: waves per SIMD that the registers must allow.
template <class TO, int WM, int WN, int MB, int NB, int WPE, bool AKC, bool BKC, int SITE, bool WIDE = false>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WPE))) void gemm_f32_kernel(
    const GemmDesc d) {
  using Off = std::conditional_t<WIDE, int64_t, uint32_t>;
  constexpr int TM = 16 * WM * MB, TN = 16 * WN * NB, NT = 64 * WM * WN;
  constexpr int SA = lds_stride(TM, AKC), SB = lds_stride(TN, BKC);
  constexpr int EA = (TM * BK + NT - 1) / NT, EB = (TN * BK + NT - 1) / NT;   // elements per thread and stage
  __shared__ __attribute__((aligned(16))) c32 sA[2][BK][SA];
  __shared__ __attribute__((aligned(16))) c32 sB[2][BK][SB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TileCoord tc = tile_coord(d, (d.M + TM - 1) / TM, (d.N + TN - 1) / TN);
  const int m0 = tc.mt * TM, n0 = tc.nt * TN;
  const c32* A = static_cast<const c32*>(d.A.ptr) + tc.b0 * d.A.bs0 +
                 (d.A.off1 ? d.A.off1[tc.b1] : tc.b1 * d.A.bs1) + (int64_t)m0 * d.A.rs;
  const c32* B = static_cast<const c32*>(d.B.ptr) + tc.b0 * d.B.bs0 +
                 (d.B.off1 ? d.B.off1[tc.b1] : tc.b1 * d.B.bs1) + (int64_t)n0 * d.B.cs;
  TO* C = static_cast<TO*>(d.C.ptr) + tc.b0 * d.C.bs0 + (d.C.off1 ? d.C.off1[tc.b1] : tc.b1 * d.C.bs1);

  // Element j of a thread: its row and k in the stage, its byte offset and that
  // of its row.  Threads past the end of the tile repeat an element of theirs.
  const Off a_rs = (Off)(d.A.rs * 8), a_ks = (Off)(d.A.cs * 8), b_rs = (Off)(d.B.cs * 8), b_ks = (Off)(d.B.rs * 8);
  auto index = [&](int j, int rows) { return tid + j * NT < rows * BK ? tid + j * NT : tid % (rows * BK); };
  int ar[EA], ak[EA], br[EB], bk[EB];
  Off ao[EA], a0[EA], bo[EB], b0[EB];
#pragma unroll
  for (int j = 0; j < EA; ++j) {
    const int e = index(j, TM);
    ar[j] = AKC ? e / BK : e % TM;
    ak[j] = AKC ? e % BK : e / TM;
    a0[j] = (Off)min(ar[j], d.M - 1 - m0) * a_rs;
    ao[j] = a0[j] + (Off)ak[j] * a_ks;
  }
#pragma unroll
  for (int j = 0; j < EB; ++j) {
    const int e = index(j, TN);
    br[j] = BKC ? e / BK : e % TN;
    bk[j] = BKC ? e % BK : e / TN;
    b0[j] = (Off)min(br[j], d.N - 1 - n0) * b_rs;
    bo[j] = b0[j] + (Off)bk[j] * b_ks;
  }
  const char *Ab = reinterpret_cast<const char*>(A), *Bb = reinterpret_cast<const char*>(B);   // of a K-batch entry
  const int64_t a_kb = d.A.kbs * 8, b_kb = d.B.kbs * 8, a_kt = d.A.cs * (8 * BK), b_kt = d.B.rs * (8 * BK);
  const int ktiles = (d.K + BK - 1) / BK, niter = d.KB * ktiles;
  const int tail = d.K - (ktiles - 1) * BK;   // k extent of a K-batch entry's last stage
  const char *pa = Ab, *pb = Bb;
  int ikt = 0;                                // stage (pa, pb) point at
  c32 xa[EA], xb[EB];
  auto gload = [&]() {
    const int rem = ikt + 1 == ktiles ? tail : BK;
#pragma unroll
    for (int j = 0; j < EA; ++j) xa[j] = *reinterpret_cast<const c32*>(pa + (ak[j] < rem ? ao[j] : a0[j]));
#pragma unroll
    for (int j = 0; j < EB; ++j) xb[j] = *reinterpret_cast<const c32*>(pb + (bk[j] < rem ? bo[j] : b0[j]));
    pa += a_kt;
    pb += b_kt;
    if (++ikt == ktiles) {
      ikt = 0;
      pa = Ab += a_kb;
      pb = Bb += b_kb;
    }
  };
  const uint32_t cA = d.A.conj ? 0x80000000u : 0u, cB = d.B.conj ? 0x80000000u : 0u;
  auto sstore = [&](int st, int rem) {
#pragma unroll
    for (int j = 0; j < EA; ++j) {
      const bool in = ak[j] < rem;
      sA[st][ak[j]][ar[j]] = c32{in ? xa[j].x : 0.f, in ? __uint_as_float(__float_as_uint(xa[j].y) ^ cA) : 0.f};
    }
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const bool in = bk[j] < rem;
      sB[st][bk[j]][br[j]] = c32{in ? xb[j].x : 0.f, in ? __uint_as_float(__float_as_uint(xb[j].y) ^ cB) : 0.f};
    }
  };

  const int wm = (w / WN) * (16 * MB), wn = (w % WN) * (16 * NB);
  const int lr = lane & 15, lk = lane >> 4;
  v4f acc[2][MB][NB];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[a][i][j] = v4f{0, 0, 0, 0};
  auto kstep = [&](int st, int kk) {
    c32 a[MB], b[NB];
    float nai[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) a[i] = sA[st][kk + lk][wm + 16 * i + lr];
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = sB[st][kk + lk][wn + 16 * j + lr];
#pragma unroll
    for (int i = 0; i < MB; ++i) nai[i] = -a[i].y;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[j].x, acc[0][i][j], 0, 0, 0);
        acc[1][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[j].y, acc[1][i][j], 0, 0, 0);
        acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(nai[i], b[j].y, acc[0][i][j], 0, 0, 0);
        acc[1][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[j].x, acc[1][i][j], 0, 0, 0);
      }
  };

  int skt = 0;                                // stage that the registers hold
  auto next_rem = [&]() {
    const int rem = skt + 1 == ktiles ? tail : BK;
    if (++skt == ktiles) skt = 0;
    return rem;
  };
  int rem = BK;
  if (niter > 0) {
    gload();
    rem = next_rem();
    sstore(0, rem);
  }
  __syncthreads();
  for (int it = 0; it < niter; ++it) {
    const int cur = rem;
    if (it + 1 < niter) gload();
    kstep(it & 1, 0);
    if (cur > 4) kstep(it & 1, 4);   // uniform: skip a step past the end of K
    if (it + 1 < niter) {
      rem = next_rem();
      sstore((it & 1) ^ 1, rem);
    }
    __syncthreads();
  }

  // v_mfma_f32_16x16x4_f32 (measured on gfx950): lane l, register r holds row
  // 4 (l / 16) + r, column l % 16
  const bool use_beta = (d.beta_re != 0.0 || d.beta_im != 0.0);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm + 16 * i + 4 * lk + r;
        const int col = n0 + wn + 16 * j + lr;
        if (row < d.M && col < d.N) {
          const double xr = acc[0][i][j][r], xi = acc[1][i][j][r];
          double vr = d.alpha_re * xr - d.alpha_im * xi;
          double vi = d.alpha_re * xi + d.alpha_im * xr;
          TO* p = C + row * d.C.rs + col * d.C.cs;
          if (use_beta) {
            const TO o = *p;
            vr += d.beta_re * o.x - d.beta_im * o.y;
            vi += d.beta_re * o.y + d.beta_im * o.x;
          }
          using TS = decltype(TO{}.x);
          *p = TO{static_cast<TS>(vr), static_cast<TS>(vi)};
        }
      }
}

// The menu of workgroup tiles: rows, columns, waves per SIMD that the
// registers and LDS leave, and the tile's own time per area against the
// others'.  All give the same sums.
enum Tile { k64x64, k48x64, k64x32, k64x48, k64x80, k64x96, k64x112, k80x64, k32x64, k64x16, k32x32, k128x64, k64x128,
            k96x64, kTiles };
struct TileShape { int m, n, waves; double time; };
constexpr TileShape kTileShape[kTiles] = {
    {64, 64, 5, 1.0},  {48, 64, 6, 1.0}, {64, 32, 6, 1.0}, {64, 48, 6, 1.05},  {64, 80, 5, 1.0},  {64, 96, 4, 1.0},
    {64, 112, 4, 1.0}, {80, 64, 5, 1.0}, {32, 64, 6, 1.0}, {64, 16, 8, 1.1}, {32, 32, 8, 1.0}, {128, 64, 4, 1.0},
    {64, 128, 4, 1.0}, {96, 64, 4, 1.0}};

// Expected time of a launch in units of matrix-pipe work per CU: the padded
// tile area each of the 256 CUs gets through (whole rounds while the grid
// fills the chip only a few times), slower by 1 + 0.15 / n with n waves per
// SIMD to hide latencies, plus the tile's operand traffic (rows + columns).
// Fitted to 42 shapes of the GW contractions (nao 10 to 104, NQ 64 to 600) timed
// with every tile: the choice is within 0.7 % of the fastest tile on
// (geometric) average, within 11 % everywhere; 64 x 64 everywhere loses 15 %
// on average and 1.4-2x where an extent is just above 16, 32 or 64
// (sig_vg TFLOP/s, 64 x 64 against the choice: nao = 26 28 / 41, nao = 41
// 54 / 66, nao = 72 60 / 92).
double tile_cost(const GemmDesc& d, const TileShape& t) {
  const double tiles = (double)((d.M + t.m - 1) / t.m) * ((d.N + t.n - 1) / t.n) * d.nb0 * d.nb1;
  double rounds = tiles / 256.0;
  if (rounds <= 4.0 * t.waves) rounds = std::ceil(rounds);
  const double n = std::min<double>(t.waves, std::max(1.0, std::ceil(tiles / 256.0)));
  return t.time * rounds * ((double)t.m * t.n * (1.0 + 0.15 / n) + 4.0 * (t.m + t.n));
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

template <class TO, int WM, int WN, int MB, int NB, int WPE, bool AKC, bool BKC, int SITE, bool WIDE = false>
void launch_one(const GemmDesc& d, hipStream_t stream) {
  constexpr int TM = 16 * WM * MB, TN = 16 * WN * NB;
  const int64_t tiles = (int64_t)((d.M + TM - 1) / TM) * ((d.N + TN - 1) / TN);
  const int64_t total = tiles * d.nb0 * d.nb1;
  require(total < (int64_t)1 << 31, "gemm: grid too large");
  hipLaunchKernelGGL((gemm_f32_kernel<TO, WM, WN, MB, NB, WPE, AKC, BKC, SITE, WIDE>), dim3((unsigned)total),
                     dim3(64 * WM * WN), 0, stream, d);
  GGPU_HIP(hipGetLastError());
}

template <class TO, bool AKC, bool BKC, int SITE>
void launch_tile(const GemmDesc& d, hipStream_t stream, Tile t) {
  switch (t) {
    case k48x64: return launch_one<TO, 1, 4, 3, 1, 6, AKC, BKC, SITE>(d, stream);
    case k64x32: return launch_one<TO, 2, 2, 2, 1, 6, AKC, BKC, SITE>(d, stream);
    case k64x48: return launch_one<TO, 4, 1, 1, 3, 6, AKC, BKC, SITE>(d, stream);
    case k64x80: return launch_one<TO, 4, 1, 1, 5, 5, AKC, BKC, SITE>(d, stream);
    case k64x96: return launch_one<TO, 4, 1, 1, 6, 4, AKC, BKC, SITE>(d, stream);
    case k64x112: return launch_one<TO, 4, 1, 1, 7, 4, AKC, BKC, SITE>(d, stream);
    case k80x64: return launch_one<TO, 1, 4, 5, 1, 5, AKC, BKC, SITE>(d, stream);
    case k32x64: return launch_one<TO, 1, 4, 2, 1, 6, AKC, BKC, SITE>(d, stream);
    case k64x16: return launch_one<TO, 4, 1, 1, 1, 8, AKC, BKC, SITE>(d, stream);
    case k32x32: return launch_one<TO, 2, 2, 1, 1, 8, AKC, BKC, SITE>(d, stream);
    case k128x64: return launch_one<TO, 2, 2, 4, 2, 4, AKC, BKC, SITE>(d, stream);
    case k64x128: return launch_one<TO, 2, 2, 2, 4, 4, AKC, BKC, SITE>(d, stream);
    case k96x64: return launch_one<TO, 2, 2, 3, 2, 4, AKC, BKC, SITE>(d, stream);
    default: return launch_one<TO, 2, 2, 2, 2, 5, AKC, BKC, SITE>(d, stream);
  }
}

template <class TO>
void launch(const GemmDesc& d, hipStream_t stream, int variant) {
  const bool akc = (d.A.cs == 1) || (d.A.rs != 1), bkc = (d.B.rs == 1) || (d.B.cs != 1);
  // lane offsets within a tile are 32 bits wide: at most 128 rows and 8 k
  auto span = [](int64_t rs, int64_t ks) { return 8.0 * (128.0 * (double)std::abs(rs) + BK * (double)std::abs(ks)); };
  const bool wide = d.A.rs < 0 || d.A.cs < 0 || d.B.rs < 0 || d.B.cs < 0 || span(d.A.rs, d.A.cs) >= 4294967296.0 ||
                    span(d.B.cs, d.B.rs) >= 4294967296.0;
  if (wide) {
    if (akc && bkc) return launch_one<TO, 2, 2, 2, 2, 2, true, true, kSiteOther, true>(d, stream);
    if (akc) return launch_one<TO, 2, 2, 2, 2, 2, true, false, kSiteOther, true>(d, stream);
    if (bkc) return launch_one<TO, 2, 2, 2, 2, 2, false, true, kSiteOther, true>(d, stream);
    return launch_one<TO, 2, 2, 2, 2, 2, false, false, kSiteOther, true>(d, stream);
  }
  const Tile t = variant == 8 ? k64x64 : variant == 16 ? k128x64 : choose_tile(d);
  // each contraction site has its own symbol, compiled for its one layout and
  // result type
  if constexpr (std::is_same_v<TO, c32>) {
    switch (d.site) {
      case kSiteP0X1: return launch_tile<TO, true, false, kSiteP0X1>(d, stream, t);
      case kSiteP0X2: return launch_tile<TO, true, true, kSiteP0X2>(d, stream, t);
      case kSiteSigY1: return launch_tile<TO, true, false, kSiteSigY1>(d, stream, t);
      case kSiteSigY2: return launch_tile<TO, false, false, kSiteSigY2>(d, stream, t);
      default: break;
    }
  } else {
    switch (d.site) {
      case kSiteP0: return launch_tile<TO, false, true, kSiteP0>(d, stream, t);
      case kSiteSigma: return launch_tile<TO, true, true, kSiteSigma>(d, stream, t);
      default: break;
    }
  }
  if (akc && bkc) return launch_tile<TO, true, true, kSiteOther>(d, stream, t);
  if (akc) return launch_tile<TO, true, false, kSiteOther>(d, stream, t);
  if (bkc) return launch_tile<TO, false, true, kSiteOther>(d, stream, t);
  return launch_tile<TO, false, false, kSiteOther>(d, stream, t);
}

}  // namespace

void launch_f32(const GemmDesc& d, hipStream_t stream, int variant) {
  if (d.out_f32) launch<c32>(d, stream, variant);
  else launch<z64>(d, stream, variant);
}

}  // namespace ggpu
