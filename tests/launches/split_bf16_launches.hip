// Host-only build of the GEMM dispatch with a HIP runtime that launches nothing
// and prints every kernel and its grid: which kernels a split-bf16 product of many
// (pair, spin) entries runs, without a GPU.
//
// usage: split_bf16_launches VARIANT M N K NB0 NB1 WORKSPACE_BYTES
#include "zgemm.hip"

#include <cstdlib>
#include <map>
#include <string>
#include <vector>

static std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
static struct { dim3 grid, block; size_t shmem; hipStream_t stream; } config;

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
  config = {g, b, s, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = config.grid; *b = config.block; *s = config.shmem; *st = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void**, size_t, hipStream_t) {
  printf("%s %u %u %u\n", names()[f].c_str(), g.x, g.y, g.z);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}

namespace ggpu {
void launch_f64(const GemmDesc&, hipStream_t, int) { abort(); }
void launch_f32(const GemmDesc&, hipStream_t, int) { abort(); }
void gemm_int8_emulated(const GemmDesc&, int, void*, size_t, hipStream_t) { abort(); }
}

int main(int argc, char** argv) {
  if (argc != 8) return 2;
  using namespace ggpu;
  const int variant = atoi(argv[1]), M = atoi(argv[2]), N = atoi(argv[3]), K = atoi(argv[4]), nb0 = atoi(argv[5]),
            nb1 = atoi(argv[6]);
  static char base[16];                       // never read
  std::vector<int64_t> offA(nb1), offB(nb1);
  for (int e = 0; e < nb1; ++e) {
    offA[e] = (int64_t)(e / 2) * M * K;       // two spins share a pair's V
    offB[e] = (int64_t)e * nb0 * K * N;
  }
  GemmDesc g;                                 // Y1[t] = V G(t) of every entry
  g.compute = Compute::BF16X3;
  g.out_f32 = 1;
  g.site = kSiteSigY1;
  g.M = M; g.N = N; g.K = K; g.nb0 = nb0; g.nb1 = nb1;
  g.A.ptr = base; g.A.rs = K; g.A.cs = 1; g.A.off1 = offA.data(); g.A.off1_host = offA.data();
  g.B.ptr = base; g.B.rs = N; g.B.cs = 1; g.B.bs0 = (int64_t)K * N; g.B.off1 = offB.data();
  g.B.off1_host = offB.data();
  g.C.ptr = base; g.C.rs = N; g.C.cs = 1; g.C.bs0 = (int64_t)M * N; g.C.bs1 = (int64_t)nb0 * M * N;
  int table[kNumSites];
  for (int& v : table) v = variant;
  set_site_variants(table);
  set_gemm_workspace(base, strtoull(argv[7], nullptr, 10));   // never written
  try {
    gemm(g, nullptr);
  } catch (const std::exception& e) {
    printf("error: %s\n", e.what());
    return 1;
  }
  return 0;
}
