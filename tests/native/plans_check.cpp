// The split-x GEMM's plans and the kernels that serve them, on the CPU: every
// plan over a grid of shapes has its kernel, and every kernel a plan.  The
// HIP calls defined here take the place of the runtime library's, so nothing
// is launched where there is a GPU either.
//
//   plans_check KERNELS    KERNELS: gemm_bf3 / bf3s / bf3k instantiations in the
//                          object; prints "plans_check: ok" and the counts
//   plans_check plan KIND M N K PAIR    the tile of one plan
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../../welvet.metal_amd/csrc/dense.hip"

namespace {
std::set<const void *> launched;
}

extern "C" {
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
  launched.insert(f);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;  // CUs of the MI355X
  return hipSuccess;
}
}

int main(int argc, char **argv) {
  using namespace wh;
  if (argc == 7) {
    const int bk = std::atoi(argv[2]), M = std::atoi(argv[3]), N = std::atoi(argv[4]), K = std::atoi(argv[5]);
    SkPlan p = plan_fwd_gemm(0, bk, M, K, N, std::atoi(argv[6]) ? 2 : 1);
    if (p.bm == 64) p = plan_fwd_gemm(0, bk, M, K, N);  // pair_gemm_plan
    std::printf("%dx%d%s%s\n", p.bm, p.bn, p.kg == 2 ? "x2" : "", p.sums ? "+" : "");
    return 0;
  }
  const int Ms[] = {5, 8, 13, 16, 17, 20, 32, 33, 48, 64, 65, 100, 128, 130, 256, 600, 2100};
  const int Ns[] = {1, 100, 300, 512, 777, 1024, 1368, 3000, 4096, 8192, 8200, 11008, 20000};
  const int Ks[] = {16, 64, 80, 128, 512, 1008, 1024, 2048, 2064, 2112, 3136, 4096, 8192, 11008, 11072};
  long plans = 0;
  for (int bk = BK_E4; bk <= BK_U8; ++bk)
    for (int M : Ms)
      for (int N : Ns)
        for (int K : Ks)
          for (int pair = 0; pair < 2; ++pair) {
            if (bk >= BK_B16 && M <= 16) continue;                                // bf3_fwd_kind
            if ((bk == BK_F32 || bk == BK_U8) && N < 512) continue;
            if (pair && bk >= BK_B16 && bk != BK_I4) continue;                    // pair_gemm_plan
            SkPlan p = plan_fwd_gemm(0, bk, M, K, N, pair ? 2 : 1);
            if (pair && p.bm == 64) p = plan_fwd_gemm(0, bk, M, K, N);
            if (p.rows) continue;
            GemmArgs a{};
            ++plans;
            const int64_t units = (int64_t)p.gx * p.gy * p.nst;
            if (launch_bf3(p, bk, a, nullptr, pair != 0) != hipSuccess || (int64_t)p.blocks * p.per_block < units ||
                (int64_t)(p.blocks - 1) * p.per_block >= units) {
              std::printf("plans_check: kind %d M %d N %d K %d pair %d\n", bk, M, N, K, pair);
              return 1;
            }
          }
  const int kernels = argc > 1 ? std::atoi(argv[1]) : -1;
  std::printf("plans_check: %ld plans on %zu of %d kernels\n", plans, launched.size(), kernels);
  if ((int)launched.size() != kernels) return 1;
  std::printf("plans_check: ok\n");
  return 0;
}
