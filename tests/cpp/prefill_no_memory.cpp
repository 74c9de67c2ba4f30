// Prefill where the device has no memory for the 32-row kernels' workspace, in
// the style of test_attn_cpp.cpp: this program's hipMalloc stands before the
// runtime's for the library too and refuses allocations past a limit, so that
// the prompts have to run as those without a workspace do, with the same
// result.  Run by tests/test_cpp_layer.py.
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "molot_amd/attn_hip.h"

#include "check_util.hpp"

static size_t limit = SIZE_MAX;

extern "C" hipError_t hipMalloc(void** p, size_t bytes) {
  using Fn = hipError_t (*)(void**, size_t);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipMalloc"));
  if (bytes > limit) return hipErrorOutOfMemory;
  return real ? real(p, bytes) : hipErrorNotInitialized;
}

static float* on_device(const std::vector<float>& x) {
  void* p = nullptr;
  if (hipMalloc(&p, x.size() * 4) != hipSuccess ||
      hipMemcpy(p, x.data(), x.size() * 4, hipMemcpyHostToDevice) != hipSuccess) {
    std::printf("no device memory\n");
    return nullptr;
  }
  return (float*)p;
}

int main() {
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    std::printf("no GPU\n");
    return 2;
  }
  const struct { int nq, nkv, d, M, N; } cases[] = {{32, 8, 128, 300, 4000}, {8, 2, 512, 100, 4000}};
  for (const auto& c : cases) {
    std::printf("[case] no memory for the workspace, d = %d\n", c.d);
    std::fflush(stdout);
    Rng rng(7);
    std::vector<float> q((size_t)c.M * c.nq * c.d), k((size_t)c.N * c.nkv * c.d), v(k.size());
    rng.normal(q);
    rng.normal(k);
    rng.normal(v);
    limit = SIZE_MAX;
    float *qd = on_device(q), *kd = on_device(k), *vd = on_device(v), *od = on_device(q);
    hipStream_t s = nullptr;
    if (!qd || !kd || !vd || !od || hipStreamCreate(&s) != hipSuccess) return 2;
    const float scale = 1.0f / std::sqrt((float)c.d);
    std::vector<float> out[2];
    // refused (28 MiB: the partials of split keys still fit), then allowed
    for (int i = 0; i < 2; ++i) {
      limit = i ? SIZE_MAX : (size_t)28 << 20;
      const int st = molot_hip_attn_prefill_gqa(qd, kd, vd, od, c.nq, c.nkv, c.M, c.N, c.d, scale,
                                                c.N - c.M, 0, MOLOT_KV_F32, s);
      CHECK(st == 0, "d = %d, %s: status %d", c.d, i ? "allowed" : "refused", st);
      CHECK(hipStreamSynchronize(s) == hipSuccess, "the stream");
      CHECK(hipGetLastError() == hipSuccess, "an error was left behind");
      out[i].resize(q.size());
      CHECK(hipMemcpy(out[i].data(), od, q.size() * 4, hipMemcpyDeviceToHost) == hipSuccess, "copy");
    }
    const double err = normwise(out[0], out[1]);
    std::printf("d = %d: normwise %.3e\n", c.d, err);
    CHECK(err < 1e-5, "d = %d: normwise %.3e", c.d, err);
    CHECK(out[0] != out[1], "d = %d: the same path both times", c.d);
  }
  std::printf(failures ? "%d FAILED\n" : "PASSED\n", failures);
  return failures ? 1 : 0;
}
