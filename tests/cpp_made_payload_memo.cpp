// The selector memo of the C++ scheduler mirror on a tensor whose ZVC payload goes out in the first iteration
// because the probe has made it, though the selector says raw: the following iterations swap it raw, without a
// probe.  Built and run by tests/test_made_payload_memory.py; prints "OK", then tag and probes of each iteration.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <string.h>

#include <vector>

#include "cswap_execution.hpp"

#define HIP_OK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { printf("hip error %d at line %d\n", (int)e_, __LINE__); return 2; } } while (0)
#define CS_OK(x) do { int r_ = (x); if (r_ != CSWAP_OK) { printf("cswap error %d (%s) at line %d\n", r_, cswap_strerror(r_), __LINE__); return 3; } } while (0)

int main()
{
  const size_t nx = 32, ny = 32, nz = 1024, n = nx * ny * nz;  // 4.2 MB
  cswap_engine_config cfg;
  cswap_engine_config_default(&cfg);
  cfg.pinned_pool_bytes = cfg.device_pool_bytes = (size_t)32 << 20;
  cswap_engine* eng = nullptr;
  CS_OK(cswap_engine_create(&eng, &cfg));

  std::vector<float> host(n), back(n);
  unsigned s = 2024;
  for (float& v : host) {
    s = s * 1664525u + 1013904223u;
    v = (s >> 24) % 20 < 11 ? 0.0f : (float)((s >> 8) & 0xffff) / 65536.0f + 0.5f;
  }
  float* dev;
  HIP_OK(hipMalloc((void**)&dev, 4 * n));
  HIP_OK(hipMemcpy(dev, host.data(), 4 * n, hipMemcpyHostToDevice));
  hipStream_t compute;
  HIP_OK(hipStreamCreate(&compute));

  cswap::Execution exe(eng);
  exe.init_(2);
  exe.policy = {-1, 0};
  std::vector<unsigned long long> seen;
  for (int iter = 0; iter < 4; iter++) {
    const unsigned long long before = cswap_engine_probe_count(eng);
    exe.preforward();
    CS_OK(exe.pre(-1, nullptr, 1, 1, 1, compute));
    exe.post();
    CS_OK(exe.pre(0, dev, nx, ny, nz, compute));
    int st = 0;
    exe.post(&st);
    CS_OK(st);
    exe.postforward();
    seen.push_back((unsigned long long)exe.com_and_tran(0));
    seen.push_back(cswap_engine_probe_count(eng) - before);
    HIP_OK(hipMemsetAsync(dev, 0xff, 4 * n, compute));
    CS_OK(exe.fetch(0, dev, compute));
    HIP_OK(hipStreamSynchronize(compute));
    HIP_OK(hipMemcpy(back.data(), dev, 4 * n, hipMemcpyDeviceToHost));
    if (memcmp(back.data(), host.data(), 4 * n) != 0) { printf("iteration %d came back different\n", iter); return 5; }
  }
  HIP_OK(hipFree(dev));
  HIP_OK(hipStreamDestroy(compute));
  cswap_engine_destroy(eng);
  printf("OK");
  for (unsigned long long v : seen) printf(" %llu", v);
  printf("\n");
  return 0;
}
