// common.h -- error plumbing shared by the translation units of libcswap_hip.so
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/cswap_hip.h"

namespace cswap {

// hipError_t of the most recent failure on this thread (0 = none)
int& last_hip_error();

inline int hip_fail(hipError_t e)
{
  last_hip_error() = (int)e;
  return CSWAP_E_HIP;
}

// compute units of the current device (0 if the query fails), looked up once per device
int device_compute_units();

// cswap_zfp_compress_f32 / cswap_zfp_decompress_f32 of a packed field without the form for the smallest
// fields (four lanes per block), whatever the size
int zfp_compress_f32_no_quad(const float* d_in, size_t nx, size_t ny, size_t nz, unsigned maxbits, uint64_t* d_stream,
                             hipStream_t stream);
int zfp_decompress_f32_no_quad(const uint64_t* d_stream, size_t nx, size_t ny, size_t nz, unsigned maxbits, float* d_out,
                               hipStream_t stream);

// Whether cswap_zvc_compress_fused runs one kernel for a shape that cswap_zvc_takes_single_pass says 0 for.
bool zvc_small_any_chunk(int n, int process);

// cswap_zvc_compress_fused for a caller that looks at the count: shapes whose workgroups would count for themselves where
// the workspace fails them, at milliseconds a call, write -1 instead.
int zvc_compress_fused_reporting(const float* d_in, int n, int process, void* d_ws, int* d_begin, int* d_nnz, float* d_values,
                                 uint32_t* d_mask, hipStream_t stream);

// Whether a ZVC payload of `bytes` that is already made is worth sending: by the selector's model, what a
// tensor of n elements has left to pay for it (link and expansion) against the raw swap.
bool made_payload_pays(size_t n, size_t bytes, const cswap_costs& costs);

// A copy between device memory and pinned host memory as a kernel on the stream (link_kernels.hip).  Addresses and
// bytes are multiples of 4.
hipError_t link_copy(void* dst, const void* src, size_t bytes, hipStream_t stream);

// *host (pinned memory) becomes *count
hipError_t publish_count(int* host, const int* count, hipStream_t stream);

// to be called right after a kernel launch: picks up launch-configuration errors
inline int check_launch()
{
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? CSWAP_OK : hip_fail(e);
}

#define CSWAP_HIP_TRY(expr)                                   \
  do {                                                        \
    hipError_t e_ = (expr);                                   \
    if (e_ != hipSuccess) return ::cswap::hip_fail(e_);       \
  } while (0)

}  // namespace cswap
