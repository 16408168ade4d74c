// link_kernels.hip -- what the swap engine moves over the link by kernels of its own: payloads that somebody waits for,
// and the count that the host decides on.
//
// A payload that is asked for on demand comes in on the compute stream, in front of its decompression: whatever is queued
// there next needs it.  On a stream of its own it takes two events and two waits as well, each some 5 us on the GPU and
// 15 us of the host's time.  From the call to a kernel behind the copy, us, the runtime's copy on another stream / on the
// same stream / this kernel: 64 KB 39 / 18.1 / 5.4, 2 MB 70 / 53.5 / 42.0, 8 MB 181 / 164 / 152.  The link bounds it: 64 workgroups
// are enough (2 MB 40.4 us, 256 workgroups 51.8; 256 MB 4668, the runtime's copy 4694).
// It is not for copies beside other work.  The way out cannot be done like this at all: what a kernel has on its way
// to host memory holds up the end of every other kernel on the GPU (a small kernel beside 8 MB going out: seen to end after
// 131 us, beside the runtime's copy, which is none, after 5; beside this kernel 20).
#include <hip/hip_runtime.h>
#include "../../include/cswap_hip.h"
#include "common.h"

namespace cswap {

constexpr unsigned kLinkGroups = 64, kLinkThreads = 256;
typedef uint32_t any_u4 __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any 4-byte boundary

__global__ __launch_bounds__(kLinkThreads) void link_copy_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                                 size_t words)
{
  const size_t threads = (size_t)gridDim.x * kLinkThreads, me = (size_t)blockIdx.x * kLinkThreads + threadIdx.x;
  const size_t pieces = words >> 2;
  for (size_t i = me; i < pieces; i += threads)
    reinterpret_cast<any_u4*>(dst)[i] = reinterpret_cast<const any_u4*>(src)[i];
  if (me < (words & 3u)) dst[4 * pieces + me] = src[4 * pieces + me];
}

hipError_t link_copy(void* dst, const void* src, size_t bytes, hipStream_t stream)
{
  const size_t want = (bytes / 16 + kLinkThreads - 1) / kLinkThreads;
  const unsigned grid = (unsigned)(want < 1 ? 1 : want < kLinkGroups ? want : kLinkGroups);
  hipLaunchKernelGGL(link_copy_kernel, dim3(grid), dim3(kLinkThreads), 0, stream, static_cast<const uint32_t*>(src),
                     static_cast<uint32_t*>(dst), bytes / 4);
  return hipGetLastError();
}

// The count to where the host can read it when it has seen an event behind this: a copy of 4 bytes by the runtime takes
// 2 us more, and 11 where a payload is on its way.
__global__ void publish_count_kernel(const int* __restrict__ count, int* __restrict__ host) { *host = *count; }

hipError_t publish_count(int* host, const int* count, hipStream_t stream)
{
  hipLaunchKernelGGL(publish_count_kernel, dim3(1), dim3(1), 0, stream, count, host);
  return hipGetLastError();
}

}  // namespace cswap
