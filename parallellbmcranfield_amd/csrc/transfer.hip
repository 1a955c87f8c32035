// transfer.hip — the copies between device memory and pinned slots (transfer.hpp).
//
// Bound by the link (56 GB/s for one large copy either way).  The runtime's
// own copy costs about 15 us each on top of the bytes, one after the other on
// a stream: 28 GB/s at 512 kB and 14 GB/s at the 170 kB that one of three
// planes has of a slot.  One kernel per slot moves all its parts instead.
#include "transfer.hpp"

namespace lbmhost {
namespace {
struct Parts {
  const char* src[Staging::MAX_PARTS];
};

// Part blockIdx.y of `n` words to dst + blockIdx.y * n.
template <class T>
__global__ __launch_bounds__(256) void k_parts(T* __restrict__ dst, Parts p, size_t n) {
  const T* __restrict__ src = (const T*)p.src[blockIdx.y];
  dst += (size_t)blockIdx.y * n;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    dst[i] = src[i];
}

template <class T>
hipError_t launch(char* dst, const Parts& p, int count, size_t bytes, hipStream_t st) {
  const size_t n = bytes / sizeof(T), blocks = std::min<size_t>((n + 255) / 256, 256);
  k_parts<T><<<dim3((unsigned)blocks, (unsigned)count), 256, 0, st>>>((T*)dst, p, n);
  return hipGetLastError();
}
}  // namespace

hipError_t Staging::copy(void* dst, const void* const* src, int count, size_t bytes,
                         hipStream_t st) const {
  if (count < 1 || count > MAX_PARTS) return hipErrorInvalidValue;
  if (bytes == 0) return hipSuccess;
  Parts p{};
  size_t low = (size_t)dst | bytes;  // alignment that all parts have
  for (int k = 0; k < count; k++) {
    p.src[k] = (const char*)src[k];
    low |= (size_t)src[k];
  }
  if (pinned_ && low % 4 == 0) {
    if (low % 16 == 0) return launch<uint4>((char*)dst, p, count, bytes, st);
    if (low % 8 == 0) return launch<uint2>((char*)dst, p, count, bytes, st);
    return launch<uint32_t>((char*)dst, p, count, bytes, st);
  }
  hipError_t e = hipSuccess;
  for (int k = 0; k < count && e == hipSuccess; k++)
    e = hipMemcpyAsync((char*)dst + (size_t)k * bytes, src[k], bytes, hipMemcpyDefault, st);
  return e;
}

}  // namespace lbmhost
