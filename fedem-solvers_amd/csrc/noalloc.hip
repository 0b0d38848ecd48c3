// The reduced load vectors without any device allocation: the work buffers
// of fgpu_reduce_loads_noalloc (the permuted load vectors, the partial sums
// of the B^T F and Phi^T F products and their results) live in one
// file-scope device array, `scratch`, that every GPU holds from library
// load until the process ends.  Host code never uses the array's name as an
// address: the per-device address comes from hipGetSymbolAddress at the
// first call on that device.  Calls on one GPU share the array, so calls
// that overlap on one GPU race; the entry point is synchronous.
#include <mutex>
#include <string>
#include "kernels.hpp"

namespace fgpu {

constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(32) << 20;  // 32 MiB per device

static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

// Device address of this GPU's scratch array (looked up once per device,
// with that device current).
int noalloc_scratch(double** ptr, size_t* bytes, std::string& err) {
  static std::mutex mu;
  static void* addr[64] = {};
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64) {
    err = std::string("no current device for the scratch array: ") + hipGetErrorString(e);
    return -3;
  }
  std::lock_guard<std::mutex> g(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      err = std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e);
      return -3;
    }
    addr[dev] = p;
  }
  *ptr = static_cast<double*>(addr[dev]);
  *bytes = NOALLOC_SCRATCH_BYTES;
  return 0;
}

}  // namespace fgpu
