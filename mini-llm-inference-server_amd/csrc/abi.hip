// Error reporting and version of the C ABI (include/minillm_hip.h).
#include <atomic>

#include "common.h"

namespace mllm {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MLLM_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
  return MLLM_OK;
}

int device_cus() {
  static std::atomic<int> known[64];  // per device, read once (0: not yet)
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64) {
    cus = known[dev].load(std::memory_order_relaxed);
    if (cus) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0) {
      known[dev].store(cus, std::memory_order_relaxed);
      return cus;
    }
  }
  (void)hipGetLastError();  // the failed query is not the next launch's error
  return 256;
}

}  // namespace mllm

extern "C" int mllm_abi_version(void) { return MLLM_ABI_VERSION; }

extern "C" const char* mllm_last_error(void) { return mllm::g_last_error.c_str(); }
