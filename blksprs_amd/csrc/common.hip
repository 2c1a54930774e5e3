// Error reporting of the C ABI, waits of the host.
#include "common.h"

namespace bsa {

char *error_buffer() {
  static thread_local char buf[512] = {0};
  return buf;
}

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(error_buffer(), 512, fmt, ap);
  va_end(ap);
  return code;
}

bool wait_for_word(const char *who, const int64_t *word, int64_t before, bsa_stream_t stream) {
  for (int turn = 1; __atomic_load_n(word, __ATOMIC_ACQUIRE) == before; ++turn) {
    if ((turn & 0xfff) != 0) {
      __builtin_ia32_pause();
      continue;
    }
    turn = 0;
    const hipError_t state = hipStreamQuery(as_stream(stream));
    if (state == hipErrorNotReady) {
      if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();  // not to be taken for a launch's
      continue;
    }
    if (state != hipSuccess) {
      fail(BSA_ELAUNCH, "%s: %s", who, hipGetErrorString(state));
      return false;
    }
    if (__atomic_load_n(word, __ATOMIC_ACQUIRE) == before) {
      fail(BSA_ELAUNCH, "%s: the kernel left no result", who);
      return false;
    }
  }
  return true;
}

}  // namespace bsa

extern "C" int bsa_abi_version(void) { return BSA_ABI_VERSION; }

extern "C" const char *bsa_last_error(void) { return bsa::error_buffer(); }

#ifndef BSA_BUILD_INFO
#define BSA_BUILD_INFO "hipcc: unknown (built without blksprs_amd/csrc/build.py)"
#endif
extern "C" const char *bsa_build_info(void) { return BSA_BUILD_INFO; }
