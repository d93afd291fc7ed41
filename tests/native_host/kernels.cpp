// The entry points of the kernel library that native_calls.cpp calls, without kernels: they count their calls and keep
// the last epilogue.
#include "../../include/aitemplate_amd_kernels.h"

extern "C" {

__attribute__((visibility("default"))) int stub_launches = 0;
__attribute__((visibility("default"))) int stub_epilogue = -1;

const char* aitamd_last_error(void) { return "stub"; }

int aitamd_gemm_rcr_ws(int epilogue, int, int, const void*, const void*, const void*, const void*, const void*, void*, int64_t, int64_t,
                       int64_t, int64_t, int64_t, int64_t, int64_t, void*, int64_t, void*) {
  ++stub_launches;
  stub_epilogue = epilogue;
  return 0;
}

int aitamd_bmm(int, int, int, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
               int64_t, int64_t, int64_t, int64_t, void*) {
  ++stub_launches;
  return 0;
}

int aitamd_bmm_softmax_bmm_permute(int, const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t,
                                   int64_t, int64_t, float, int, void*) {
  ++stub_launches;
  return 0;
}

int aitamd_mem_eff_attention(int, const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t,
                             int64_t, float, int, const int32_t*, const int32_t*, void*) {
  ++stub_launches;
  return 0;
}

}
