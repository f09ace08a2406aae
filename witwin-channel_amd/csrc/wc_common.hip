// Library identity and HIP errors of the C ABI.
#include "wc_api_internal.h"

int wc_fail_hip(const char* where, hipError_t err) {
    wc_fail("%s: HIP error %d (%s)", where, (int)err, hipGetErrorString(err));
    return 2;
}

extern "C" int wc_abi_version(void) { return 1; }

extern "C" const char* wc_build_target(void) { return "gfx950"; }
