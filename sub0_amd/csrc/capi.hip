// Library-wide pieces: version, per-thread error text, the device's CU count.
#include "cda_common.h"

namespace cda {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string &msg) { g_last_error = msg; }

int num_cus() {
    static const int cus = [] {
        int dev = 0, n = 0;
        return hipGetDevice(&dev) == hipSuccess &&
                       hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) ==
                           hipSuccess && n > 0
                   ? n : 256;
    }();
    return cus;
}

}  // namespace cda

extern "C" int cda_hip_version(void) { return 100; }

extern "C" const char *cda_hip_last_error(void) { return cda::g_last_error.c_str(); }
