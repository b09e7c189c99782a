// Library-level entry points of libvxmix: version, limits, error messages.
#include <map>
#include <mutex>

#include "vx_common.hpp"

namespace vx {
std::string& last_error() {
    static thread_local std::string msg;
    return msg;
}

int cu_count() {
    static std::mutex m;
    static std::map<int, int> per_device;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    std::lock_guard<std::mutex> lk(m);
    auto it = per_device.find(dev);
    if (it != per_device.end()) return it->second;
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    return per_device[dev] = n;
}
}  // namespace vx

extern "C" const char* vx_version(void) { return "vxmix 0.1 (gfx950)"; }

extern "C" int32_t vx_max_nz(void) { return vx::kMaxNz; }

extern "C" const char* vx_last_error(void) { return vx::last_error().c_str(); }
