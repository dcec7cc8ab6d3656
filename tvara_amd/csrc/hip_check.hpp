// HIP status codes as exceptions.
#pragma once
#include <hip/hip_runtime_api.h>

#include <stdexcept>
#include <string>

namespace tvara_amd {

inline void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}
#define TVARA_HIP(x) ::tvara_amd::hip_check((x), #x)

}  // namespace tvara_amd
