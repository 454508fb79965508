// hip_error.hpp -- error plumbing of the VCSR-MC sources (host code only).
#pragma once
#include <hip/hip_runtime_api.h>

#include <stdexcept>
#include <string>

namespace vcsrmc {

// Internal error: carries a C-ABI status code; converted to a return value at the ABI.
struct Error : std::runtime_error {
    int status;
    Error(int s, const std::string& m) : std::runtime_error(m), status(s) {}
};

[[noreturn]] void throw_hip(hipError_t e, const char* what, const char* file, int line);

#define VCSRMC_HIP(call)                                                        \
    do {                                                                        \
        const hipError_t e_ = (call);                                           \
        if (e_ != hipSuccess) ::vcsrmc::throw_hip(e_, #call, __FILE__, __LINE__); \
    } while (0)

}  // namespace vcsrmc
