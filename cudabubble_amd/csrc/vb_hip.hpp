// vb_hip.hpp -- checked HIP calls of the host code.
#pragma once
#include <hip/hip_runtime_api.h>

#include <string>

namespace vb {

// Every HIP call is checked; a failure becomes VB_ERR_HIP with a message.
struct HipError {
  hipError_t err;
  std::string where;
};
#define VB_HIP(call)                                                              \
  do {                                                                            \
    hipError_t e_ = (call);                                                       \
    if (e_ != hipSuccess) throw ::vb::HipError{e_, std::string(#call) + " @ " +   \
                                                  std::to_string(__LINE__)};      \
  } while (0)

}  // namespace vb
