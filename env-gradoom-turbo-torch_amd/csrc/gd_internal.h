// Shared by the library's sources: how an entry point reports an error (gd_last_error).
#ifndef GD_INTERNAL_H
#define GD_INTERNAL_H

#include <hip/hip_runtime.h>

#include <string>

int gd_fail(int code, const std::string &message);   // keeps the message for gd_last_error and returns the code

#define GD_HIP_TRY(expr)                                                                       \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) return gd_fail(GD_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// A descriptor filled in against another version of the header is refused before any of its fields is trusted.
#define GD_SIZE_CHECK(ptr, type)                                                               \
    do {                                                                                       \
        if ((ptr)->struct_size != sizeof(type))                                                \
            return gd_fail(GD_E_ARG, #type ".struct_size is " + std::to_string((ptr)->struct_size) + ", this library expects " + \
                                         std::to_string(sizeof(type)) + ": the caller was built against another gradoom_amd.h"); \
    } while (0)

#endif
