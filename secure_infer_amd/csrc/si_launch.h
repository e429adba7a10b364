// Kernel launches and allocations that report their own status.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <tuple>
#include <type_traits>
#include <utility>

namespace si {

// Launches `kernel` and returns this launch's status.  HIP's last error is the
// thread's: a failure of any earlier call stays in it until somebody reads it,
// so reading it after a launch can report a kernel that is queued as refused.
// A refused launch is reported here and leaves no last error behind; an earlier
// call's stays for whoever made that call.  `start` and `stop`, unless null, are
// recorded at the kernel's dispatch start and end.
template <class... P, class... A>
hipError_t launch_timed(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t stream, hipEvent_t start,
                        hipEvent_t stop, A&&... a)
{
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    std::tuple<std::remove_cv_t<P>...> params(std::forward<A>(a)...);
    const hipError_t e = std::apply(
        [&](auto&... p) {
            void* args[] = {const_cast<void*>(static_cast<const volatile void*>(&p))...};
            const void* const f = reinterpret_cast<const void*>(kernel);
            return start || stop ? hipExtLaunchKernel(f, grid, block, args, 0, stream, start, stop, 0)
                                 : hipLaunchKernel(f, grid, block, args, 0, stream);
        },
        params);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

template <class... P, class... A>
hipError_t launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t stream, A&&... a)
{
    return launch_timed(kernel, grid, block, stream, nullptr, nullptr, std::forward<A>(a)...);
}

// An allocation's status, for a caller that reports a refusal itself: none stays
// behind as the thread's last error.
inline bool granted(hipError_t e)
{
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

}  // namespace si
