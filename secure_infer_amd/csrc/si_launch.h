// Kernel launches that report their own status.
#pragma once

#include <hip/hip_runtime.h>

#include <tuple>
#include <type_traits>
#include <utility>

namespace si {

// Launches `kernel` and returns this launch's status.  HIP's last error is the
// thread's: a failure of any earlier call stays in it until somebody reads it,
// so reading it after a launch can report a kernel that is queued as refused.
// A refused launch is reported here and leaves no last error behind; an earlier
// call's stays for whoever made that call.
template <class... P, class... A>
hipError_t launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t stream, A&&... a)
{
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    std::tuple<std::remove_cv_t<P>...> params(std::forward<A>(a)...);
    const hipError_t e = std::apply(
        [&](auto&... p) {
            void* args[] = {const_cast<void*>(static_cast<const volatile void*>(&p))...};
            return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, args, 0, stream);
        },
        params);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

}  // namespace si
