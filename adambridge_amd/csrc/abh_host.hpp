// abh_host.hpp -- what the library's sources share on the host: the calling thread's stream and
// error text (defined in abh_host.inc).
#pragma once

#include <hip/hip_runtime.h>

namespace abh {

extern thread_local hipStream_t t_stream;   // adambridge_set_stream

// Notes a HIP failure for adambridge_last_error and returns ADAMBRIDGE_EHIP.
int hip_fail(hipError_t e, const char* what);

}  // namespace abh
