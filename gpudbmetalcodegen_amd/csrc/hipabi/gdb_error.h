#pragma once
// The library's error text, one per host thread: every file of the library
// sets the same one, so gdb_last_error() always tells of the last failure.

#include "gdb/gdb_hip.h"

#include <hip/hip_runtime.h>

#include <string>

namespace gdbhip {

gdb_status fail(gdb_status code, const std::string& message);
gdb_status hipFail(hipError_t e, const char* what);  // GDB_ERR_OOM or GDB_ERR_HIP, with the error's name
// The error of the kernel launches since the last call, if any.
inline gdb_status launchCheck(const char* what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? GDB_OK : hipFail(e, what);
}

}  // namespace gdbhip
