// Shared helpers for libqmlhip: status codes, the thread-local error message, launch checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "qmlhip.h"

namespace qmlh {

// Record a message for qmlh_last_error() and return `code`.
int set_error(int code, const char* fmt, ...);

// Fold a HIP status into the library status convention.
inline int check_hip(hipError_t e, const char* what) {
    if (e != hipSuccess) return set_error(QMLH_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
    return QMLH_OK;
}

#define QMLH_CHECK_LAUNCH(what)                                                      \
    do {                                                                             \
        int _rc = ::qmlh::check_hip(hipGetLastError(), what);                        \
        if (_rc) return _rc;                                                         \
    } while (0)

#define QMLH_TRY(expr)                                                               \
    do {                                                                             \
        int _rc = (expr);                                                            \
        if (_rc) return _rc;                                                         \
    } while (0)

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline int64_t round_up(int64_t a, int64_t b) { return ceil_div(a, b) * b; }

// Workgroups of 256 lanes that a launch of work in a grid-stride loop takes at most: a grid of 2^32
// lanes and more is cut short without an error.
static constexpr int64_t MAX_GRID = (int64_t)1 << 23;

// FP64 MFMA operand/accumulator vector types.
typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

}  // namespace qmlh
