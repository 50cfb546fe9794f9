// Shared host-side helpers of libeet_hip.so: error reporting across the C ABI.
#pragma once
#include <cstdarg>
#include <cstdio>
#include <string>

#include "eet_hip.h"

namespace eet {

std::string &last_error_slot();

inline int fail(int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    last_error_slot() = buf;
    return code;
}

// glue.hip: eet_qkv_split, rotating by a caller's table (cos | sin of each position, [>= S][dh]) instead of its own
// angles where one is given.
int qkv_split(const void *qkv, void *q_out, void *k_cache, void *v_cache, int B, int S, int H, int dh, int rope,
              int time_step, int t0, int T_cap, const float *rope_cos_sin, void *stream);

}  // namespace eet

#define EET_REQUIRE(cond, code, ...)              \
    do {                                          \
        if (!(cond))                              \
            return ::eet::fail((code), __VA_ARGS__); \
    } while (0)

#define EET_HIP_CHECK(expr)                                                                   \
    do {                                                                                      \
        hipError_t _e = (expr);                                                               \
        if (_e != hipSuccess)                                                                 \
            return ::eet::fail(EET_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(_e));   \
    } while (0)
