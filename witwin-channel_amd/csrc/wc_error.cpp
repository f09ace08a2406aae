// Error channel of the C ABI (host code: linked into both libraries).
#include "wc_error.h"

#include <cstdarg>
#include <cstdio>
#include <string>

namespace {
thread_local std::string g_last_error;
}

int wc_fail(const char* format, ...) {
    if (!format) {
        g_last_error = "unknown error";
        return 1;
    }
    char buffer[512];
    va_list args;
    va_start(args, format);
    std::vsnprintf(buffer, sizeof(buffer), format, args);
    va_end(args);
    g_last_error = buffer;
    return 1;
}

extern "C" const char* wc_last_error(void) { return g_last_error.c_str(); }

extern "C" void wc_clear_error(void) { g_last_error.clear(); }
