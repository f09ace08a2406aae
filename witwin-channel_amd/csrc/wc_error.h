// Error channel of the C ABI, for host sources too.
#pragma once

// printf-style message for wc_last_error(); returns 1
int wc_fail(const char* format, ...) __attribute__((format(printf, 1, 2)));
