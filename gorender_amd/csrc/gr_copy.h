// Copy of host memory, shared by several threads when it is large (gr_copy.cpp).
#pragma once

#include <stddef.h>

namespace gr_internal {

void host_copy(void* dst, const void* src, size_t n);
// Zeroes a byte in every page of memory that nothing has been written to, so that its
// pages are mapped.
void host_touch(void* p, size_t n);

}  // namespace gr_internal
