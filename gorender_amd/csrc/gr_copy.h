// Copy of host memory, shared by several threads when it is large (gr_copy.cpp).
#pragma once

#include <stddef.h>

namespace gr_internal {

void host_copy(void* dst, const void* src, size_t n);

}  // namespace gr_internal
