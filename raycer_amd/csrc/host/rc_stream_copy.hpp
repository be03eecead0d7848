#pragma once
#include <cstddef>

// memcpy for blocks of a megabyte and more.
void rc_stream_copy(void* dst, const void* src, size_t bytes);
