// Copy of a large block that its writer will not read again soon: 16-byte
// nontemporal stores, which write whole lines without reading them first
// (a memcpy of a 2 MiB chunk stays below the C library's own threshold for
// them and reads every destination line).
#include <emmintrin.h>

#include <cstdint>
#include <cstring>

#include "rc_stream_copy.hpp"

void rc_stream_copy(void* dst, const void* src, size_t bytes) {
    uint8_t* d = static_cast<uint8_t*>(dst);
    const uint8_t* s = static_cast<const uint8_t*>(src);
    const size_t head = (64 - (reinterpret_cast<uintptr_t>(d) & 63)) & 63;  // whole lines
    if (bytes < head + 64) {
        std::memcpy(d, s, bytes);
        return;
    }
    std::memcpy(d, s, head);
    d += head;
    s += head;
    bytes -= head;
    for (; bytes >= 64; d += 64, s += 64, bytes -= 64) {
        const __m128i a = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s));
        const __m128i b = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 16));
        const __m128i c = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 32));
        const __m128i e = _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + 48));
        _mm_stream_si128(reinterpret_cast<__m128i*>(d), a);
        _mm_stream_si128(reinterpret_cast<__m128i*>(d + 16), b);
        _mm_stream_si128(reinterpret_cast<__m128i*>(d + 32), c);
        _mm_stream_si128(reinterpret_cast<__m128i*>(d + 48), e);
    }
    std::memcpy(d, s, bytes);
    _mm_sfence();
}
