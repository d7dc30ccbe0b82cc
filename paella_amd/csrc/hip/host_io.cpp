// The aperture side of host_io.h.

#include "host_io.h"

#include <immintrin.h>

#include "direct_dispatch.h"

#include <cstring>

namespace paella {

namespace {

__attribute__((target("avx512f"))) size_t store_512(char* dst, const char* src, size_t bytes) {
    size_t i = 0;
    for (; i + 64 <= bytes; i += 64) _mm512_stream_si512(reinterpret_cast<__m512i*>(dst + i), _mm512_loadu_si512(src + i));
    return i;
}
size_t store_128(char* dst, const char* src, size_t bytes) {
    size_t i = 0;
    for (; i + 16 <= bytes; i += 16) _mm_stream_si128(reinterpret_cast<__m128i*>(dst + i), _mm_loadu_si128(reinterpret_cast<const __m128i*>(src + i)));
    return i;
}

__attribute__((target("avx512f"))) void load_line_512(char* dst, const char* src) {
    _mm512_storeu_si512(dst, _mm512_stream_load_si512(const_cast<char*>(src)));
}
__attribute__((target("sse4.1"))) void load_line_128(char* dst, const char* src) {
    for (int i = 0; i < 64; i += 16)
        _mm_storeu_si128(reinterpret_cast<__m128i*>(dst + i), _mm_stream_load_si128(reinterpret_cast<__m128i*>(const_cast<char*>(src + i))));
}
template <void (*Line)(char*, const char*)>
void load_lines(char* dst, const char* src, size_t bytes) {
    for (; bytes >= 64; bytes -= 64, dst += 64, src += 64) Line(dst, src);
    if (bytes) {
        char last[64];
        Line(last, src);
        std::memcpy(dst, last, bytes);
    }
}

bool wide() {
    static const bool has = __builtin_cpu_supports("avx512f");
    return has;
}

}  // namespace

bool host_map_device(void* p) { return __builtin_cpu_supports("sse4.1") && direct_allow_host_access(p); }

void host_store(void* dst, const void* src, size_t bytes) {
    char* d = static_cast<char*>(dst);
    const char* s = static_cast<const char*>(src);
    const size_t done = wide() ? store_512(d, s, bytes) : store_128(d, s, bytes);
    std::memcpy(d + done, s + done, bytes - done);
    _mm_sfence();
}

void host_settle(const void* dst, size_t bytes) {
    _mm_mfence();
    if (bytes) (void)*(static_cast<const volatile char*>(dst) + bytes - 1);
    _mm_lfence();
}

void host_load(void* dst, const void* src, size_t bytes) {
    _mm_mfence();  // a line that an earlier call left in a streaming buffer is fetched again
    if (wide()) load_lines<load_line_512>(static_cast<char*>(dst), static_cast<const char*>(src), bytes);
    else load_lines<load_line_128>(static_cast<char*>(dst), static_cast<const char*>(src), bytes);
}

}  // namespace paella
