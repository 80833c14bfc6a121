// Host-only check of the shared copy (gr_copy.cpp) for the sanitizer builds: callers
// at once, of whom most find the helper threads taken, copies one after the other,
// sizes around a piece and around the least shared size, and a forked child.
#include <sys/wait.h>
#include <unistd.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "gorender_hip.h"
#include "gr_copy.h"
#include "gr_error.h"

namespace gr_internal {
gr_status fail(gr_status s, const std::string&) { return s; }
}  // namespace gr_internal

namespace {

bool copies(size_t n, uint32_t seed) {
    std::vector<uint32_t> src(n / 4 + 2), dst(n / 4 + 18, 0u);
    for (size_t i = 0; i < src.size(); i++) src[i] = (uint32_t)i * 2654435761u ^ seed;
    if (gr_host_copy(dst.data(), src.data(), n) != GR_OK) return false;
    const unsigned char* past = (const unsigned char*)dst.data() + n;
    for (int k = 0; k < 64; k++)
        if (past[k]) return false;
    return std::memcmp(src.data(), dst.data(), n) == 0;
}

// host_touch of [skew, skew + n) of a buffer: a byte of every page of it cleared,
// nothing around it.
bool touches(size_t skew, size_t n) {
    std::vector<unsigned char> buf(skew + n + 4096, 1);
    gr_internal::host_touch(buf.data() + skew, n);
    for (size_t i = 0; i < skew; i++)
        if (!buf[i]) return false;
    for (size_t i = skew + n; i < buf.size(); i++)
        if (!buf[i]) return false;
    const uintptr_t at = (uintptr_t)buf.data() + skew;
    for (uintptr_t page = at / 4096; n && page <= (at + n - 1) / 4096; page++) {
        bool any = false;
        for (uintptr_t i = page * 4096; i < (page + 1) * 4096; i++)
            if (i >= at && i < at + n) any = any || !buf[skew + (i - at)];
        if (!any) return false;
    }
    return true;
}

}  // namespace

int main() {
    constexpr size_t kPiece = 128u << 10, kShared = 512u << 10;
    const size_t sizes[] = {0,           1,           kPiece,      kShared - 1,      kShared,
                            kShared + 1, 8 * kPiece + 3, 9u << 20, 2 * kPiece + 77};
    int bad = 0;
    for (size_t n : sizes) bad += !copies(n, (uint32_t)n);
    for (size_t skew : {(size_t)0, (size_t)1, (size_t)4096, (size_t)2000000})
        for (size_t n : {(size_t)0, (size_t)1, (size_t)4096, (size_t)4097, (size_t)2u << 20,
                         ((size_t)2u << 20) + 1, (size_t)11u << 20})
            bad += !touches(skew, n);
    std::vector<std::thread> callers;
    std::vector<int> wrong(4, 0);
    for (uint32_t t = 0; t < 4; t++)
        callers.emplace_back([&, t] {
            for (uint32_t k = 0; k < 60; k++) wrong[t] += !copies(kShared + 4096 * k + t, 100 * t + k);
        });
    for (std::thread& c : callers) c.join();
    for (int w : wrong) bad += w;
    const pid_t child = fork();
    if (child == 0) _exit(copies(4u << 20, 7) ? 0 : 1);
    int status = 1;
    if (child < 0 || waitpid(child, &status, 0) != child || status != 0) bad++;
    std::printf("%d wrong\n", bad);
    return bad ? 1 : 0;
}
