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

}  // namespace

int main() {
    constexpr size_t kPiece = 128u << 10, kShared = 512u << 10;
    const size_t sizes[] = {0,           1,           kPiece,      kShared - 1,      kShared,
                            kShared + 1, 8 * kPiece + 3, 9u << 20, 2 * kPiece + 77};
    int bad = 0;
    for (size_t n : sizes) bad += !copies(n, (uint32_t)n);
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
