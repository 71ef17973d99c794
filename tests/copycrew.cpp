// Copies of CopyCrew over sizes around its limits, then the CPU time that its
// helpers take while there is nothing to copy.
#include <sys/resource.h>

#include <chrono>
#include <cstdio>
#include <vector>

#include "lb3d_copycrew.h"

static double cpu_seconds()
{
    rusage u;
    getrusage(RUSAGE_SELF, &u);
    return u.ru_utime.tv_sec + u.ru_stime.tv_sec + 1e-6 * (u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

int main()
{
    const size_t MB = 1u << 20;
    std::vector<unsigned char> src(8 * MB + 5), dst(8 * MB + 5);
    for (size_t k = 0; k < src.size(); k++) src[k] = (unsigned char)(k * 2654435761u >> 13);
    for (size_t total : {(size_t)1, 16 * MB - 1, 16 * MB, 64 * MB}) {
        lb3d::CopyCrew crew(total);
        for (size_t n : {(size_t)0, (size_t)1, MB - 1, MB, MB + 4097, 8 * MB - 3, 8 * MB}) {
            for (int pause = 0; pause < 2; pause++) {  // helpers awake, and after a pause
                if (pause) std::this_thread::sleep_for(std::chrono::milliseconds(5));
                std::fill(dst.begin(), dst.end(), (unsigned char)0xa5);
                crew.copy(dst.data() + 2, src.data() + 1, n);
                if (std::memcmp(dst.data() + 2, src.data() + 1, n) || dst[0] != 0xa5 || dst[1] != 0xa5 ||
                    dst[n + 2] != 0xa5) {
                    std::printf("wrong copy of %zu bytes\n", n);
                    return 1;
                }
            }
        }
    }
    lb3d::CopyCrew crew(64 * MB);
    crew.copy(dst.data(), src.data(), 8 * MB);
    const double t0 = cpu_seconds();
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
    std::printf("%.4f\n", cpu_seconds() - t0);
    return 0;
}
