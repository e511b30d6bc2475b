// Prints resident_min_iters() of batches on 256 compute units: count x
// workgroups a cloth, of half groups and of whole groups.
#include <cstdio>

#include "pcg_resident.hpp"

using namespace chysx_amd;

int main() {
    const int batches[][2] = {{1, 256}, {5, 44}, {2000, 1}, {2, 130}, {3, 130}, {8, 130}, {16, 130},
                              {8, 176}, {16, 64}, {64, 32}, {128, 20}, {8, 256}, {4096, 2}};
    for (const auto& b : batches) {
        const std::vector<int> c(size_t(b[0]), b[1]);
        std::printf("%dx%d %d %d\n", b[0], b[1], resident_min_iters(c, b[0] * ((b[1] + 1) / 2), true, 256),
                    resident_min_iters(c, b[0] * b[1], false, 256));
    }
    return 0;
}
