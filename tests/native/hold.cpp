// The steps that stay on the streaming kernels after solves whose workgroups
// did not meet.
#include <cstdio>

#include "pcg_resident.hpp"

using namespace chysx_amd;

// steps until the next try
int held(ResidentHold& H) {
    int n = 0;
    while (!H.may_run()) ++n;
    return n;
}

int main() {
    ResidentHold H;
    std::printf("%d", held(H));
    for (int k = 0; k < 9; ++k) {  // every try misses
        H.missed();
        std::printf(" %d", held(H));
    }
    for (int k = 0; k < ResidentHold::kLongest; ++k) held(H);  // as many meet
    H.missed();
    std::printf(" %d\n", held(H));
    return 0;
}
