// Lanes per wave of small batches (sirius_amd/csrc/sirius_internal.hpp, thin_lanes): whatever grid the caller
// chose, either whole waves take rays or every ray of the batch is in flight at once, and on a grid of
// a wave for each SIMD or more no wave takes more than its share. Prints "OK".
#include "../../sirius_amd/csrc/sirius_internal.hpp"

#include <cstdio>

int main() {
    const int64_t simds = 1024;
    for (int64_t n : {1, 3, 64, 255, 256, 1000, 4095, 4096, 4097, 8000, 15000, 22500, 65535})
        for (int64_t waves : {1, 4, 64, 255, 256, 257, 512, 1023, 1024, 1025, 2048, 4096, 16384}) {
            const int64_t l = sirius::thin_lanes(n, waves, simds);
            const int64_t share = (n + simds - 1) / simds;
            if (l < 1 || l > 64 || (l < 64 && l * waves < n) || (waves >= simds && l > (share > 4 ? share : 4)))
                return std::printf("%lld rays on %lld waves: %lld lanes\n", (long long)n, (long long)waves, (long long)l), 1;
        }
    std::puts("OK");
    return 0;
}
