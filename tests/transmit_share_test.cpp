// Which payload wavefronts may transmit while rows are left to receive (wire.h), over every number of them that a
// launch can have.  Host compiler only.
#include <cstdio>

#include "wire.h"

int main() {
    using pcie_ep::transmit_wavefronts;
    // Up to 192 payload workgroups of 10 wavefronts.
    for (int waves = 1; waves <= 1920; ++waves) {
        for (int batch = 1; batch <= 2; ++batch) {
            const int transmit = transmit_wavefronts(waves, batch);
            bool fits = transmit >= 1 && transmit <= waves;  // somebody transmits
            if (waves >= 2) fits = fits && transmit <= waves - 1;  // and somebody only receives
            // At least a third of them receive only, at least half (rounded down) where rows come in pairs.
            fits = fits && (batch > 1 ? waves - transmit >= waves / 2 : waves == 1 || 3 * (waves - transmit) >= waves);
            if (!fits) {
                std::fprintf(stderr, "FAILED: %d of %d wavefronts may transmit (rows received %d at a time)\n", transmit, waves, batch);
                return 1;
            }
        }
    }
    const int cases[][3] = {{1, 1, 1}, {2, 1, 1}, {3, 1, 2}, {4, 1, 2}, {8, 1, 5}, {192, 1, 128}, {2, 2, 1}, {3, 2, 2}, {4, 2, 2}, {384, 2, 192}};
    for (const auto& item : cases) {
        if (transmit_wavefronts(item[0], item[1]) == item[2]) continue;
        std::fprintf(stderr, "FAILED: %d wavefronts, batch %d\n", item[0], item[1]);
        return 1;
    }
    std::printf("transmit share test passed\n");
    return 0;
}
