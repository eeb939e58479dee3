// Host check of residency.h: with the padding, exactly the asked number of
// workgroups fits a compute unit's LDS, for every static size a march kernel
// may have, whichever of the two allocation units the device uses.
#include <cstdio>
#include <initializer_list>

#include "residency.h"

using namespace hipdvr;

int main() {
    for (size_t fixed = 0; fixed <= 20480; fixed += 32)
        for (int r = 1; r <= 8; ++r) {
            const size_t total = fixed + residency_pad(fixed, r);
            for (const size_t unit : {(size_t)kLdsUnit, (size_t)512}) {
                const size_t taken = (total + unit - 1) / unit * unit;
                const size_t fits = kCuLds / taken;
                // a workgroup that is larger than its share cannot be padded to it
                const bool large = fixed > (kCuLds / kLdsUnit / (size_t)(r + 1) + 1) * kLdsUnit;
                if (large ? fits > (size_t)r : fits != (size_t)r) {
                    std::printf("fixed %zu, %d per CU, unit %zu: %zu fit\n", fixed, r, unit, fits);
                    return 1;
                }
            }
        }
    std::printf("ok\n");
    return 0;
}
