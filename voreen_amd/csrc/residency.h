// residency.h -- workgroups of a kernel per compute unit, limited through LDS.
#pragma once

#include <stddef.h>

namespace hipdvr {

// A compute unit's LDS, and the unit it is allocated in.
constexpr size_t kCuLds = 160 * 1024, kLdsUnit = 1280;

// Dynamic LDS with which at most `per_cu` workgroups of `fixed` bytes of
// static LDS are resident on a compute unit, and `per_cu` where their
// registers allow it: the least that leaves no room for one more.
constexpr size_t residency_pad(size_t fixed, int per_cu) {
    const size_t bytes = (kCuLds / kLdsUnit / (size_t)(per_cu + 1) + 1) * kLdsUnit;
    return bytes > fixed ? bytes - fixed : 0;
}

}  // namespace hipdvr
