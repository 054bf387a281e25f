// Host-side checks shared by the launchers of the int4 library.
#pragma once

#include "common.hpp"

namespace {

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int check_problem(const void *x, const void *qw, const void *sc, const void *qz, const void *y,
                         long M, long N, long K, long G) {
    if (!x || !qw || !sc || !qz || !y) return VRL_INT4_ENULL;
    if (M < 1 || N < 1 || K < 8 || G < 8) return VRL_INT4_ESHAPE;
    if (K % 8 != 0 || G % 8 != 0 || K % G != 0) return VRL_INT4_ESHAPE;
    if (N * K >= (1L << 40) || M * K >= (1L << 31) || M * N >= (1L << 31)) return VRL_INT4_ESHAPE;
    if (!aligned16(x) || !aligned16(qw) || !aligned16(sc) || !aligned16(qz) || !aligned16(y))
        return VRL_INT4_EALIGN;
    return VRL_INT4_OK;
}

inline bool pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }

inline int device_cu_count() {
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            cus = v;
    }
    return cus;
}

}  // namespace
