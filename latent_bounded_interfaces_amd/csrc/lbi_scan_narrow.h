// Suffix scan of matrices up to 128 wide (lbi_scan_narrow.hip).
#pragma once

#include <cstdlib>

#include "lbi_common.h"

namespace lbi {

// LBI_SCAN_CHUNK: 0 forces the plain chain, n >= 2 chunks of n; -1 where it is not set.
inline int scan_forced_chunk() {
    static const int forced = std::getenv("LBI_SCAN_CHUNK") ? std::atoi(std::getenv("LBI_SCAN_CHUNK")) : -1;
    return forced;
}

namespace scan_narrow {
// Row tiles of 16 that a scan of this width runs on: 16-bit rows come through LDS in pairs of k tiles from 64 columns on.
inline int row_tiles(int d, int dtype) {
    const int nt = (d + 15) / 16;
    return dtype != LBI_F32 && nt > 4 ? nt + nt % 2 : nt;
}
// Whether a scan of B chains of K matrices runs here.
bool takes(const void* mats, int B, int K, int d, int in_dtype);
// The scan of K >= 1 matrices, with the cotangents where `cot` is given.
int scan(const void* mats, int in_dtype, void* out, const void* g, void* cot, int B, int K, int d, hipStream_t stream);
// The cotangents alone.
bool takes_chain(const void* mats, int B, int K, int d, int in_dtype);
int chain(const void* mats, int in_dtype, const void* g, void* cot, int B, int K, int d, hipStream_t stream);
}  // namespace scan_narrow
}  // namespace lbi
