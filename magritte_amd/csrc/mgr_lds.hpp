// mgr_lds.hpp -- LDS of the radiation-field kernel's workgroups (host
// arithmetic, no device code).
#pragma once

#include <algorithm>
#include <cstddef>

namespace mgr {

constexpr size_t LDS_LIMIT = 64 * 1024;   // dynamic LDS per workgroup

struct FieldLds {
    int    points;   // of a window
    size_t wave;     // bytes of each wave
    size_t total;    // of the workgroup
};

// nwg windows of up to `points` points, each `fixed` bytes and points + 1 rows
// of `row` bytes in a multiple of 64 bytes, and the line table behind them.
// With many lines and waves a window holds fewer points than asked for; 0 if
// not even two fit.
inline FieldLds field_lds(size_t fixed, size_t row, size_t table, int nwg, int points)
{
    const size_t share = (LDS_LIMIT - table) / nwg / 64 * 64;
    const size_t rows = share > fixed ? (share - fixed) / row : 0;
    if (rows < 3 || points < 2) return {0, 0, 0};
    points = (int)std::min<size_t>(points, rows - 1);
    const size_t wave = (fixed + row * (points + 1) + 63) / 64 * 64;
    return {points, wave, wave * nwg + table};
}

}  // namespace mgr
