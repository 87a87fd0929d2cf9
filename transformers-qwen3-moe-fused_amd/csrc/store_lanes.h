// Which of a wave's output stores are issued at all.  Plain constant-expression arithmetic, for host and device.
#pragma once

namespace mfl {

// Store u of a part of 32 rows x `cpr` 16-byte pieces covers pieces 64 u .. 64 u + 63, row-major.  Whether any of its lanes
// lies inside the first `rows` rows and `cols` columns (a piece holds 8; cols a multiple of 8): it starts in the middle of a
// row where cpr does not divide 64, and with the rest of that row past the last column its first piece to be stored is the
// first one of the row below (64 > cpr: every store reaches that row).
constexpr bool store_has_lane(int u, int cpr, int rows, int cols) {
    const int row = 64 * u / cpr, col = 64 * u % cpr * 8;
    return col < cols ? row < rows : cols > 0 && row + 1 < rows;
}

}  // namespace mfl
