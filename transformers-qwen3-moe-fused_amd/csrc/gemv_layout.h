// Which lanes of the packed matrix-vector kernel hold what of a column (gemm_nf4_gemv.hip).
#pragma once

namespace mfl {

// `lanes` to a column, each with `dwords` of 8 packed weights; side by side, or `lanes` dwords apart.
struct GemvLayout {
    int lanes, dwords;
    bool side_by_side;
    constexpr int reach() const { return 8 * lanes * dwords; }  // longest reduction that it covers
};

// 256 < K <= 2048, K % 32 == 0, N % 32 == 0; 1 << bs_shift: the smaller of the blocks of the one matrix or two.  A lane's run lies
// under one scale (two, in blocks of 64, with six dwords), which is loaded once.  Smaller blocks take their dwords apart, where
// neighbouring lanes load neighbouring scales: with the scales of a run each loaded where it is used, 128 experts and rows, blocks of
// 8 / 16, us: K = 2048, N = 768 plain 41 / 30, gated 67 / 53, against 30 / 24 and 53 / 43 apart; K = 768, N = 2048 39 / 33 and 72 / 57
// against 30 / 26 and 53 / 45, blocks of 32 30 and 52 against 24 and 42.  (With a run's scales in registers ahead 35 / 29 and 61 /
// 51 at K = 2048: the lanes' loads of a scale lie in as many lines as there are lanes.  K = 512 in blocks of 16 alone is behind
// apart, gated, 42 against 35.)  The gated form's products are the same bits as the plain one's where both matrices' blocks are
// equal.
constexpr GemvLayout gemv_layout(int K, int N, int bs_shift) {
    const bool runs = bs_shift >= 5;
    if (K > 1024) return {64, 4, runs};
    // (16 lanes: plain product, N = 2048, 16 tokens of 8 experts each, fp32 / 8-bit scales: K = 768 22.1 / 25.6 -> 19.9 / 20.2
    // us, K = 512 21.4 / 25.1 -> 15.8 / 16.8.  K = 1024 with eight dwords a lane spills: 25.8 -> 30.9.)
    if (N % 64 == 0) {
        if (K <= 512 && runs) return {16, 4, true};
        if (K > 512 && K <= 768 && K % 192 == 0 && bs_shift >= 6) return {16, 6, true};
    }
    if (K <= 768) return {32, 3, false};
    return {32, 4, runs};
}

// Halves of a row per expert up to which the kernel is taken: where it is ahead of the one that would follow, or even.
// Against the streaming kernel (K % 128 == 0, blocks of 64 and more), 128 experts, gated / plain us, H = 2048, I = 768, fp32
// scales: 48 / 26 against 57 / 27 at 1.5 rows, 58 / 31 against 58 / 31 at 2; I = 512: 32 / 18 against 39 / 20 at 1.5, 39 / 22
// against 40 / 20 at 2; K = 896: 59 / 32 against 59 / 33 at 1.5; 8-bit ones, whose sums are the same bits and the line
// therefore the same: 53 / 30 against 54 / 28 at 1.75, 59 / 32 against 55 / 30 at 2; I = 512: 34 / 19 against 37 / 20 at 1.5,
// 41 / 23 against 38 / 20 at 2.  Short reductions with the dwords apart are behind it past a row: K = 640, 1.125 rows 47 / 25
// against 41 / 23, 1.5 rows 54 / 28 against 42 / 24, 8-bit scales 64 / 33 against 41 / 23; K = 384 is in either layout (side by
// side, 1.25 rows, N = 448 / 1280 / 2048, plain 9.7 / 13.7 / 16.7 against 7.4 / 12.2 / 16.2, with 8-bit scales gated 13.5 / 22.2 /
// 29.8 against 11.8 / 19.8 / 26.4; N = 4096 27.7 against 31.1 and 52.6 against 54.0).  What the streaming kernel does not take
// goes to the register-decoding one, which is further behind: K = 704, 1.5 rows 54 / 29 against 61 / 33; K = 768 in blocks
// of 32 58 / 31 against 78 / 41, of 16 60 / 33 against 127 / 69; but below 512 in blocks of 32 and more it is ahead there: 60
// experts, K = 320, N = 992, 1.5 rows 17 / 10 against 13 / 7; 64 experts, K = 448, N = 1376, blocks of 32, 1.1 rows 19 / 12
// against 18 / 10.
constexpr int gemv_half_rows(int K, GemvLayout l, int bs_shift) {
    const bool streams = K % 128 == 0 && bs_shift >= 6;
    const bool decodes = K < 512 && bs_shift >= 5;
    if (streams && K < 512) return 2;
    return K > 1024 ? 4 : (streams || decodes) && !l.side_by_side ? 2 : 3;
}

constexpr bool gemv_layouts_reach() {
    for (int K = 288; K <= 2048; K += 32)
        for (int N = 32; N <= 64; N += 32)
            for (int bs_shift = 3; bs_shift <= 6; ++bs_shift)
                if (gemv_layout(K, N, bs_shift).reach() < K) return false;
    return true;
}
static_assert(gemv_layouts_reach(), "a layout leaves elements of the reduction out");

}  // namespace mfl
