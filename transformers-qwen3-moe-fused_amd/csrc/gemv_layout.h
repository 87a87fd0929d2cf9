// Which lanes of the packed matrix-vector kernel hold what of a column (gemm_nf4_gemv.hip).
#pragma once

namespace mfl {

// `lanes` to a column, each with `dwords` of 8 packed weights; side by side, or `lanes` dwords apart.
struct GemvLayout {
    int lanes, dwords;
    bool side_by_side;
    constexpr int reach() const { return 8 * lanes * dwords; }  // longest reduction that it covers
};

// By the sizes alone (256 < K <= 2048, K % 32 == 0, N % 32 == 0): the gated form's products are the same bits as the plain one's.
constexpr GemvLayout gemv_layout(int K, int N) {
    if (K > 1024) return {64, 4, true};
    // (16 lanes: plain product, N = 2048, 16 tokens of 8 experts each, fp32 / 8-bit scales: K = 768 22.1 / 25.6 -> 19.9 / 20.2
    // us, K = 512 21.4 / 25.1 -> 15.8 / 16.8.  K = 1024 with eight dwords a lane spills: 25.8 -> 30.9.)
    if (N % 64 == 0) {
        if (K <= 512) return {16, 4, true};
        if (K <= 768 && K % 192 == 0) return {16, 6, true};
    }
    if (K <= 768) return {32, 3, false};
    return {32, 4, true};
}

constexpr bool gemv_layouts_reach() {
    for (int K = 288; K <= 2048; K += 32)
        for (int N = 32; N <= 64; N += 32)
            if (gemv_layout(K, N).reach() < K) return false;
    return true;
}
static_assert(gemv_layouts_reach(), "a layout leaves elements of the reduction out");

}  // namespace mfl
