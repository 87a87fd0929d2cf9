// Fused NF4 grouped product for batches of a few rows per expert (256 < K <= 2048): a matrix-vector form.
//
// With one or two rows per expert there is nothing for a matrix core to share: a 32-row MFMA tile would
// be 3 to 6 % full, and what the launch has to do is pull every routed expert's packed weights through
// the chip once.  So no tile and no LDS stage:
//   * a wave owns two output columns at a time, 16 apart (one of both matrices in the gated form, where the second matrix
//     takes the registers).  Its 64 lanes lie along the reduction, 32 weights in a row to a lane: one load of 16 bytes a
//     lane takes a column of K = 2048, and the lane's weights lie under one scale.  (With the lanes' dwords 64 dwords
//     apart a column took four loads of weights and four of scales, eight of 8-bit ones, which spilled: 16 tokens of 8
//     experts out of 128, gated, N = 768, fp32 / 8-bit scales 40.8 / 51.2 -> 36.8 / 37.3 us; one token 8.2 / 12.0 -> 8.5 /
//     9.2.  Blocks of fewer weights than a lane's run still take that form.)
//   * the rows of the group (up to two of one expert) stay in registers for all columns of the group: 16
//     bytes per lane, load and row.
//   * a byte of packed weights is two weights and one dword of bf16 pairs: a 256-entry table in LDS holds
//     the finished pair, and v_dot2_f32_bf16 multiplies it with the row's pair.  An entry is 256 bytes: 32
//     copies for the first matrix, 32 for the second of the gated form; lane l reads copy l & 31, so the 64
//     lookups of a wave meet no bank conflict, and the address 256 * byte + 4 * copy is ONE byte permute.
//     One vector instruction per byte for the address, one per byte and row for the product; the scale goes
//     onto the partial sum of the 8 weights in fp32.
//   * the 64 partial sums of each of the two columns (or of the two matrices' column) become 32 + 32 in one swap of half
//     waves (v_permlane32_swap) and an add, and five data-parallel-primitive adds finish both at once.
//   * one workgroup of 16 waves per CU, as many workgroups as CUs, and the (row group, 32 columns) units of
//     the launch (16 columns in the gated form) dealt out in equal contiguous shares: no second round of
//     workgroups, and a workgroup changes rows once or twice.  Each wave keeps the loads of four columns ahead
//     in registers.
//   * rows of at most 1024 elements: 32 lanes to a column, the wave's second column (16 further on) in lanes 32..63; up to
//     512, and for 576 and 768: 16 lanes and four columns, four or six dwords to a lane (gemv_layout.h).  No swap before
//     the adds.
//   What the loop is short of, with 16 waves to a CU, is issue slots, scalar ones first: addresses move by
//   increments, the row count is branched on once per column, and the lookups of a dword wait once.
//
// The product is the sum over pieces of 32 weights (16 of six dwords a lane, 8 where the dwords lie apart) of absmax * (x . bf16(code)), as in the streaming form.
#include <mutex>
#include <type_traits>

#include "common.h"
#include "gemm.h"
#include "gemv_layout.h"

namespace mfl {

namespace {

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((address_space(3))) void *lds_void_ptr;
typedef const __attribute__((address_space(3))) uint32_t *lds_u32_ptr;

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_fadd_step(float x) {
    // lanes without a source, and rows that the mask leaves out, add 0
    const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROW_MASK, 0xf, true);
    return x + __builtin_bit_cast(float, y);
}
// a: 64 partial sums of one column, b: of another.  Returns the first column's sum in lane 31 and the second's in
// lane 63: v_permlane32_swap exchanges lanes 32..63 of its first operand with lanes 0..31 of its second, so the
// sum of the two holds a[l] + a[l + 32] in lanes 0..31 and b[l - 32] + b[l] in lanes 32..63.  (Written out: through
// __builtin_amdgcn_permlane32_swap, with both results feeding one add, the compiler added the first result to
// itself.  The no-ops keep the wait states that the swap and the moves after it need from their neighbours.)
__device__ __forceinline__ float two_sums_to_31_and_63(float a, float b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    float x = a + b;
    x = dpp_fadd_step<0x111, 0xf>(x);  // row_shr 1
    x = dpp_fadd_step<0x112, 0xf>(x);  // row_shr 2
    x = dpp_fadd_step<0x114, 0xf>(x);  // row_shr 4
    x = dpp_fadd_step<0x118, 0xf>(x);  // row_shr 8
    x = dpp_fadd_step<0x142, 0xa>(x);  // row_bcast 15 into rows 1 and 3
    return x;
}

// each run of CL lanes (16 or 32) holds the partial sums of a column: the sums in the last lanes of the runs
template <int CL>
__device__ __forceinline__ float sums_to_last_lanes(float x) {
    x = dpp_fadd_step<0x111, 0xf>(x);  // row_shr 1
    x = dpp_fadd_step<0x112, 0xf>(x);  // row_shr 2
    x = dpp_fadd_step<0x114, 0xf>(x);  // row_shr 4
    x = dpp_fadd_step<0x118, 0xf>(x);  // row_shr 8
    if constexpr (CL == 32) x = dpp_fadd_step<0x142, 0xa>(x);  // row_bcast 15 into rows 1 and 3
    return x;
}

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

// Four table reads and one wait for all of them, written out: the compiler would wait before each use, and with
// 16 waves to a CU the issue slots of those waits are not free.  The addresses count from LDS address 0.
__device__ __forceinline__ void lookup4(uint32_t (&pr)[4], uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
    asm volatile(
        "ds_read_b32 %0, %4\n\tds_read_b32 %1, %5\n\tds_read_b32 %2, %6\n\tds_read_b32 %3, %7\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(pr[0]), "=&v"(pr[1]), "=&v"(pr[2]), "=&v"(pr[3])
        : "v"(a0), "v"(a1), "v"(a2), "v"(a3));
}

// the same with a fifth read of its own address
__device__ __forceinline__ void lookup5(uint32_t (&pr)[4], float &f, uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3,
                                        uint32_t af) {
    asm volatile(
        "ds_read_b32 %4, %9\n\tds_read_b32 %0, %5\n\tds_read_b32 %1, %6\n\tds_read_b32 %2, %7\n\tds_read_b32 %3, %8\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(pr[0]), "=&v"(pr[1]), "=&v"(pr[2]), "=&v"(pr[3]), "=&v"(f)
        : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "v"(af));
}

constexpr int kGemvThreads = 1024;
constexpr int kGemvTable = 65536;
constexpr int kGemvScales = 2048;  // scales by 8-bit value, of either matrix (double-quantised matrices)

__device__ __forceinline__ uint16_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, (bf16_t)v); }

// The LDS address of the pair of packed byte `B` of w: 256 * byte + lane_copy (the lane's copy of the table, one
// byte), put together by one byte permute.
template <int B>
__device__ __forceinline__ uint32_t pair_address(uint32_t w, uint32_t lane_copy) {
    // byte 0 of the result: byte 0 of lane_copy; byte 1: byte B of w; bytes 2 and 3: zero
    return __builtin_amdgcn_perm(w, lane_copy, 0x0c0c0000u | ((4u + B) << 8));
}

// CL: lanes per column; NL: dwords of a column per lane (K <= 8 CL NL); ROWS: rows per group; D: columns whose loads a wave
// keeps in flight; WIDE: the dwords of a lane lie side by side (above), else CL dwords apart
template <int CL, int NL, int ROWS, int D, bool GLU, bool WIDE, bool NESTED, typename TO>
__global__ __launch_bounds__(kGemvThreads) void nf4_gemv_kernel(const bf16_t *__restrict__ x,
                                                                const int32_t *__restrict__ row_idx, int idx_div,
                                                                Nf4Matrix w0, Nf4Matrix w1,
                                                                const void *__restrict__ m_sizes, int ms_i64,
                                                                TO *__restrict__ y, TO *__restrict__ e_out,
                                                                TO *__restrict__ g_out, int64_t R, int N, int K,
                                                                int E, int units_n, int max_groups) {
    constexpr int CB = GLU ? 2 : 1;
    // CL < 64: the wave's other columns (16 further on each) lie in its other lanes: a load serves all of them, and the sums
    // need no swap.
    constexpr int SUB = 64 / CL;
    // Columns in registers of their own: two, 16 apart, for the plain product with all 64 lanes to a column (the loop's
    // scalar work and the sum over the lanes are shared by both); one for the gated form, whose second matrix leaves no
    // registers for a second column.
    constexpr int COLS = (GLU || SUB > 1) ? 1 : 2;
    constexpr int UCOLS = 16 * SUB * COLS;  // columns of a unit
    // Scales of a column per lane: the 48 weights of six dwords lie under one or two blocks of 64, two neighbouring dwords
    // always under one; the 32 of four dwords under one.
    constexpr bool TWO = WIDE && NL == 6;
    static_assert(!WIDE || NL == 4 || (CL == 16 && NL == 6), "");
    constexpr int NS = TWO ? 2 : WIDE ? 1 : NL;
    static_assert(D % CB == 0, "the matrix of a ring slot is fixed");
    extern __shared__ __attribute__((aligned(256))) unsigned char smem[];
    unsigned char *const table = smem;                      // kGemvTable bytes
    int *const grp_e = (int *)(smem + kGemvTable + (NESTED ? kGemvScales : 0));          // expert | rows << 16
    int *const grp_r = grp_e + max_groups;                  // first row
    int *const n_groups_s = grp_r + max_groups;
    uint16_t *const code_s = (uint16_t *)(n_groups_s + 1);  // the code values of either matrix as bf16
    int *const ms_s = n_groups_s + 17;                      // the E counts
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // the lookups address the table from LDS address 0: the kernel has no static LDS in front of the dynamic
    // (the launcher asks the runtime and does not launch a build that has)
    // the counts and the codes: one round trip
    int ms_own[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int e = tid + j * kGemvThreads;
        ms_own[j] = e < E ? load_msize(m_sizes, ms_i64, e) : 0;
    }
    if (tid < 16 * CB) code_s[tid] = bf16_bits((tid < 16 ? w0 : w1).code16[tid & 15]);
    if constexpr (NESTED)
        if (tid < 256 * CB) ((float *)(table + kGemvTable))[tid] = (tid < 256 ? w0 : w1).code256[tid & 255];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int e = tid + j * kGemvThreads;
        if (e < E) ms_s[e] = ms_own[j];
    }
    __syncthreads();
    // ---- row groups in the order of the experts: group g = rows grp_r[g] .. of expert grp_e[g] & 0xffff
    if (wave == 0) {
        int row_carry = 0, grp_carry = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            int m = e < E ? ms_s[e] : 0;
            if (m < 0) m = 0;
            const int minc = wave_inclusive_scan(m);
            const int64_t start = (int64_t)row_carry + minc - m;
            if (start + m > R) m = start < R ? (int)(R - start) : 0;  // counts that run past the rows given
            const int g = ceil_div(m, ROWS);
            const int ginc = wave_inclusive_scan(g);
            const int gb = grp_carry + ginc - g;
            for (int q = 0; q < g && gb + q < max_groups; ++q) {
                const int rows = m - q * ROWS < ROWS ? m - q * ROWS : ROWS;
                grp_e[gb + q] = e | (rows << 16);
                grp_r[gb + q] = (int)start + q * ROWS;
            }
            row_carry += wave_last(minc);
            grp_carry += wave_last(ginc);
        }
        if (lane == 0) *n_groups_s = grp_carry < max_groups ? grp_carry : max_groups;
    } else {
        // ---- pair table, filled by the other waves meanwhile: entry b = bf16(code[b >> 4]) in the low half (the first of
        // the two weights is the high nibble), bf16(code[b & 15]) in the high half.  Entry b is the 256 bytes at 256 b: 32
        // copies for the first matrix, 32 for the second.  Neighbouring threads write neighbouring 16 bytes: written 64
        // bytes of an entry to a thread, the 64 lanes of a store met in the same four banks (3600 cycles of conflicts a CU,
        // 1.7 us of the gated form's 14 at one token).
        for (int p = tid - 64; p < 256 * 8 * CB; p += kGemvThreads - 64) {
            const int b = p / (8 * CB), piece = p % (8 * CB);
            const uint16_t *const code = code_s + (piece >> 3) * 16;
            const uint32_t u = code[b >> 4] | (uint32_t)code[b & 15] << 16;
            const uint4_t v = {u, u, u, u};
            *(uint4_t *)(table + b * 256 + piece * 16) = v;
        }
    }
    __syncthreads();

    // ---- this workgroup's share of the units (row group, 16 columns), row group major
    // (equal shares, the first U % gridDim.x workgroups one unit more; the host keeps U below 2^31)
    const uint32_t U = (uint32_t)*n_groups_s * (uint32_t)units_n;
    const uint32_t share = U / gridDim.x, extra = U % gridDim.x;
    const uint32_t u_begin = blockIdx.x * share + (blockIdx.x < extra ? blockIdx.x : extra);
    const uint32_t u_end = u_begin + share + (blockIdx.x < extra ? 1 : 0);
    if (u_begin >= u_end) return;
    const int n_items = (int)(u_end - u_begin) * CB;  // (unit, matrix) pairs, matrix minor

    // ---- what a lane reads of a column: dword i of its NL, if that is inside the row (else it reads the row's first)
    uint32_t x_off[NL];
    bool inside[NL];
    const Nf4Matrix mat[2] = {w0, w1};
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int l = lane % CL;
        const int k = WIDE ? l * (8 * NL) : (i * CL + l) * 8;
        inside[i] = k < K;
        x_off[i] = (uint32_t)(inside[i] ? k : 0) + (WIDE ? 8 * i : 0);
    }
    const uint32_t copy_off = (lane & 31) * 4;  // + 128 for the second matrix

    // ---- the ring of columns ahead
    uint32_t ring_w[D][COLS][NL];  // a slot: the wave's columns of a unit
    float ring_a[D][COLS][NS];     // the scale; double-quantised: its second-level factor,
    uint32_t ring_q[NESTED ? D : 1][COLS][NS];  // and its 8-bit value
    float q_off[CB];
    if constexpr (NESTED) {
        q_off[0] = *w0.offset;
        if constexpr (CB == 2) q_off[1] = *w1.offset;
    }
    // Cursor of the loads: the wave's column of unit ic of group ig.  The pointers move on by 16 columns per unit
    // (N % 16 == 0: every unit is whole) and are set up afresh when the group changes: a handful of scalar
    // instructions per column instead of the 64-bit products, which with 16 waves to a CU are what the scalar
    // unit has no time for.
    const int ig0 = (int)(u_begin / (uint32_t)units_n), ic0 = (int)(u_begin % (uint32_t)units_n);
    int ig = ig0, ic = ic0;
    int i_units_left = (int)(u_end - u_begin);
    const uint32_t *i_wp[CB];
    const float *i_ap[CB];
    const uint8_t *i_qp[CB];
    int64_t i_b[CB];  // double-quantised: number of the first scale behind i_qp
    auto point_loads = [&]() {
        const int expert = __builtin_amdgcn_readfirstlane(grp_e[ig]) & 0xffff;
        const int64_t base = ((int64_t)expert * N + ic * UCOLS + wave) * K;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            i_wp[cb] = (const uint32_t *)(mat[cb].wq + (base >> 1));
            if constexpr (NESTED) {
                i_b[cb] = base >> mat[cb].bs_shift;
                i_qp[cb] = mat[cb].absmax_u8 + i_b[cb];
            } else {
                i_ap[cb] = mat[cb].absmax + (base >> mat[cb].bs_shift);
            }
        }
    };
    point_loads();
    const int w_step = 2 * K;  // dwords of 16 columns
    int a_step[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) a_step[cb] = (16 * K) >> mat[cb].bs_shift;
    auto issue = [&](int d) {
        const int cb = d % CB;
        auto weights = [&](uint32_t (&to)[NL], const uint32_t *from) {
            if constexpr (SUB > 1) from += (lane / CL) * w_step;
            if constexpr (WIDE) {
                typedef uint4_t __attribute__((aligned(8))) piece_t;  // (24 bytes a lane)
                const uint4_t v = *(const piece_t *)(from + (x_off[0] >> 3));
#pragma unroll
                for (int i = 0; i < 4; ++i) to[i] = v[i];
                if constexpr (NL == 6) {
                    const uint2_t u = *(const uint2_t *)(from + (x_off[0] >> 3) + 4);
                    to[4] = u[0], to[5] = u[1];
                }
            } else {
#pragma unroll
                for (int i = 0; i < NL; ++i) to[i] = from[x_off[i] >> 3];
            }
        };
        weights(ring_w[d][0], i_wp[cb]);
        if constexpr (COLS == 2) weights(ring_w[d][1], i_wp[cb] + w_step);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            // (computed here: a register per load and matrix less)
            const uint32_t a_off = (x_off[i * (TWO ? NL - 1 : 1)] >> mat[cb].bs_shift) + (SUB > 1 ? (lane / CL) * a_step[cb] : 0);
#pragma unroll
            for (int c = 0; c < COLS; ++c) {
                const uint32_t at = a_off + c * a_step[cb];
                // (E N K / 64 scales: their numbers fit 32 bits, which the launcher checks)
                if constexpr (NESTED) {
                    ring_q[d][c][i] = i_qp[cb][at];
                    ring_a[d][c][i] = mat[cb].absmax2[((uint32_t)i_b[cb] + at) >> mat[cb].bs2_shift];
                } else {
                    ring_a[d][c][i] = i_ap[cb][at];
                }
            }
        }
        // past the end the cursor stays on the last unit: loads that nobody uses
        if (cb == CB - 1 && i_units_left > 1) {
            --i_units_left;
            if (++ic == units_n) {
                ic = 0;
                ++ig;
                point_loads();
            } else {
#pragma unroll
                for (int c2 = 0; c2 < CB; ++c2) {
                    i_wp[c2] += (UCOLS / 16) * w_step;
                    if constexpr (NESTED) {
                        i_b[c2] += (UCOLS / 16) * a_step[c2];
                        i_qp[c2] += (UCOLS / 16) * a_step[c2];
                    } else {
                        i_ap[c2] += (UCOLS / 16) * a_step[c2];
                    }
                }
            }
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d);

    // ---- the loop over the columns
    uint4_t xr[ROWS][NL];
    int cg = ig0, cc = ic0;  // cursor of the arithmetic
    int rows = 0, row0 = 0, o_col = cc * UCOLS;
    int64_t o_row[ROWS];  // where the wave's column of unit 0 is in the output, per row of the group
    bool fresh = true;
    float first[ROWS];  // the gate projection's sums (of a lane, or finished), until the up projection's are there
    // One column: the arithmetic on ring slot d, then (in the loop) the loads of the column D further on into it.
    auto column = [&](const int d, const bool more) {
            const int cb = d % CB;
            if (fresh) {
                fresh = false;
                const int ge = __builtin_amdgcn_readfirstlane(grp_e[cg]);
                rows = ge >> 16;
                row0 = __builtin_amdgcn_readfirstlane(grp_r[cg]);
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    // (CL = 64: lanes 32..63 end up with the second column)
                    o_row[r] = (int64_t)(row0 + r) * N + wave + (SUB > 1 ? lane / CL : COLS == 2 ? lane >> 5 : 0) * 16;
                    int64_t src_row = row0 + (r < rows ? r : rows - 1);
                    if (row_idx != nullptr) src_row = (uint32_t)row_idx[src_row] / (uint32_t)idx_div;
                    const bf16_t *const xp = x + src_row * K;
#pragma unroll
                    for (int i = 0; i < NL; ++i) {
                        const uint4_t v = *(const uint4_t *)(xp + x_off[i]);
                        const uint4_t zero = {0, 0, 0, 0};
                        xr[r][i] = inside[i] ? v : zero;
                    }
                }
            }
            const uint32_t lane_copy = copy_off + cb * 128;
            // The slot's values move to registers of the column and the slot is asked for again right away, in one
            // place for all row counts: were the loads issued inside the branches below, the branches would load
            // into different registers, and the copy that reconciles them would wait for the load just issued.
            // (the next loads are asked for behind the arithmetic, in one place for all row counts: asked for inside
            // the branches below they would land in different registers per branch, and the copy that reconciles
            // them would wait for the load just issued)
            // the arithmetic of the two columns for RN rows: one branch on the number of rows per unit, none inside
            auto arithmetic = [&](auto RN) {
                constexpr int rn = decltype(RN)::value;
                float acc[COLS][rn];
#pragma unroll
                for (int c = 0; c < COLS; ++c)
#pragma unroll
                    for (int r = 0; r < rn; ++r) acc[c][r] = 0.f;
                float scale[COLS][NS], part[COLS][rn];
                constexpr int RUN = TWO ? 2 : WIDE ? NL : 1;  // dwords whose products are summed before they are scaled
#pragma unroll
                for (int i = 0; i < NL; ++i) {
#pragma unroll
                    for (int c = 0; c < COLS; ++c) {
                        uint32_t pr[4];
                        const uint32_t w = ring_w[d][c][i];
                        if (NESTED && i < NS) {
                            float q;
                            lookup5(pr, q, pair_address<0>(w, lane_copy), pair_address<1>(w, lane_copy),
                                    pair_address<2>(w, lane_copy), pair_address<3>(w, lane_copy),
                                    ring_q[d][c][i] * 4 + (kGemvTable + cb * 1024));
                            scale[c][i] = q * ring_a[d][c][i] + q_off[cb];
                        } else {
                            lookup4(pr, pair_address<0>(w, lane_copy), pair_address<1>(w, lane_copy),
                                    pair_address<2>(w, lane_copy), pair_address<3>(w, lane_copy));
                            if (i < NS) scale[c][i] = ring_a[d][c][i];
                        }
                        const float under = TWO && i > 1 && ((x_off[i] ^ x_off[0]) >> 6) != 0 ? scale[c][NS - 1] : scale[c][WIDE ? 0 : i];
#pragma unroll
                        for (int r = 0; r < rn; ++r) {
                            float s = dot2_bf16(pr[0], xr[r][i][0], i % RUN == 0 ? 0.f : part[c][r]);
                            s = dot2_bf16(pr[1], xr[r][i][1], s);
                            s = dot2_bf16(pr[2], xr[r][i][2], s);
                            s = dot2_bf16(pr[3], xr[r][i][3], s);
                            part[c][r] = s;
                            if (i % RUN == RUN - 1) acc[c][r] = RUN == NL ? under * s : __builtin_fmaf(under, s, acc[c][r]);
                        }
                    }
                }
                // the 64 partial sums of each of two columns (the gated form: of the same column of the two matrices) become
                // 32 + 32 in one swap of half waves and one add, and five data-parallel-primitive adds finish both: the
                // first one's sum in lane 31, the second's in 63
                float tot[rn];
                if constexpr (GLU && SUB == 1) {
                    if (cb == 0) {
#pragma unroll
                        for (int r = 0; r < rn; ++r) first[r] = acc[0][r];
                        return;
                    }
                }
#pragma unroll
                for (int r = 0; r < rn; ++r) {
                    if constexpr (SUB > 1)
                        tot[r] = sums_to_last_lanes<CL>(acc[0][r]);
                    else
                        tot[r] = two_sums_to_31_and_63(GLU ? first[r] : acc[0][r], acc[COLS - 1][r]);
                }
                if constexpr (GLU && SUB > 1) {
                    if (cb == 0) {
#pragma unroll
                        for (int r = 0; r < rn; ++r) first[r] = tot[r];
                        return;
                    }
                }
                if constexpr (GLU && SUB == 1) {
#pragma unroll
                    for (int r = 0; r < rn; ++r)
                        first[r] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tot[r]), 31));
                }
                if (SUB > 1 ? lane % CL == CL - 1 : COLS == 2 ? (lane & 31) == 31 : lane == 63) {  // one lane per column
#pragma unroll
                    for (int r = 0; r < rn; ++r) {
                        const int64_t o = o_row[r] + o_col;
                        if constexpr (GLU) {
                            const bf16_t pe = (bf16_t)first[r], pg = (bf16_t)tot[r];
                            ((bf16_t *)y)[o] = silu_fwd_one<bf16_t>(pe, pg);
                            if (e_out) ((bf16_t *)e_out)[o] = pe;
                            if (g_out) ((bf16_t *)g_out)[o] = pg;
                        } else {
                            y[o] = from_f32<TO>(tot[r]);
                        }
                    }
                }
            };
            static_assert(ROWS == 2, "");
            if (rows == 1)
                arithmetic(std::integral_constant<int, 1>());
            else
                arithmetic(std::integral_constant<int, 2>());
            if (more) issue(d);
            if (cb == CB - 1) {
                o_col += UCOLS;
                if (++cc == units_n) {
                    cc = 0;
                    o_col = 0;
                    ++cg;
                    fresh = true;
                }
            }
    };
    // Whole rounds of the ring in a loop without a way out of its middle, the rest behind it: with an exit
    // between two columns the compiler sees a path from a column's loads straight to the head of the loop,
    // where they would be the youngest in flight, and waits for every load at every column.
    const int rounds = n_items / D, rest = n_items % D;
    for (int q = 0; q < rounds; ++q) {
#pragma unroll
        for (int d = 0; d < D; ++d) column(d, true);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (d < rest) column(d, false);
}

template <int CL, int NL, int ROWS, int D, bool GLU, bool WIDE, bool NESTED, typename TO>
int launch_gemv(const bf16_t *x, const int32_t *row_idx, int idx_div, const Nf4Matrix &w0, const Nf4Matrix &w1,
                const void *m_sizes, int ms_i64, TO *y, TO *e_out, TO *g_out, int64_t R, int N, int K, int E,
                hipStream_t stream) {
    if (K > 8 * CL * NL) return MFL_ERR_UNSUPPORTED;  // the lanes would leave the end of the reduction out
    const int64_t max_groups = R / ROWS + (R < E ? R : E);  // upper bound on sum over experts of ceil(m / ROWS)
    const int lds = kGemvTable + kGemvScales + (int)max_groups * 8 + 80 + E * 4;
    auto *kernel = nf4_gemv_kernel<CL, NL, ROWS, D, GLU, WIDE, NESTED, TO>;
    static PerDeviceOnce attr;
    // The table lookups take the dynamic LDS to start at address 0; static LDS in this kernel would move it, so
    // such a build is left to the kernels that decode in registers.
    static std::atomic<int> static_lds{-1};
    const hipError_t e = attr.run([&] {
        hipFuncAttributes fa;
        const hipError_t e1 = hipFuncGetAttributes(&fa, (const void *)kernel);
        if (e1 != hipSuccess) return e1;
        static_lds.store((int)fa.sharedSizeBytes, std::memory_order_release);
        return hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kGemvTable + kGemvScales + 4096 * 8 + 80 + 2048 * 4);
    });
    if (e != hipSuccess) return (int)e;
    if (static_lds.load(std::memory_order_acquire) != 0) return MFL_ERR_UNSUPPORTED;
    kernel<<<(unsigned)device_info().cu_count, kGemvThreads, lds, stream>>>(x, row_idx, idx_div, w0, w1, m_sizes, ms_i64,
                                                                            y, e_out, g_out, R, N, K, E,
                                                                            N / (CL < 64 ? 1024 / CL : GLU ? 16 : 32), (int)max_groups);
    return launch_status();
}

// ---- the down projection of a token or two with the routing-weighted sum behind it
//
// At one token the product is 4 us of loads, and the sum over its selections behind it another launch of 4 us that waits for
// it.  A workgroup takes 8 output columns of all selections: its 16 waves are 8 selections x 2 times 4 columns of 16 lanes each
// (the layout, the sums and so the bits of the kernel above), the selections' results meet in LDS, rounded as they would be in
// memory, and one thread per token and column adds them up in the order of the selections, as the combine kernel does.
// A selection's expert and its row come from the routing's own arrays, so nothing waits for counts and row groups.
// One token, 8 of 128 experts, K = 768, N = 2048: 6.8 + 3.9 us -> 5.6, and a launch less (a pass alone 79 ->
// 67 us with the gated product's).
constexpr int kDownRows = 16;  // selections of all tokens

template <int NL, bool NESTED>
__global__ __launch_bounds__(kGemvThreads) void nf4_down_combine_kernel(const bf16_t *__restrict__ h, const int32_t *__restrict__ inv,
                                                                        const int64_t *__restrict__ idx,
                                                                        const bf16_t *__restrict__ weights, Nf4Matrix w0,
                                                                        bf16_t *__restrict__ out, int R, int k, int N, int K,
                                                                        int E) {
    constexpr bool TWO = NL == 6;
    constexpr int RUN = TWO ? 2 : NL;
    extern __shared__ __attribute__((aligned(256))) unsigned char smem[];
    unsigned char *const table = smem;  // at LDS address 0, entries of 256 bytes, 128 of them used
    float *const scales_s = (float *)(smem + kGemvTable);
    float *const ys = scales_s + 256;            // (selection, column)
    float *const weights_s = ys + kDownRows * 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15;
    const int col = (wave & 1) * 4 + (lane >> 4), j0 = blockIdx.x * 8;
    const int first = l * (8 * NL);  // the lane's weights of a column
    const bool inside = first < K;
    const int x_off = inside ? first : 0;
    const bool crosses = TWO && inside && (first & 63) != 0;

    uint32_t w[NL];
    float a[TWO ? 2 : 1];
    uint32_t q[TWO ? 2 : 1];
    uint4_t x[NL];
    bool routed = false;
    auto load = [&](int s) {
        const int64_t e = idx[s];
        routed = e >= 0 && e < E;  // (a token of NaN logits selects no expert; its weights are NaN)
        if (!routed) return;
        const int64_t at = (e * N + j0 + col) * K + x_off;
        typedef uint4_t __attribute__((aligned(8))) piece_t;
        const uint4_t v = *(const piece_t *)(w0.wq + (at >> 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = v[i];
        if constexpr (TWO) {
            const uint2_t u = *(const uint2_t *)(w0.wq + (at >> 1) + 16);
            w[4] = u[0], w[5] = u[1];
        }
#pragma unroll
        for (int i = 0; i < (TWO ? 2 : 1); ++i) {
            const int64_t b = (at + i * 8 * (NL - 1)) >> w0.bs_shift;
            if constexpr (NESTED) {
                q[i] = w0.absmax_u8[b];
                a[i] = w0.absmax2[b >> w0.bs2_shift];
            } else {
                a[i] = w0.absmax[b];
            }
        }
        const bf16_t *const row = h + (int64_t)inv[s] * K + x_off;
        const uint4_t zero = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint4_t v8 = *(const uint4_t *)(row + 8 * i);
            x[i] = inside ? v8 : zero;
        }
    };
    int s = wave >> 1;
    if (s < R) load(s);
    if constexpr (NESTED)
        if (tid < 256) scales_s[tid] = w0.code256[tid];
    if (tid < R) weights_s[tid] = to_f32(weights[tid]);
#pragma unroll
    for (int p = tid; p < 256 * 8; p += kGemvThreads) {
        const int b = p >> 3;
        const uint32_t u = bf16_bits(w0.code16[b >> 4]) | (uint32_t)bf16_bits(w0.code16[b & 15]) << 16;
        const uint4_t v = {u, u, u, u};
        *(uint4_t *)(table + b * 256 + (p & 7) * 16) = v;
    }
    float offset = 0.f;
    if constexpr (NESTED) offset = *w0.offset;
    __syncthreads();
    const uint32_t lane_copy = (lane & 31) * 4;
    while (s < R) {
        float acc = 0.f, part = 0.f;
        if (routed) {
            float scale[TWO ? 2 : 1];
#pragma unroll
            for (int i = 0; i < (TWO ? 2 : 1); ++i) scale[i] = NESTED ? scales_s[q[i]] * a[i] + offset : a[i];
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                uint32_t pr[4];
                lookup4(pr, pair_address<0>(w[i], lane_copy), pair_address<1>(w[i], lane_copy), pair_address<2>(w[i], lane_copy),
                        pair_address<3>(w[i], lane_copy));
                const float under = TWO && i > 1 && crosses && (((first + 8 * i) ^ first) >> 6) != 0 ? scale[TWO ? 1 : 0] : scale[0];
                float t = dot2_bf16(pr[0], x[i][0], i % RUN == 0 ? 0.f : part);
                t = dot2_bf16(pr[1], x[i][1], t);
                t = dot2_bf16(pr[2], x[i][2], t);
                t = dot2_bf16(pr[3], x[i][3], t);
                part = t;
                if (i % RUN == RUN - 1) acc = RUN == NL ? under * t : __builtin_fmaf(under, t, acc);
            }
        }
        const float y = sums_to_last_lanes<16>(acc);
        if (l == 15) ys[s * 8 + col] = to_f32((bf16_t)y);
        s += 8;
        if (s < R) load(s);
    }
    __syncthreads();
    if (tid < R / k * 8) {
        const int t = tid >> 3, c = tid & 7;
        float acc = 0.f;
        for (int j = 0; j < k; ++j) acc = __builtin_fmaf(ys[(t * k + j) * 8 + c], weights_s[t * k + j], acc);
        out[(int64_t)t * N + j0 + c] = (bf16_t)acc;
    }
}

template <int NL, bool NESTED>
int launch_down_combine(const bf16_t *h, const int32_t *inv, const int64_t *idx, const bf16_t *weights, const Nf4Matrix &w,
                        bf16_t *out, int R, int k, int N, int K, int E, hipStream_t stream) {
    constexpr int lds = kGemvTable + (256 + kDownRows * 9) * 4;
    auto *kernel = nf4_down_combine_kernel<NL, NESTED>;
    static PerDeviceOnce attr;
    static std::atomic<int> static_lds{-1};
    const hipError_t e = attr.run([&] {
        hipFuncAttributes fa;
        const hipError_t e1 = hipFuncGetAttributes(&fa, (const void *)kernel);
        if (e1 != hipSuccess) return e1;
        static_lds.store((int)fa.sharedSizeBytes, std::memory_order_release);
        return hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    });
    if (e != hipSuccess) return (int)e;
    if (static_lds.load(std::memory_order_acquire) != 0) return MFL_ERR_UNSUPPORTED;
    kernel<<<(unsigned)(N / 8), kGemvThreads, lds, stream>>>(h, inv, idx, weights, w, out, R, k, N, K, E);
    return launch_status();
}

template <int CL, int NL, int ROWS, bool WIDE>
int dispatch_gemv(const bf16_t *x, const int32_t *row_idx, int idx_div, const Nf4Matrix &w0, const Nf4Matrix &w1,
                  bool glu, const void *m_sizes, int ms_i64, void *y, void *e_out, void *g_out, int64_t R, int N,
                  int K, int E, int out_dtype, hipStream_t stream) {
// (four scales a column of 8-bit values and factors: two columns ahead, four spill: 128 rows, K = 1024, gated 84 -> 62 us)
#define MFL_GEMV(GLU, TO, Y, EO, GO)                                                                               \
    (w0.nested() ? launch_gemv<CL, NL, ROWS, ((NL <= (WIDE ? 4 : 3) && (GLU || CL < 64)) ? 4 : 2), GLU, WIDE, true, TO>( \
                       x, row_idx, idx_div, w0, w1, m_sizes, ms_i64, Y, EO, GO, R, N, K, E, stream)                 \
                 : launch_gemv<CL, NL, ROWS, ((NL <= 4 && (GLU || CL < 64)) ? 4 : 2), GLU, WIDE, false, TO>(                       \
                       x, row_idx, idx_div, w0, w1, m_sizes, ms_i64, Y, EO, GO, R, N, K, E, stream))
    if (glu) return MFL_GEMV(true, bf16_t, (bf16_t *)y, (bf16_t *)e_out, (bf16_t *)g_out);
    if (out_dtype == MFL_BF16) return MFL_GEMV(false, bf16_t, (bf16_t *)y, nullptr, nullptr);
    return MFL_GEMV(false, float, (float *)y, nullptr, nullptr);
#undef MFL_GEMV
}

}  // namespace

int gemm_nf4_gemv(const bf16_t *x, const int32_t *row_idx, int idx_div, const Nf4Matrix &w0, const Nf4Matrix &w1,
                  bool glu, const void *m_sizes, int ms_i64, void *y, void *e_out, void *g_out, int64_t R, int N,
                  int K, int E, int out_dtype, hipStream_t stream) {
    if (R <= 0 || R > 2 * (int64_t)E || E > 2048) return MFL_ERR_UNSUPPORTED;  // a few rows per expert only
    const bool half = K <= 1024;
    const int smallest = glu && w1.bs_shift < w0.bs_shift ? w1.bs_shift : w0.bs_shift;
    const GemvLayout l = gemv_layout(K, N, smallest);
    if (2 * R > (int64_t)E * gemv_half_rows(K, l, smallest)) return MFL_ERR_UNSUPPORTED;
    if (K % 32 != 0 || K > 2048 || K <= 256) return MFL_ERR_UNSUPPORTED;
    // whole units (32 columns; 16 in the gated form with 64 lanes to a column); fewer than 2^31 units in all
    if (N % ((glu && !half) ? 16 : 32) != 0 || N > (1 << 18)) return MFL_ERR_UNSUPPORTED;
    const Nf4Matrix *mats[2] = {&w0, &w1};
    for (int cb = 0; cb < (glu ? 2 : 1); ++cb) {
        const Nf4Matrix &m = *mats[cb];
        // a lane's 8 weights under one scale, and every column starts a quantisation block
        if (m.bs_shift < 3 || (K & ((1 << m.bs_shift) - 1)) != 0) return MFL_ERR_UNSUPPORTED;
        if (!aligned(m.absmax, 4) || !aligned(m.wq, 16)) return MFL_ERR_UNSUPPORTED;
        if (m.nested() != w0.nested() || (m.nested() && (((int64_t)E * N * K) >> m.bs_shift) > 0x7fffffff))
            return MFL_ERR_UNSUPPORTED;
    }
    if (!aligned(x, 16)) return MFL_ERR_UNSUPPORTED;
#define MFL_GEMV_D(CL, NL, WIDE) \
    dispatch_gemv<CL, NL, 2, WIDE>(x, row_idx, idx_div, w0, w1, glu, m_sizes, ms_i64, y, e_out, g_out, R, N, K, E, out_dtype, stream)
    if (l.lanes == 64) return l.side_by_side ? MFL_GEMV_D(64, 4, true) : MFL_GEMV_D(64, 4, false);
    if (l.lanes == 16) return l.dwords == 6 ? MFL_GEMV_D(16, 6, true) : MFL_GEMV_D(16, 4, true);
    if (l.dwords == 3) return MFL_GEMV_D(32, 3, false);
    return l.side_by_side ? MFL_GEMV_D(32, 4, true) : MFL_GEMV_D(32, 4, false);
#undef MFL_GEMV_D
}

int gemm_nf4_down_combine(const bf16_t *h, const int32_t *inv, const int64_t *idx, const bf16_t *weights, const Nf4Matrix &w,
                          bf16_t *out, int64_t T, int k, int N, int K, int E, hipStream_t stream) {
    // (the sizes at which the plain product runs on the same layout of a column's weights: the same bits.  Ahead of the two
    // kernels at every number of selections: a block of 128 experts, 2048 x 768, 1 / 4 / 8 / 12 / 16 of them, fp32 scales, all
    // its kernels: 17.5 / 20.1 / 24.8 / 26.8 / 28.6 -> 13.4 / 15.1 / 19.2 / 22.2 / 23.6 us; 16 of one token 32.7 -> 24.8)
    const int64_t R = T * k;
    if (R <= 0 || R > kDownRows || N % 64 != 0 || N > (1 << 18)) return MFL_ERR_UNSUPPORTED;
    if (K <= 256 || K > 768 || K % 64 != 0) return MFL_ERR_UNSUPPORTED;
    const GemvLayout l = gemv_layout(K, N, w.bs_shift);
    if (l.lanes != 16 || !l.side_by_side || (K & ((1 << w.bs_shift) - 1)) != 0) return MFL_ERR_UNSUPPORTED;
    if (2 * R > (int64_t)E * gemv_half_rows(K, l, w.bs_shift)) return MFL_ERR_UNSUPPORTED;
    if (!aligned(h, 16) || !aligned(w.wq, 16) || !aligned(w.absmax, 4) || !aligned(out, 2)) return MFL_ERR_UNSUPPORTED;
#define MFL_DOWN(NL, NESTED) \
    launch_down_combine<NL, NESTED>(h, inv, idx, weights, w, out, (int)R, k, N, K, E, stream)
    if (l.dwords == 6) return w.nested() ? MFL_DOWN(6, true) : MFL_DOWN(6, false);
    return w.nested() ? MFL_DOWN(4, true) : MFL_DOWN(4, false);
#undef MFL_DOWN
}

}  // namespace mfl
