// Shape- and type-generic grouped GEMM on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 products, fp32
// sums, at the rate of the vector ALU but without its operand traffic).
//
// This is the path for fp32 / fp16 inputs and for bf16 shapes the bf16 kernels do not take (dimensions that are not
// multiples of 8): every dimension is masked, nothing is assumed about alignment beyond the element size.
//
//   MODE_FWD : c[m, n]    = sum_k a[m, k] * b[e(m), n, k]     a = x (R,K),  b = w (E,N,K)
//   MODE_DX  : c[m, n]    = sum_k a[m, k] * b[e(m), k, n]     a = dy (R,K), b = w (E,K,N)
//   MODE_DW  : c[e, n, k] = sum_{m in e} a[m, n] * b[m, k]    a = dy (R,N), b = x (R,K)
//
// Operands go global -> registers (the next step's, while the present one is multiplied) -> LDS as fp32.  One LDS
// stage and two barriers a step: what hides the loads is the number of workgroups on a CU (six of the 16-row tile,
// 24 KiB each), not a second stage.
#include "common.h"
#include "gemm.h"

namespace mfl {

namespace {

constexpr int kThreads = 256;
constexpr int kPad = 4;  // floats: rows stay 16-byte aligned and 16 consecutive rows start in 16 different bank quads

// An operand tile of BI rows (output side) by BK reduction elements.
//   RC (reduction-contiguous): element (i, r) at base[i * ld + r], in LDS at [i][r]
//   RS (reduction-strided):    element (i, r) at base[r * ld + i], in LDS at [r][i]
template <typename TI, int BI, int BK, bool RC, int VEC, bool NT = false>
struct Operand {
    static constexpr int kRow = RC ? BK : BI;                  // contiguous elements of a tile row
    static constexpr int kStride = kRow + kPad;                // floats
    static constexpr int kFloats = (RC ? BI : BK) * kStride;
    static constexpr int kGroups = BI * BK / 4;                // groups of four contiguous elements
    static constexpr int kPerThread = (kGroups + kThreads - 1) / kThreads;
    floatx4 v[kPerThread];

    __device__ __forceinline__ void load(const TI *base, int64_t ld, int i0, int i_end, int r0, int r_end, int tid) {
#pragma unroll
        for (int q = 0; q < kPerThread; ++q) {
            const int g = q * kThreads + tid;
            const int row = g / (kRow / 4), col = (g % (kRow / 4)) * 4;
            const int i = i0 + (RC ? row : col), r = r0 + (RC ? col : row);
            const TI *p = base + (RC ? (int64_t)i * ld + r : (int64_t)r * ld + i);
            v[q] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (kGroups % kThreads != 0 && g >= kGroups) continue;
            if constexpr (VEC == 4) {  // the contiguous dimension is a multiple of four: a group is inside or outside
                if (i < i_end && r < r_end) {
                    typedef __attribute__((ext_vector_type(4))) TI vec_t;
                    const vec_t t = NT ? __builtin_nontemporal_load((const vec_t *)p) : *(const vec_t *)p;
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[q][u] = to_f32(t[u]);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i + (RC ? 0 : u) < i_end && r + (RC ? u : 0) < r_end) v[q][u] = to_f32(p[u]);
            }
        }
    }
    __device__ __forceinline__ void store(float *lds, int tid) const {
#pragma unroll
        for (int q = 0; q < kPerThread; ++q) {
            const int g = q * kThreads + tid;
            if (kGroups % kThreads != 0 && g >= kGroups) continue;
            *(floatx4 *)(lds + (g / (kRow / 4)) * kStride + (g % (kRow / 4)) * 4) = v[q];
        }
    }
    // The lane's values of four matrix instructions: reduction elements k + 4 * (lane / 16) + 0..3 of row i + lane % 16
    // (which of the 16 elements of a chunk goes to which instruction is the same for both operands, so free).
    __device__ static __forceinline__ floatx4 frag(const float *lds, int i, int k, int lane) {
        const int row = i + (lane & 15), r = k + (lane >> 4) * 4;
        if constexpr (RC) return *(const floatx4 *)(lds + row * kStride + r);
        floatx4 f;  // four rows apart, the lane groups of a read lie 16 banks apart: no conflicts
#pragma unroll
        for (int u = 0; u < 4; ++u) f[u] = lds[(r + u) * kStride + row];
        return f;
    }
};

// (expert, first row, rows) of the slot-th tile of BM rows, by prefix sums over the experts 64 at a time.
// false: the slot lies past the last tile.  Every wave does it for itself; the row counts come from the cache.
template <int BM>
__device__ __forceinline__ bool find_tile(const void *m_sizes, int ms_i64, int E, int slot, int lane, int &expert,
                                          int &tile, int &m_start, int &m_size) {
    int tiles_before = 0, rows_before = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
        const int m = e0 + lane < E ? load_msize(m_sizes, ms_i64, e0 + lane) : 0;
        const int tiles_to = tiles_before + wave_inclusive_scan(ceil_div(m, BM));
        const int rows_to = rows_before + wave_inclusive_scan(m);
        const uint64_t past = __ballot(tiles_to > slot);
        if (past != 0) {
            const int l = __builtin_ctzll(past);
            expert = e0 + l;
            m_size = __builtin_amdgcn_readlane(m, l);
            m_start = __builtin_amdgcn_readlane(rows_to, l) - m_size;
            tile = slot - (__builtin_amdgcn_readlane(tiles_to, l) - ceil_div(m_size, BM));
            return true;
        }
        tiles_before = wave_last(tiles_to), rows_before = wave_last(rows_to);
    }
    return false;
}

// rows of the experts before e
__device__ __forceinline__ int rows_before_expert(const void *m_sizes, int ms_i64, int e, int lane) {
    int m = 0;
    for (int q = lane; q < e; q += kWave) m += load_msize(m_sizes, ms_i64, q);
    return wave_last(wave_inclusive_scan(m));
}

// NT: the weights are read, a weight gradient is written past the caches (non-temporal; where, is at the launch).
// WM x WN waves over the tile; WK > 1: the waves share the tile and split the reduction (partial sums meet in LDS).
template <typename TI, typename TO, int MODE, int BM, int BN, int WM, int WN, int WK, int BK, int VEC, bool NT>
__global__ __launch_bounds__(kThreads) void gemm_generic_kernel(const TI *__restrict__ a, const TI *__restrict__ b,
                                                                const void *__restrict__ m_sizes, int ms_i64, TO *c,
                                                                int64_t R, int N, int K, int E, float alpha,
                                                                int accumulate, int vec_out) {
    static_assert(WM * WN * WK * kWave == kThreads && BK % (16 * WK) == 0, "four waves");
    constexpr int TM = BM / WM / 16, TN = BN / WN / 16, KW = BK / WK;
    // whether a lane ends with four consecutive columns of one row (16-byte stores) or with four rows of one column
    // (consecutive lanes then store consecutive single elements, where rows are not aligned)
    constexpr bool kRowLanes = VEC == 4;
    typedef Operand<TI, BM, BK, MODE != MODE_DW, VEC> OpA;
    typedef Operand<TI, BN, BK, MODE == MODE_FWD, VEC, NT && MODE != MODE_DW> OpB;
    constexpr int kPartFloats = WM * WN * TM * TN * (WK - 1) * 4 * kWave;  // partial sums of the waves that share a tile
    static_assert(kPartFloats <= OpA::kFloats + OpB::kFloats, "partial sums go where the stage was");
    // weight gradients in fp32 leave by way of LDS, 16 rows of a wave at a time
    constexpr bool kStaged = MODE == MODE_DW && kRowLanes && WK == 1 && TN >= 2 && sizeof(TO) == 4;
    constexpr int kOutRow = TN * 16 + kPad;
    constexpr int kOutFloats = kStaged ? WM * WN * 16 * kOutRow : 0;
    constexpr int kStageFloats = OpA::kFloats + OpB::kFloats;
    __shared__ __align__(16) float smem[kStageFloats > kOutFloats ? kStageFloats : kOutFloats];
    float *As = smem, *Bs = smem + OpA::kFloats;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wn = wave / WK % WN, wm = wave / WK / WN;

    // Output tile [i0, i_end) x [j0, j_end), reduction range [r_begin, r_end).
    int i0, i_end, j0, j_end, r_begin, r_end;
    const TI *b_base = b;
    int64_t lda, ldb, ldc;
    TO *c_base = c;
    if (MODE == MODE_DW) {
        const int e = blockIdx.z;
        r_begin = rows_before_expert(m_sizes, ms_i64, e, lane);
        r_end = r_begin + load_msize(m_sizes, ms_i64, e);
        if ((int64_t)r_end > R) r_end = (int)R;
        i0 = blockIdx.y * BM, i_end = N;
        j0 = blockIdx.x * BN, j_end = K;
        lda = N, ldb = K, ldc = K;
        c_base = c + (int64_t)e * N * K;
    } else {
        int e, tile, m_start, m_size;
        if (!find_tile<BM>(m_sizes, ms_i64, E, blockIdx.x, lane, e, tile, m_start, m_size)) return;
        i0 = m_start + tile * BM;
        i_end = m_start + m_size;
        if ((int64_t)i_end > R) i_end = (int)R;
        j0 = blockIdx.y * BN, j_end = N;
        r_begin = 0, r_end = K;
        lda = K, ldb = MODE == MODE_FWD ? K : N, ldc = N;
        b_base = b + (int64_t)e * N * K;
    }

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    OpA ra;
    OpB rb;
    ra.load(a, lda, i0, i_end, r_begin, r_end, tid);
    rb.load(b_base, ldb, j0, j_end, r_begin, r_end, tid);
    for (int r0 = r_begin; r0 < r_end; r0 += BK) {
        __syncthreads();  // the previous step's fragments have been read
        ra.store(As, tid);
        rb.store(Bs, tid);
        __syncthreads();
        if (r0 + BK < r_end) {
            ra.load(a, lda, i0, i_end, r0 + BK, r_end, tid);
            rb.load(b_base, ldb, j0, j_end, r0 + BK, r_end, tid);
        }
#pragma unroll
        for (int kk = 0; kk < KW; kk += 16) {
            const int k = wk * KW + kk;
            if (r0 + k >= r_end) break;  // the rest of the stage is zeros
            floatx4 fa[TM], fb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = OpA::frag(As, (wm * TM + i) * 16, k, lane);
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[j] = OpB::frag(Bs, (wn * TN + j) * 16, k, lane);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = kRowLanes ? __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][u], fa[i][u], acc[i][j], 0, 0, 0)
                                              : __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i][u], fb[j][u], acc[i][j], 0, 0, 0);
        }
    }

    if constexpr (WK > 1) {
        // of the waves that share a tile, wave t % WK ends with output block t: the others' sums, in wave order
        float *part = smem + (wave / WK) * TM * TN * (WK - 1) * kWave * 4 + lane * 4;
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TM * TN; ++t)
            if (wk != t % WK)
                *(floatx4 *)(part + (t * (WK - 1) + wk - (wk > t % WK)) * kWave * 4) = acc[t / TN][t % TN];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TM * TN; ++t)
            if (wk == t % WK)
#pragma unroll
                for (int s = 0; s < WK - 1; ++s)
                    acc[t / TN][t % TN] += *(const floatx4 *)(part + (t * (WK - 1) + s) * kWave * 4);
    }

    if constexpr (kStaged) {
        if (vec_out && !accumulate) {
            // A lane's four columns of 16 rows are 64 bytes of each row to a store; put together in LDS a store takes 128 to
            // 256 bytes a row, whole lines, and may pass the caches by where the output is larger than they are.
            __syncthreads();  // the last step's fragments have been read
            float *const st = smem + wave * (16 * kOutRow);
            // (asked for again here: what follows from the lane's number otherwise takes two registers through the reduction, which
            // leave room for five workgroups a CU instead of six: 8 experts x 768 x 2048, 1536 tiles, 4096 rows 133 against 119 us.
            // Past the caches, where the write rate is what counts, five are ahead: 128 experts, 1024 rows 134 against 136.)
            int ln = tid & 63;
            if constexpr (!NT) asm volatile("" : "+v"(ln));
#pragma unroll
            for (int i = 0; i < TM; ++i) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    floatx4 o;
#pragma unroll
                    for (int u = 0; u < 4; ++u) o[u] = alpha * acc[i][j][u];
                    *(floatx4 *)(st + (ln & 15) * kOutRow + j * 16 + (ln >> 4) * 4) = o;
                }
                // The same wave reads back what it wrote, and its LDS operations complete in order; that lanes read what other
                // lanes wrote, and overwrite what others read, has to be said (no instructions)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int q = ln; q < 16 * TN * 4; q += kWave) {
                    const int row_l = q / (TN * 4), col_l = (q % (TN * 4)) * 4;
                    const int row = i0 + (wm * TM + i) * 16 + row_l, col = j0 + wn * TN * 16 + col_l;
                    const floatx4 o = *(const floatx4 *)(st + row_l * kOutRow + col_l);
                    if (row >= i_end || col >= j_end) continue;
                    floatx4 *const p = (floatx4 *)(c_base + (int64_t)row * ldc + col);
                    if constexpr (NT)
                        __builtin_nontemporal_store(o, p);
                    else
                        *p = o;
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if (WK > 1 && wk != (i * TN + j) % WK) continue;
            const int across = lane & 15, along = (lane >> 4) * 4;
            const int row = i0 + (wm * TM + i) * 16 + (kRowLanes ? across : along);
            const int col = j0 + (wn * TN + j) * 16 + (kRowLanes ? along : across);
            TO *p = c_base + (int64_t)row * ldc + col;
            if (kRowLanes && vec_out) {
                if (row >= i_end || col >= j_end) continue;
                typedef __attribute__((ext_vector_type(4))) TO vec_t;
                vec_t o;
                if (accumulate) o = *(const vec_t *)p;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    float v = alpha * acc[i][j][u];
                    if (accumulate) v += to_f32(o[u]);
                    o[u] = from_f32<TO>(v);
                }
                *(vec_t *)p = o;
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (row + (kRowLanes ? 0 : u) >= i_end || col + (kRowLanes ? u : 0) >= j_end) continue;
                    TO *q = p + (kRowLanes ? u : u * ldc);
                    float v = alpha * acc[i][j][u];
                    if (accumulate) v += to_f32(*q);
                    *q = from_f32<TO>(v);
                }
            }
        }
    }
}

struct Args {
    const void *a, *b, *m_sizes;
    void *c;
    int64_t R;
    int ms_i64, N, K, E, accumulate, vec_out;
    float alpha;
    hipStream_t stream;
};

template <typename TI, typename TO, int MODE, int BM, int BN, int WM, int WN, int WK, int BK, int VEC>
int launch_tile(const Args &g) {
    dim3 grid;
    if (MODE == MODE_DW) {
        if (ceil_div(g.N, BM) > 65535 || g.E > 65535) return MFL_ERR_UNSUPPORTED;
        grid = dim3(ceil_div(g.K, BN), ceil_div(g.N, BM), g.E);
    } else {
        const int64_t slots = (g.R + BM - 1) / BM + g.E;
        if (slots > 0x7fffffff || ceil_div(g.N, BN) > 65535) return MFL_ERR_UNSUPPORTED;
        grid = dim3((unsigned)slots, ceil_div(g.N, BN), 1);
    }
    // Past the caches: matrices larger than the 256 MB of the last one.  A weight gradient, because its own writes, written
    // back behind it, cost the kernels after it more than it gained; the weights where nearly every expert's rows are one
    // tile and each weight is read once.  Rows of whole lines only: a line that two stores fill, or two loads take, moves
    // twice.  fp32, 128 experts of 8 rows, 768 x 2048 (805 MB), forward / input gradient / weight gradient and the three in
    // turn: 154 / 159 / 177, 559 us; with the gradient's rows put together in LDS 154 / 159 / 147, 507; that past the caches
    // 154 / 159 / 126, 446; the weights too 145 / 147 / 126, 411.  64 experts (403 MB) 293 -> 230.  Rows of 6048 bytes: weight
    // gradient 61 -> 96, input gradient 76 -> 83.  Experts with a second tile: input gradient at 16 rows per expert 187 ->
    // 248, at 32 (32-row tiles) 231 -> 269; at 8 under Zipf(1) routing 155 -> 171, the three in turn 549 -> 474.  Of the weights
    // what counts is what is read, at most an expert's a row: 64 rows over 160 experts of 544 x 1056, which fit, 27 -> 29 past the
    // caches.
    constexpr bool kNt = VEC == 4 && sizeof(TI) == 4 && (MODE == MODE_DW || BM <= 32);
    [[maybe_unused]] const void *const streamed = MODE == MODE_DW ? g.c : g.b;
    const int64_t matrices = MODE != MODE_DW && g.R < g.E ? g.R : g.E;
    [[maybe_unused]] const bool nt = matrices * g.N * g.K * 4 > ((int64_t)256 << 20) && aligned(streamed, 128) &&
                                     (MODE == MODE_DX ? g.N : g.K) % 32 == 0 &&
                                     (MODE == MODE_DW || 4 * g.R <= (int64_t)3 * BM * g.E);
    auto *kernel = gemm_generic_kernel<TI, TO, MODE, BM, BN, WM, WN, WK, BK, VEC, false>;
    if constexpr (kNt)
        if (nt) kernel = gemm_generic_kernel<TI, TO, MODE, BM, BN, WM, WN, WK, BK, VEC, true>;
    kernel<<<grid, kThreads, 0, g.stream>>>((const TI *)g.a, (const TI *)g.b, g.m_sizes, g.ms_i64, (TO *)g.c, g.R, g.N, g.K,
                                            g.E, g.alpha, g.accumulate, g.vec_out);
    return launch_status();
}

// Tiles, with fp32 times at 128 experts, K = 2048, N = 768 (us; the plain FMA kernel that stood here in brackets):
// * up to 16 rows per expert the product streams the weights: 16-row tiles whose waves split the reduction, so that a
//   step asks for 512 consecutive bytes of every weight row and 24 KiB workgroups keep 96 KiB a CU in flight: 145 us
//   forward at 8 rows per expert = 5.6 TB/s (712), 147 dX (533); 64 x 64 tiles with the waves side by side: 285.
// * up to 48, and where 64-row tiles would leave CUs without a second and third workgroup, 32 x 64 tiles: 191 us
//   forward at 24 rows per expert (746; 64 x 64 tiles 275, 16-row tiles 295), 154 us at 8 experts of 512 rows (518;
//   64 x 64 166).
// * beyond, 64 x 64 tiles: 373 us at 64 rows per expert (1584; 128 x 128 tiles 392, whose 64 accumulators and 32
//   registers in transit leave two workgroups a CU).
// * the weight gradient writes more than it reads up to about 100 rows per expert: 64 x 128 tiles and 16-row steps,
//   126 us at 8 rows per expert = 6.4 TB/s (294; before its rows left as whole lines 177, with 32-row steps 225, the zeros
//   of a half-empty stage cost as much as rows do); outputs of at most 16 rows per expert (N: the rank in the gradient of an adapter's A) take
//   16-row tiles.
// * short reductions (adapter ranks, toy sizes) leave most of a 64- or 128-wide step empty: 16-wide steps.  16000 rows of 8
//   experts, 1500 outputs, reduction 8 / 32 / 64 / 128: 64 x 64 tiles 22.0 / 31.0 / 46 / 75 us (64-wide steps 34.9 / 44.5 / 54 /
//   84, the kernel before 28.5 / 57 / 100 / 182); few rows 32 x 64 tiles (128 experts of 8 rows, 2048 outputs, reduction 16: 10.5
//   us, 16-row tiles 23.9).  Where the output's rows are not aligned either, the stores decide: operands loaded one by one leave
//   a lane with four rows of a column, and a store's lanes next to each other (8000 rows, 1001 outputs, reduction 8: 11.3 against
//   22.4 us, 13.8 before; at 32 on 32 x 64 tiles 18.3 against 24.7).
// * fp16 in odd sizes is bound by its single two-byte loads: 32 x 64 tiles, waves side by side (11311 rows of 8 experts, 1161 x
//   793: 507 us; 64 x 64 588; before 530).
// * weight gradients of a few rows per expert only store: smaller tiles, more of them (1 expert of 4 rows, 4096 x 4096: 15.6
//   against 19.5 us, 16.6 before; 128 experts, 64 rows, 768 x 2048: 139 against 191).
template <typename TI, typename TO, int MODE, int VEC>
int launch_mode(const Args &g) {
    if (MODE == MODE_DW) {
        if (g.N <= 16) return launch_tile<TI, TO, MODE, 16, 64, 1, 4, 1, 32, VEC>(g);
        const bool few = g.R <= (int64_t)4 * g.E || (g.R <= (int64_t)16 * g.E && (int64_t)g.E * g.N * g.K <= 1 << 25);
        if (g.N >= 64 && g.K >= 128 && !few) return launch_tile<TI, TO, MODE, 64, 128, 2, 2, 1, 16, VEC>(g);
        if (g.N >= 64 && g.K >= 128) return launch_tile<TI, TO, MODE, 64, 64, 2, 2, 1, 16, VEC>(g);
        return launch_tile<TI, TO, MODE, 64, 64, 2, 2, 1, 32, VEC>(g);
    } else {
        const bool few_tiles = (g.R / 64 + g.E) * ceil_div(g.N, 64) < 4 * device_info().cu_count;
        const bool few = g.R <= (int64_t)48 * g.E || few_tiles;
        if (VEC == 1 && !g.vec_out && g.K > 16 && g.K <= 32) return launch_tile<TI, TO, MODE, 32, 64, 2, 2, 1, 32, VEC>(g);
        if (g.K <= 32 && few) return launch_tile<TI, TO, MODE, 32, 64, 2, 2, 1, 16, VEC>(g);
        if (g.K <= 128 && !few) return launch_tile<TI, TO, MODE, 64, 64, 2, 2, 1, 16, VEC>(g);
        // (their 32 columns would be more tiles than a grid has rows past two million outputs)
        if (g.R <= (int64_t)16 * g.E && ceil_div(g.N, 32) <= 65535) return launch_tile<TI, TO, MODE, 16, 32, 1, 1, 4, 128, VEC>(g);
        if (VEC == 1 && sizeof(TI) == 2 && !few_tiles) return launch_tile<TI, TO, MODE, 32, 64, 2, 2, 1, 32, VEC>(g);
        if (few) return launch_tile<TI, TO, MODE, 32, 64, 1, 2, 2, 64, VEC>(g);
        return launch_tile<TI, TO, MODE, 64, 64, 2, 1, 2, 64, VEC>(g);
    }
}

template <typename TI, typename TO>
int launch_generic(int mode, const Args &g) {
    // groups of four elements: every contiguous dimension that is read has to be a multiple of four
    const size_t align = 4 * sizeof(TI);
    bool vec = aligned(g.a, align) && aligned(g.b, align) && g.K % 4 == 0 && (mode == MODE_FWD || g.N % 4 == 0);
    if (mode != MODE_DW && g.K <= 32 && !g.vec_out) vec = false;  // short reductions: the stores decide
    if (vec) {
        if (mode == MODE_FWD) return launch_mode<TI, TO, MODE_FWD, 4>(g);
        if (mode == MODE_DX) return launch_mode<TI, TO, MODE_DX, 4>(g);
        return launch_mode<TI, TO, MODE_DW, 4>(g);
    }
    if (mode == MODE_FWD) return launch_mode<TI, TO, MODE_FWD, 1>(g);
    if (mode == MODE_DX) return launch_mode<TI, TO, MODE_DX, 1>(g);
    return launch_mode<TI, TO, MODE_DW, 1>(g);
}

}  // namespace

int gemm_generic(int mode, const void *a, const void *b, const void *m_sizes, int ms_i64, void *c, int64_t R, int N,
                 int K, int E, int in_dtype, int out_dtype, float alpha, int accumulate, hipStream_t stream) {
    const int ldc = mode == MODE_DW ? K : N;
    const int vec_out = ldc % 4 == 0 && aligned(c, 4 * dtype_size(out_dtype));
    const Args g = {a, b, m_sizes, c, R, ms_i64, N, K, E, accumulate, vec_out, alpha, stream};
    int rc = MFL_ERR_DTYPE;
    MFL_DISPATCH_FLOAT(in_dtype, TI, MFL_DISPATCH_FLOAT(out_dtype, TO, rc = (launch_generic<TI, TO>(mode, g))));
    return rc;
}

}  // namespace mfl
