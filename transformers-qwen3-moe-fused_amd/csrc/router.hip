// The router projection: logits (T, E) = x (T, H) w (E, H)^T for few tokens, and the gradient of its weight,
// dw (E, H) = dlogits (T, E)^T x (T, H), for any number of them; bf16 in and out, fp32 sums.  Both outputs are small
// and their reductions long (2048 and the number of tokens), so both split the reduction.
#include "ops.h"
#include "pipe_parts.h"

namespace mfl {

namespace {

// ---- forward: a workgroup of eight waves owns 16 tokens x 16 experts; the waves take the reduction's pieces of 64 in
// turn, straight from memory (a lane holds 16 consecutive elements of its token and of its expert), and meet in LDS.
// What bounds it is one round trip to memory: 3.8 us at 1 token, 5.3 at 16 to 512 (E = 128, H = 2048).  The library
// product it stands in for takes 5.3 us on the device, and 19 us of the host's time against 5, which at these sizes is
// what counts.  More tokens re-read the weights once per 16 of them (15 against 7 us at 2048 tokens).
constexpr int kFwdWaves = 8;

template <typename TO>
__global__ __launch_bounds__(kFwdWaves * 64) void router_fwd_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ w,
                                                                   TO *__restrict__ out, int T, int H, int E) {
    __shared__ float part[kFwdWaves][4][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int e0 = blockIdx.x * 16, t0 = blockIdx.y * 16;
    const bf16_t *const wp = w + (int64_t)(e0 + r < E ? e0 + r : E - 1) * H + g * 16;
    const bf16_t *const xp = x + (int64_t)(t0 + r < T ? t0 + r : T - 1) * H + g * 16;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    const int pieces = H / 64;
    constexpr int U = 4;  // pieces in flight
    for (int c0 = wave; c0 < pieces; c0 += kFwdWaves * U) {
        bf16x8 wf[U][2], xf[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int c = c0 + u * kFwdWaves;
            if (c >= pieces) c = c0;  // loaded, not multiplied
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                wf[u][h] = *(const bf16x8 *)(wp + c * 64 + h * 8);
                xf[u][h] = *(const bf16x8 *)(xp + c * 64 + h * 8);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u * kFwdWaves >= pieces) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u][h], wf[u][h], acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) part[wave][u][lane] = acc[u];
    __syncthreads();
    if (tid < 256) {
        const int u = tid >> 6;
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < kFwdWaves; ++v) s += part[v][u][lane];
        // lane l holds expert l % 16 of tokens 4 (l / 16) + u
        const int t = t0 + 4 * g + u, e = e0 + r;
        if (t < T && e < E) out[(int64_t)t * E + e] = from_f32<TO>(s);
    }
}

// ---- weight gradient: the tokens are cut into as many parts as fill the chip; a workgroup of four waves multiplies its
// part into a 128 x 128 tile of the result (steps of 32 tokens through a ring of four stages, both operands read with
// transposing LDS reads) and leaves fp32 sums, which a second kernel adds up.  8192 / 4096 / 1024 tokens:
// 19 / 16 / 10.5 us against 67 / 34 / 12.3 of the library product, which gives the 128 x 2048 output to 32 workgroups
// (9.0 against 6.7 at 256).
constexpr int kDwTile = 128, kDwStep = 32, kDwRing = 4;
typedef Stage<kDwTile, kDwStep, false> DwStage;

__global__ __launch_bounds__(256) void router_dw_kernel(const bf16_t *__restrict__ d, const bf16_t *__restrict__ x,
                                                        float *__restrict__ out, int T, int H, int E, int per_part) {
    constexpr int LOADS = DwStage::kWaveLoads / 4;  // copies per wave, operand and stage
    __shared__ __attribute__((aligned(1024))) unsigned char smem[kDwRing * 2 * DwStage::kBytes];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int h0 = blockIdx.x * kDwTile, e0 = blockIdx.y * kDwTile;
    const int t_begin = blockIdx.z * per_part;
    const int t_end = t_begin + per_part < T ? t_begin + per_part : T;
    const int e_lim = E - e0 < kDwTile ? E - e0 : kDwTile, h_lim = H - h0 < kDwTile ? H - h0 : kDwTile;
    FragOffsets<kDwTile, kDwStep, false, 2> fo_a, fo_b;
    fo_a.init(wm * 64, 32, lane);
    fo_b.init(wn * 64, 32, lane);
    int row[LOADS];
    int64_t off_d[LOADS], off_x[LOADS];
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int load = wave * LOADS + q;
        row[q] = DwStage::row_of(load, lane);
        off_d[q] = lane_src_offset<kDwTile, kDwStep, false>(load, lane, E, e_lim);
        off_x[q] = lane_src_offset<kDwTile, kDwStep, false>(load, lane, H, h_lim);
    }
    const int steps = ceil_div(t_end - t_begin, kDwStep);
    // rows past the last token: zeros in both operands (an infinity of a row read again would turn into NaN)
    auto issue = [&](int s) {
        unsigned char *const base = smem + (s % kDwRing) * 2 * DwStage::kBytes;
        const int t0 = t_begin + s * kDwStep;
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            const bool in = t0 + row[q] < t_end;
            const unsigned char *const pd = in ? (const unsigned char *)(d + (int64_t)t0 * E + e0) + off_d[q]
                                               : (const unsigned char *)&g_zero_chunk;
            const unsigned char *const px = in ? (const unsigned char *)(x + (int64_t)t0 * H + h0) + off_x[q]
                                               : (const unsigned char *)&g_zero_chunk;
            copy_to_lds<0, true>(pd, base + (wave * LOADS + q) * 1024);
            copy_to_lds<0, true>(px, base + DwStage::kBytes + (wave * LOADS + q) * 1024);
        }
    };
    floatx16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int u = 0; u < 16; ++u) acc[i][j][u] = 0.f;
#pragma unroll
    for (int s = 0; s < kDwRing - 1; ++s)
        if (s < steps) issue(s);
    for (int s = 0; s < steps; ++s) {
        // my copies of step s have landed: at most those of the steps behind it are outstanding
        const int behind = steps - 1 - s < kDwRing - 2 ? steps - 1 - s : kDwRing - 2;
        if (behind == 2) wait_vmcnt<2 * 2 * LOADS>();
        else if (behind == 1) wait_vmcnt<2 * LOADS>();
        else wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // my reads of the stage before are done
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (s + kDwRing - 1 < steps) issue(s + kDwRing - 1);
        const unsigned char *const base = smem + (s % kDwRing) * 2 * DwStage::kBytes;
#pragma unroll
        for (int ks = 0; ks < kDwStep / 16; ++ks) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) fa[i] = fo_a.load(base, i, ks);
#pragma unroll
            for (int j = 0; j < 2; ++j) fb[j] = fo_b.load(base + DwStage::kBytes, j, ks);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    }
    // a lane holds expert row lane % 32, four groups of four consecutive columns per block
    float *const o = out + (int64_t)blockIdx.z * E * H;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = wm * 64 + i * 32 + (lane & 31);
        if (e >= e_lim) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = wn * 64 + j * 32 + 8 * q + 4 * (lane >> 5);
                if (c >= h_lim) continue;  // H is a multiple of 8
                floatx4 v;
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = acc[i][j][4 * q + u];
                *(floatx4 *)(o + (int64_t)(e0 + e) * H + h0 + c) = v;
            }
    }
}

__global__ __launch_bounds__(256) void router_dw_sum_kernel(const float *__restrict__ part, bf16_t *__restrict__ dw, int64_t n,
                                                            int parts) {
    const int64_t i = (blockIdx.x * 256ll + threadIdx.x) * 4;
    if (i >= n) return;
    floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int p = 0; p < parts; ++p) s += *(const floatx4 *)(part + p * n + i);
    bf16x4 o;
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] = (bf16_t)s[u];
    *(bf16x4 *)(dw + i) = o;
}

// parts of at least 256 tokens, whole steps, up to about one workgroup per CU
int dw_parts(int64_t T, int H, int E) {
    const int tiles = ceil_div(H, kDwTile) * ceil_div(E, kDwTile);
    int64_t parts = ceil_div(device_info().cu_count, tiles);
    if (parts > (T + 255) / 256) parts = (T + 255) / 256;
    return parts < 1 ? 1 : (int)parts;
}

}  // namespace

int router_fwd(const void *x, const void *w, void *logits, int64_t T, int H, int E, int out_dtype, hipStream_t stream) {
    if (H % 64 != 0 || T > (1 << 20) || !aligned(x, 16) || !aligned(w, 16)) return MFL_ERR_UNSUPPORTED;
    const dim3 grid(ceil_div(E, 16), ceil_div((int)T, 16));
#define MFL_RF(TO)                                                                                                   \
    router_fwd_kernel<TO><<<grid, kFwdWaves * 64, 0, stream>>>((const bf16_t *)x, (const bf16_t *)w, (TO *)logits, (int)T, \
                                                               H, E)
    if (out_dtype == MFL_F32) MFL_RF(float);
    else if (out_dtype == MFL_BF16) MFL_RF(bf16_t);
    else return MFL_ERR_UNSUPPORTED;
#undef MFL_RF
    return launch_status();
}

size_t router_dw_workspace(int64_t T, int H, int E) {
    if (H % 8 != 0 || E % 8 != 0) return 0;
    return (size_t)dw_parts(T, H, E) * E * H * sizeof(float);
}

int router_dw(const void *x, const void *dlogits, void *dw, int64_t T, int H, int E, void *workspace, size_t ws_bytes,
              hipStream_t stream) {
    if (H % 8 != 0 || E % 8 != 0 || T > 0x7fffffff - 4096) return MFL_ERR_UNSUPPORTED;
    if (!aligned(x, 16) || !aligned(dlogits, 16) || !aligned(dw, 8)) return MFL_ERR_UNSUPPORTED;
    if (!workspace || ws_bytes < router_dw_workspace(T, H, E)) return MFL_ERR_WORKSPACE;
    if (!aligned(workspace, 16)) return MFL_ERR_ALIGN;
    int parts = dw_parts(T, H, E);
    const int per_part = ceil_div(ceil_div((int)T, parts), kDwStep) * kDwStep;
    parts = ceil_div((int)T, per_part);
    router_dw_kernel<<<dim3(ceil_div(H, kDwTile), ceil_div(E, kDwTile), parts), 256, 0, stream>>>(
        (const bf16_t *)dlogits, (const bf16_t *)x, (float *)workspace, (int)T, H, E, per_part);
    const int64_t n = (int64_t)E * H;
    router_dw_sum_kernel<<<(unsigned)((n / 4 + 255) / 256), 256, 0, stream>>>((const float *)workspace, (bf16_t *)dw, n, parts);
    return launch_status();
}

}  // namespace mfl
