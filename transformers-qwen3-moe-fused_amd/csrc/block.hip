// The sparse MoE block after its router projection, forward and backward, as one call each: the launches of
// api.hip's entry points one behind the other, with every intermediate in one buffer of the caller's.  The kernels
// and their results are those of the separate calls.  What it saves is the host's time between the launches: at
// decode sizes the block is a chain of five kernels of 5 to 40 us (on packed weights four up to 16 selections, the down projection
// with the sum over them in one), and preparing each from the caller's language
// (a tensor per output, an autograd node per step) took longer than the kernels run: 118 us of host time against
// 95 us of kernels at 16 tokens on packed weights, 690 us for a training step of a toy block whose kernels take 120.
#include <initializer_list>

#include "common.h"
#include "gemm.h"

namespace mfl {

namespace {

size_t up256(size_t n) { return (n + 255) / 256 * 256; }

// Shapes whose front half (gather, gate, up, SiLU-mul) is one kernel, which keeps the two products to itself
bool front_is_one_kernel(const mfl_moe_block &b) {
    return b.dtype == MFL_BF16 && b.H % 8 == 0 && b.I % 8 == 0 && b.E <= 512;
}

struct Layout {
    size_t idx, w32, sort, inv, counts, weights, route, e, g, h, y, scales, total, route_bytes, scale_bytes;
    int scale_slots;  // written-out scales there is room for: gate and up's, or one after the other the three matrices'
};

// Whether a product (R rows, reduction length K) on these weights needs no room for written-out scales: they are not
// double-quantised, or a decode-sized kernel reads them as they are.  By the sizes: should that kernel refuse the call all
// the same, the block does, and the caller makes the separate calls.
bool scales_as_they_are(const mfl_moe_block &b, const mfl_nf4_weight &w, int K, int rows_per_expert) {
    if (w.absmax_u8 == nullptr) return true;
    return w.blocksize == 64 && K % 128 == 0 && K / 64 <= w.blocksize2 && b.H % 8 == 0 && b.I % 8 == 0 &&
           b.T * b.k <= (int64_t)rows_per_expert * b.E && aligned(w.absmax_u8, 2) && aligned(w.packed, 16) && aligned(b.tokens, 16);
}

Layout layout(const mfl_moe_block &b) {
    const size_t R = (size_t)b.T * b.k, es = dtype_size(b.dtype);
    Layout l = {};
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += up256(bytes);
        return at;
    };
    l.idx = take(R * 8);
    l.w32 = take(R * 4);
    l.sort = take(R * 4);
    l.inv = take(R * 4);
    l.counts = take((size_t)b.E * 4);
    l.weights = take(R * es);
    l.route_bytes = mfl_route_sort_workspace(b.T, b.E, b.k);
    l.route = take(l.route_bytes);
    if (b.training || (b.q_gate == nullptr && !front_is_one_kernel(b))) {
        l.e = take(R * b.I * es);
        l.g = take(R * b.I * es);
    }
    l.h = take(R * b.I * es);
    l.y = take(R * b.H * es);
    if (b.q_gate != nullptr) {
        const mfl_nf4_weight &gate = *b.q_gate, &up = *b.q_up, &down = *b.q_down;
        const bool alike = (gate.absmax_u8 != nullptr) == (up.absmax_u8 != nullptr) && gate.blocksize2 == up.blocksize2;
        const bool front_ok = scales_as_they_are(b, gate, b.H, kNf4StreamGatedRowsPerExpert) &&
                              scales_as_they_are(b, up, b.H, kNf4StreamGatedRowsPerExpert) &&
                              (alike || (gate.absmax_u8 == nullptr && up.absmax_u8 == nullptr));
        l.scale_slots = !front_ok ? 2 : scales_as_they_are(b, down, b.I, kNf4StreamRowsPerExpert) ? 0 : 1;
        size_t most = 0;
        for (const mfl_nf4_weight *w : {b.q_gate, b.q_up, b.q_down}) {
            const size_t bytes = (size_t)((int64_t)b.E * b.H * b.I / w->blocksize) * 4;
            most = bytes > most ? bytes : most;
        }
        l.scale_bytes = up256(most);
        l.scales = take(l.scale_slots * l.scale_bytes);
    }
    l.total = o;
    return l;
}

int check_block(const mfl_moe_block *b) {
    if (!b) return MFL_ERR_NULL;
    if (b->T <= 0 || b->E <= 0 || b->k <= 0 || b->k > b->E || b->k > 64 || b->H <= 0 || b->I <= 0 ||
        b->T * b->k > 0x7fffffff)
        return MFL_ERR_SHAPE;
    if (!dtype_ok(b->dtype) || !dtype_ok(b->logits_dtype)) return MFL_ERR_DTYPE;
    if (b->q_gate != nullptr) {
        if (!b->q_up || !b->q_down) return MFL_ERR_NULL;
        for (const mfl_nf4_weight *w : {b->q_gate, b->q_up, b->q_down})
            if (w->blocksize < 2 || ((int64_t)b->E * b->H * b->I) % w->blocksize != 0) return MFL_ERR_SHAPE;
        if (b->dtype != MFL_BF16 || b->training) return MFL_ERR_UNSUPPORTED;
    }
    return MFL_OK;
}

// Every token's row to the places of its selections (times their weights)
int spread_rows(const mfl_moe_block &b, const void *src, const char *ws, const Layout &l, const void *scale, void *dst,
                void *stream) {
    if (b.k > 1) return mfl_scatter_rows(src, (const int32_t *)(ws + l.inv), b.k, scale, dst, b.T, b.H, b.dtype, stream);
    return mfl_gather_rows(src, (const int32_t *)(ws + l.sort), 1, scale, dst, b.T, b.H, b.dtype, stream);
}

// The matrices (two at most) with the scales of double-quantised ones written out in one launch, matrix i's from out + i *
// scale_bytes on; others as they are
int write_out_scales(const mfl_moe_block &b, std::initializer_list<const mfl_nf4_weight *> from, mfl_nf4_weight *plain,
                     char *out, size_t scale_bytes, void *stream) {
    mfl_nf4_weight nested[2];
    int64_t n[2];
    float *to[2];
    int count = 0, i = 0;
    for (const mfl_nf4_weight *w : from) {
        plain[i] = *w;
        if (w->absmax_u8 != nullptr) {
            nested[count] = *w;
            n[count] = (int64_t)b.E * b.H * b.I / w->blocksize;
            to[count] = (float *)(out + i * scale_bytes);
            plain[i].absmax = to[count];
            plain[i].absmax_tiled = nullptr;
            plain[i].absmax_u8 = nullptr;
            ++count;
        }
        ++i;
    }
    return mfl_nf4_write_out_scales(nested, n, to, count, stream);
}

#define MFL_TRY(call)                \
    do {                             \
        const int rc_ = (call);      \
        if (rc_ != MFL_OK) return rc_; \
    } while (0)

int front(const mfl_moe_block &b, char *ws, const Layout &l, void *stream) {
    const int64_t R = b.T * b.k;
    const int32_t *sort = (const int32_t *)(ws + l.sort), *ms = (const int32_t *)(ws + l.counts);
    void *e = l.e ? ws + l.e : nullptr, *g = l.g ? ws + l.g : nullptr, *h = ws + l.h;
    if (b.q_gate != nullptr) {
        int rc = mfl_glu_fwd_nf4_packed(b.tokens, b.T, sort, b.k, b.q_gate, b.q_up, ms, MFL_I32, h, e, g, R, b.I, b.H, b.E,
                                        b.dtype, stream);
        if (rc == MFL_ERR_UNSUPPORTED && (b.q_gate->absmax_u8 != nullptr || b.q_up->absmax_u8 != nullptr) && l.scale_slots == 2) {
            mfl_nf4_weight w[2];
            MFL_TRY(write_out_scales(b, {b.q_gate, b.q_up}, w, ws + l.scales, l.scale_bytes, stream));
            rc = mfl_glu_fwd_nf4_packed(b.tokens, b.T, sort, b.k, &w[0], &w[1], ms, MFL_I32, h, e, g, R, b.I, b.H, b.E, b.dtype,
                                        stream);
        }
        return rc;
    }
    if (front_is_one_kernel(b)) {
        const int rc = mfl_glu_fwd(b.tokens, b.T, sort, b.k, b.w_gate, b.w_up, ms, MFL_I32, h, e, g, R, b.I, b.H, b.E, b.dtype,
                                   stream);
        if (rc != MFL_ERR_UNSUPPORTED || e == nullptr) return rc;
    }
    void *x = ws + l.y;  // the rows, until the down projection writes its own
    MFL_TRY(spread_rows(b, b.tokens, ws, l, nullptr, x, stream));
    MFL_TRY(mfl_gemm_fwd(x, b.w_gate, ms, MFL_I32, e, R, b.I, b.H, b.E, b.dtype, b.dtype, 1.0f, 0, stream));
    MFL_TRY(mfl_gemm_fwd(x, b.w_up, ms, MFL_I32, g, R, b.I, b.H, b.E, b.dtype, b.dtype, 1.0f, 0, stream));
    return mfl_silu_mul_fwd(e, g, h, R * b.I, b.dtype, stream);
}

int down(const mfl_moe_block &b, char *ws, const Layout &l, void *stream) {
    const int64_t R = b.T * b.k;
    const int32_t *ms = (const int32_t *)(ws + l.counts);
    if (b.q_down == nullptr)
        return mfl_gemm_fwd(ws + l.h, b.w_down, ms, MFL_I32, ws + l.y, R, b.H, b.I, b.E, b.dtype, b.dtype, 1.0f, 0, stream);
    int rc = mfl_gemm_fwd_nf4_packed(ws + l.h, 0, nullptr, 1, b.q_down, ms, MFL_I32, ws + l.y, R, b.H, b.I, b.E, b.dtype,
                                     b.dtype, stream);
    if (rc == MFL_ERR_UNSUPPORTED && b.q_down->absmax_u8 != nullptr && l.scale_slots != 0) {
        mfl_nf4_weight w;
        MFL_TRY(write_out_scales(b, {b.q_down}, &w, ws + l.scales, l.scale_bytes, stream));
        rc = mfl_gemm_fwd_nf4_packed(ws + l.h, 0, nullptr, 1, &w, ms, MFL_I32, ws + l.y, R, b.H, b.I, b.E, b.dtype, b.dtype,
                                     stream);
    }
    return rc;
}

// The down projection and the sum over each token's selections as one launch, where there is a kernel for it
int down_and_combine(const mfl_moe_block &b, const char *ws, const Layout &l, void *out, void *stream) {
    if (b.q_down == nullptr || !b.q_down->packed || !b.q_down->code16 || (b.q_down->blocksize & (b.q_down->blocksize - 1)) != 0)
        return MFL_ERR_UNSUPPORTED;
    const mfl_nf4_weight &w = *b.q_down;
    auto log2_of = [](int v) { return 31 - __builtin_clz((unsigned)v); };
    Nf4Matrix m = {w.packed, w.code16, w.absmax, log2_of(w.blocksize)};
    if (w.absmax_u8 != nullptr) {
        if (!w.code256 || !w.absmax2 || !w.offset || w.blocksize2 < 2 || (w.blocksize2 & (w.blocksize2 - 1)) != 0)
            return MFL_ERR_UNSUPPORTED;
        m.absmax = nullptr;
        m.absmax_u8 = w.absmax_u8, m.code256 = w.code256, m.absmax2 = w.absmax2, m.offset = w.offset;
        m.bs2_shift = log2_of(w.blocksize2);
    } else if (!w.absmax) {
        return MFL_ERR_UNSUPPORTED;
    }
    return gemm_nf4_down_combine((const bf16_t *)(ws + l.h), (const int32_t *)(ws + l.inv), (const int64_t *)(ws + l.idx),
                                 (const bf16_t *)(ws + l.weights), m, (bf16_t *)out, b.T, b.k, b.H, b.I, b.E, (hipStream_t)stream);
}

// What the backward needs besides the forward's buffer: the output gradient's rows (then, in their place, the input
// gradient's), the tokens' rows, dh, de and dg
struct BackLayout {
    size_t dy, x, dh, de, dg, dw, split, total;
};

// Scratch of a weight gradient (E, N, K) with one thin side (8 to 64) whose rows are dealt out evenly over the workgroups;
// 0: the general kernel, whose launch under skewed routing lasts as long as its largest expert.  A step, hidden 2048,
// general against even shares, routing uniform / Zipf 1.25 / Zipf 4:
//   16 experts, side 32, 65536 rows: 815 / 1193 / 1437 against 809 / 810 / 805 us; 16384 rows: 271 / 357 / 405 against
//   292 / 302 / 298; 8192 rows: 263 / 259 / 278 against 285 / 283 / 281 (nothing left to even out);
//   128 experts, side 32, 32768 rows: 477 / 496 / 455 against 441 / 478 / 519;
//   side 64, which leaves the even shares fewer stages: 16 experts, 65536 rows 845 / 1298 / 1607 against 876 / 888 / 874, but
//   128 experts 843 / 865 / 854 against 856 / 971 / 930: from 1024 rows per expert on.
size_t split_bytes(const mfl_moe_block &b, int N, int K) {
    const int64_t R = b.T * b.k;
    if (b.dtype != MFL_BF16 || R < 16384 || ((N < K ? N : K) > 32 && R < (int64_t)1024 * b.E)) return 0;
    return mfl_gemm_dw_split_workspace(R, N, K, b.E);
}

int weight_grad(const mfl_moe_block &b, const void *x, const void *dy, const int32_t *ms, void *dw, int N, int K, void *scratch,
                void *stream) {
    const int64_t R = b.T * b.k;
    const size_t bytes = split_bytes(b, N, K);
    if (bytes != 0 && aligned(dw, 16))
        return mfl_gemm_dw_split(x, dy, ms, MFL_I32, dw, R, N, K, b.E, b.dtype, b.dtype, 1.0f, scratch, bytes, stream);
    return mfl_gemm_dw(x, dy, ms, MFL_I32, dw, R, N, K, b.E, b.dtype, b.dtype, 1.0f, 0, stream);
}

BackLayout back_layout(const mfl_moe_block &b) {
    const size_t R = (size_t)b.T * b.k, es = dtype_size(b.dtype);
    BackLayout l;
    l.dy = 0;
    l.x = l.dy + up256(R * b.H * es);
    l.dh = l.x + up256(R * b.H * es);
    l.de = l.dh + up256(R * b.I * es);
    l.dg = l.de + up256(R * b.I * es);
    l.dw = l.dg + up256(R * b.I * es);
    l.split = l.dw + up256(R * es);
    const size_t down = split_bytes(b, b.H, b.I), front = split_bytes(b, b.I, b.H);
    l.total = l.split + up256(down > front ? down : front);
    return l;
}

}  // namespace

}  // namespace mfl

using namespace mfl;

extern "C" {

size_t mfl_moe_block_workspace(const mfl_moe_block *b) { return check_block(b) == MFL_OK ? layout(*b).total : 0; }

int mfl_moe_block_fwd(const mfl_moe_block *b, void *out, void *workspace, size_t ws_bytes, void *stream) {
    MFL_TRY(check_block(b));
    if (!b->tokens || !b->logits || !out || !workspace) return MFL_ERR_NULL;
    if (b->q_gate == nullptr && (!b->w_gate || !b->w_up || !b->w_down)) return MFL_ERR_NULL;
    if (!aligned(workspace, 256)) return MFL_ERR_ALIGN;
    const Layout l = layout(*b);
    if (ws_bytes < l.total) return MFL_ERR_WORKSPACE;
    char *ws = (char *)workspace;
    MFL_TRY(mfl_route_sort(b->logits, b->logits_dtype, b->T, b->E, b->k, b->renorm, (float *)(ws + l.w32), ws + l.weights,
                           b->dtype, (int64_t *)(ws + l.idx), (int32_t *)(ws + l.counts), (int32_t *)(ws + l.sort),
                           (int32_t *)(ws + l.inv), ws + l.route, l.route_bytes, stream));
    MFL_TRY(front(*b, ws, l, stream));
    const int rc = down_and_combine(*b, ws, l, out, stream);
    if (rc != MFL_ERR_UNSUPPORTED) return rc;
    MFL_TRY(down(*b, ws, l, stream));
    return mfl_combine_rows(ws + l.y, (const int32_t *)(ws + l.inv), ws + l.weights, out, b->T, b->k, b->H, b->dtype, stream);
}

size_t mfl_moe_block_bwd_workspace(const mfl_moe_block *b) { return check_block(b) == MFL_OK ? back_layout(*b).total : 0; }

int mfl_moe_block_bwd(const mfl_moe_block *b, const void *dout, const void *saved, void *d_tokens, void *d_logits,
                      void *d_gate, void *d_up, void *d_down, void *workspace, size_t ws_bytes, void *stream) {
    MFL_TRY(check_block(b));
    if (!b->training || b->q_gate != nullptr) return MFL_ERR_UNSUPPORTED;
    if (!b->tokens || !b->logits || !b->w_gate || !b->w_up || !b->w_down || !dout || !saved || !workspace) return MFL_ERR_NULL;
    if (!aligned(workspace, 256)) return MFL_ERR_ALIGN;
    const Layout l = layout(*b);
    const BackLayout t = back_layout(*b);
    if (ws_bytes < t.total) return MFL_ERR_WORKSPACE;
    const char *fw = (const char *)saved;
    char *ws = (char *)workspace;
    const int64_t R = b->T * b->k;
    const int dt = b->dtype;
    const int32_t *ms = (const int32_t *)(fw + l.counts), *inv = (const int32_t *)(fw + l.inv);
    if (d_logits != nullptr) {
        MFL_TRY(mfl_rows_dot(dout, fw + l.y, inv, ws + t.dw, b->T, b->k, b->H, dt, stream));
        MFL_TRY(mfl_route_softmax_topk_bwd(b->logits, b->logits_dtype, b->T, b->E, b->k, b->renorm,
                                           (const int64_t *)(fw + l.idx), (const float *)(fw + l.w32), ws + t.dw, dt, d_logits,
                                           stream));
    }
    if (d_tokens == nullptr && d_gate == nullptr && d_up == nullptr && d_down == nullptr) return MFL_OK;
    MFL_TRY(spread_rows(*b, dout, fw, l, fw + l.weights, ws + t.dy, stream));
    if (d_down != nullptr)
        MFL_TRY(weight_grad(*b, fw + l.h, ws + t.dy, ms, d_down, b->H, b->I, ws + t.split, stream));
    if (d_tokens == nullptr && d_gate == nullptr && d_up == nullptr) return MFL_OK;
    MFL_TRY(mfl_gemm_dx(ws + t.dy, b->w_down, ms, MFL_I32, ws + t.dh, R, b->I, b->H, b->E, dt, dt, 1.0f, 0, stream));
    MFL_TRY(mfl_silu_mul_bwd(ws + t.dh, fw + l.e, fw + l.g, ws + t.de, ws + t.dg, nullptr, R * b->I, dt, stream));
    if (d_tokens != nullptr) {
        void *dx = ws + t.dy;
        int rc = mfl_gemm_dx_dual(ws + t.de, b->w_gate, ws + t.dg, b->w_up, ms, MFL_I32, dx, R, b->H, b->I, b->E, dt, dt, stream);
        if (rc == MFL_ERR_UNSUPPORTED) {
            MFL_TRY(mfl_gemm_dx(ws + t.de, b->w_gate, ms, MFL_I32, dx, R, b->H, b->I, b->E, dt, dt, 1.0f, 0, stream));
            rc = mfl_gemm_dx(ws + t.dg, b->w_up, ms, MFL_I32, dx, R, b->H, b->I, b->E, dt, dt, 1.0f, 1, stream);
        }
        MFL_TRY(rc);
        MFL_TRY(mfl_combine_rows(dx, inv, nullptr, d_tokens, b->T, b->k, b->H, dt, stream));
    }
    if (d_gate != nullptr || d_up != nullptr) {
        // the replicated, sorted rows again: the forward pass did not keep them
        MFL_TRY(spread_rows(*b, b->tokens, fw, l, nullptr, ws + t.x, stream));
        if (d_gate != nullptr)
            MFL_TRY(weight_grad(*b, ws + t.x, ws + t.de, ms, d_gate, b->I, b->H, ws + t.split, stream));
        if (d_up != nullptr)
            MFL_TRY(weight_grad(*b, ws + t.x, ws + t.dg, ms, d_up, b->I, b->H, ws + t.split, stream));
    }
    return MFL_OK;
}

}  // extern "C"
