// One Transformer block, backwards, in one call: the launches of lbi_gated_mlp_pullback, lbi_small_product, lbi_weight_gradient, lbi_rmsnorm_pullback,
// lbi_attn_pullback, lbi_attn_qkv_conv_pullback (and of the parameter gradients) one after the other, on buffers of one workspace.
//
// For blocks whose products are all small ones.  A block is nine launches of a few microseconds each (nineteen with the parameter
// gradients), and issued one by one from Python each takes 7-10 us of host time, which is what such a call waited for.
#include "lbi_common.h"

namespace lbi {
namespace region_layer {
namespace {

// fp32 values rounded to the storage type, for up to three arrays that lie one behind the other.
struct CastTargets {
    void* out[3];
    int64_t end[3];
};
template <typename T> __device__ __forceinline__ T narrow(float x);
template <> __device__ __forceinline__ _Float16 narrow(float x) { return (_Float16)x; }
template <> __device__ __forceinline__ bf16_raw narrow(float x) { return bf16_raw{f32_to_bf16_bits(x)}; }

template <typename T>
__global__ __launch_bounds__(256) void cast_kernel(const float* __restrict__ in, CastTargets to) {
    for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < to.end[2]; i += (int64_t)gridDim.x * 256) {
        const int which = i < to.end[0] ? 0 : i < to.end[1] ? 1 : 2;
        const int64_t from = which == 0 ? 0 : to.end[which - 1];
        static_cast<T*>(to.out[which])[i - from] = narrow<T>(in[i]);
    }
}

int cast(const float* in, const CastTargets& to, int dtype, hipStream_t stream) {
    const int64_t blocks = (to.end[2] + 255) / 256;
    const dim3 grid((unsigned)(blocks < 4096 ? blocks : 4096));
    if (dtype == LBI_F16) hipLaunchKernelGGL(cast_kernel<_Float16>, grid, dim3(256), 0, stream, in, to);
    else hipLaunchKernelGGL(cast_kernel<bf16_raw>, grid, dim3(256), 0, stream, in, to);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

// Pieces of the workspace, 256-byte aligned, handed out in order.
struct Pieces {
    char* base;
    size_t used = 0;
    void* take(size_t bytes) {
        void* p = base ? base + used : nullptr;
        used += (bytes + 255) & ~(size_t)255;
        return p;
    }
};

struct Buffers {
    void *g_hidden, *g_down, *g_fc1, *g_norm2, *g_res2, *g_attn_out, *g_heads, *dq, *dk, *dv, *attn, *g_qkv, *g_in_proj, *g_norm1, *x_pre,
        *norm_ws, *conv_ws, *sums;
    float* small_grads;   // norm2, norm, convolution
    size_t attn_bytes, norm_bytes, conv_bytes, sums_bytes, used;
};

Buffers lay_out(const lbi_region_layer& s, void* base) {
    Pieces ws{static_cast<char*>(base)};
    const size_t e = dtype_size(s.dtype), positions = (size_t)(s.B * s.T), rows = positions * (size_t)s.P;
    const size_t g_rows = s.g_broadcast_t ? (size_t)(s.B * s.P) : rows;
    const size_t q_width = (size_t)(s.H * s.Dh), packed = (size_t)((s.H + 2 * s.Hkv) * s.Dh);
    Buffers b{};
    b.g_hidden = s.g_hidden ? nullptr : ws.take(g_rows * s.D * e);
    b.g_down = ws.take(g_rows * s.hidden * e);
    b.g_fc1 = ws.take(rows * 2 * s.hidden * e);
    b.g_norm2 = ws.take(rows * s.D * e);
    b.g_res2 = ws.take(rows * s.D * 4);
    b.g_attn_out = ws.take(rows * s.D * e);
    b.g_heads = ws.take(rows * q_width * e);
    b.dq = ws.take(rows * q_width * e);
    b.dk = ws.take(rows * q_width * e);
    b.dv = ws.take(rows * q_width * e);
    b.attn_bytes = s.attn_edge ? lbi_attn_pullback_edge_workspace_bytes(s.B, s.H, s.T, s.Dh, s.P, s.dtype)
                               : lbi_attn_pullback_workspace_bytes(s.B, s.H, s.T, s.Dh, s.P, s.dtype);
    b.attn = ws.take(b.attn_bytes);
    b.g_in_proj = ws.take(rows * packed * e);
    b.g_norm1 = ws.take(rows * s.D * e);
    if (s.grad_fc2) {
        b.g_qkv = ws.take(rows * packed * e);
        b.x_pre = ws.take(rows * packed * e);
        b.norm_bytes = lbi_rmsnorm_weight_grad_workspace_bytes((int64_t)rows, s.D);
        b.conv_bytes = lbi_causal_conv1d_weight_grad_workspace_bytes(s.B, s.T, (int64_t)packed, s.ksize);
        b.norm_ws = ws.take(b.norm_bytes);
        b.conv_ws = ws.take(b.conv_bytes);
        for (const auto& [m, n] : {std::pair<int64_t, int64_t>{s.D, s.hidden}, {2 * s.hidden, s.D}, {s.D, (int64_t)q_width}, {(int64_t)packed, s.D}})
            b.sums_bytes = std::max(b.sums_bytes, lbi_weight_gradient_workspace_bytes(m, n, (int64_t)rows));
        b.sums = ws.take(b.sums_bytes);
        b.small_grads = static_cast<float*>(ws.take((2 * s.D + packed * (s.ksize + 1)) * 4));
    }
    b.used = ws.used;
    return b;
}

int check(const lbi_region_layer* s) {
    if (!s) return fail(LBI_ERR_INVALID, "lbi_region_layer_pullback: null description");
    if (s->dtype != LBI_F16 && s->dtype != LBI_BF16)
        return fail(LBI_ERR_UNSUPPORTED, "lbi_region_layer_pullback: needs half or bfloat16 (got %d)", s->dtype);
    for (const int64_t n : {s->B, s->P, s->T, s->D, s->hidden, s->H, s->Hkv, s->Dh, s->ksize})
        if (n < 1 || n > (int64_t)1 << 30) return fail(LBI_ERR_INVALID, "lbi_region_layer_pullback: size %lld out of range", (long long)n);
    if (s->ksize > 8 || s->H % s->Hkv || s->Dh % 4)
        return fail(LBI_ERR_UNSUPPORTED, "lbi_region_layer_pullback: filters of up to 8 taps, whole groups of heads, Dh a multiple of 4");
    // every product is a small one (lbi_small_product): 2^30 elements at most, so that no size here overflows
    const double rows = (double)s->B * (double)s->P * (double)s->T, packed = (double)(s->H + 2 * s->Hkv) * (double)s->Dh;
    const double widest = packed > 2.0 * (double)s->hidden ? packed : 2.0 * (double)s->hidden;
    if (rows * widest > 1073741824.0 || rows * (double)s->D > 1073741824.0)
        return fail(LBI_ERR_UNSUPPORTED, "lbi_region_layer_pullback: products too large");
    if (s->grad_fc2 && (s->P != 1 || s->g_broadcast_t))
        return fail(LBI_ERR_INVALID, "lbi_region_layer_pullback: parameter gradients are those of one dense direction");
    for (const void* p : {s->g_residual, s->fc2_weight, s->fc1_weight, s->out_weight, s->in_weight, s->norm2_weight, s->norm1_weight,
                          s->conv_weight, s->fc1_output, s->norm2_input, s->norm1_input, s->q, s->k, s->v, (const void*)s->rope_cos, (const void*)s->rope_sin,
                          (const void*)s->g_input})
        if (!p) return fail(LBI_ERR_INVALID, "lbi_region_layer_pullback: null tensor pointer");
    if (s->grad_fc2)
        for (const void* p : {s->down_input, s->norm2_output, s->out_input, s->norm1_output, (const void*)s->grad_fc1,
                              (const void*)s->grad_out, (const void*)s->grad_in, (const void*)s->grad_norm2, (const void*)s->grad_norm1,
                              (const void*)s->grad_conv})
            if (!p) return fail(LBI_ERR_INVALID, "lbi_region_layer_pullback: null tensor pointer");
    return LBI_OK;
}

#define LBI_STEP(call)          \
    do {                        \
        if (int rc = (call)) return rc; \
    } while (0)

int run(const lbi_region_layer& s, const Buffers& b, void* stream_v) {
    hipStream_t stream = static_cast<hipStream_t>(stream_v);
    const int64_t rows = s.B * s.P * s.T, g_rows = s.g_broadcast_t ? s.B * s.P : rows;
    const int64_t q_width = s.H * s.Dh, packed = (s.H + 2 * s.Hkv) * s.Dh;
    const bool grads = s.grad_fc2 != nullptr;
    auto product = [&](const void* a, const void* w, void* out, int64_t m, int64_t n, int64_t k, int form, int64_t t, int64_t dh) {
        return lbi_small_product(a, w, out, m, n, k, form, t, dh, s.dtype, stream_v);
    };
    auto weight_gradient = [&](const void* a, const void* w, void* out, int64_t m, int64_t n) {
        return lbi_weight_gradient(a, w, out, b.sums_bytes ? b.sums : nullptr, b.sums_bytes, m, n, rows, s.dtype, stream_v);
    };
    const void* g_hidden = s.g_hidden;
    if (!g_hidden) {
        const int64_t n = g_rows * s.D;
        LBI_STEP(cast(static_cast<const float*>(s.g_residual), CastTargets{{b.g_hidden, b.g_hidden, b.g_hidden}, {n, n, n}}, s.dtype, stream));
        g_hidden = b.g_hidden;
    }
    // gated MLP
    if (grads) LBI_STEP(weight_gradient(g_hidden, s.down_input, s.grad_fc2, s.D, s.hidden));
    LBI_STEP(product(g_hidden, s.fc2_weight, b.g_down, g_rows, s.hidden, s.D, LBI_PRODUCT_ROWS_BY_WEIGHT, 1, s.hidden));
    LBI_STEP(lbi_gated_mlp_pullback(b.g_down, s.fc1_output, b.g_fc1, s.B, s.P, s.T, s.hidden, s.g_broadcast_t, s.dtype, stream_v));
    if (grads) LBI_STEP(weight_gradient(b.g_fc1, s.norm2_output, s.grad_fc1, 2 * s.hidden, s.D));
    LBI_STEP(product(b.g_fc1, s.fc1_weight, b.g_norm2, rows, s.D, 2 * s.hidden, LBI_PRODUCT_ROWS_BY_WEIGHT, 1, s.D));
    if (grads)
        LBI_STEP(lbi_rmsnorm_weight_grad(b.g_norm2, s.norm2_input, b.small_grads, b.norm_ws, b.norm_bytes, rows, s.D, s.norm2_eps, s.dtype,
                                         s.norm2_dtype, stream_v));
    LBI_STEP(lbi_rmsnorm_pullback(b.g_norm2, s.norm2_input, s.norm2_weight, s.g_residual, b.g_res2, b.g_attn_out, s.B, s.P, s.T, s.D,
                                  s.norm2_eps, s.g_broadcast_t, s.dtype, s.norm2_dtype, stream_v));
    // attention
    if (grads) LBI_STEP(weight_gradient(b.g_attn_out, s.out_input, s.grad_out, s.D, q_width));
    LBI_STEP(product(b.g_attn_out, s.out_weight, b.g_heads, rows, q_width, s.D, LBI_PRODUCT_ROWS_BY_WEIGHT, s.T, s.Dh));
    LBI_STEP((s.attn_edge ? lbi_attn_pullback_edge : lbi_attn_pullback)(s.q, s.k, s.v, b.g_heads, b.dq, b.dk, b.dv, b.attn, b.attn_bytes, s.B,
                                                                        s.H, s.T, s.Dh, s.P, s.softmax_scale, 1, s.dtype, stream_v));
    if (!grads) {
        LBI_STEP(lbi_attn_qkv_conv_pullback(b.dq, b.dk, b.dv, s.rope_cos, s.rope_sin, s.conv_weight, b.g_in_proj, s.B, s.P, s.T, s.H, s.Hkv,
                                            s.Dh, s.rope_interleaved, s.ksize, s.dtype, stream_v));
    } else {
        LBI_STEP(lbi_attn_qkv_pullback(b.dq, b.dk, b.dv, s.rope_cos, s.rope_sin, b.g_qkv, s.B, s.P, s.T, s.H, s.Hkv, s.Dh, s.rope_interleaved,
                                       s.dtype, stream_v));
        // the cache keeps the projection after the convolution only: redo the projection
        LBI_STEP(product(s.norm1_output, s.in_weight, b.x_pre, rows, packed, s.D, LBI_PRODUCT_FORWARD, 1, packed));
        LBI_STEP(lbi_causal_conv1d_weight_grad(b.g_qkv, b.x_pre, b.small_grads + 2 * s.D, b.conv_ws, b.conv_bytes, s.B, s.T, packed, s.ksize,
                                               s.dtype, stream_v));
        LBI_STEP(lbi_causal_conv1d_pullback(b.g_qkv, s.conv_weight, b.g_in_proj, s.B * s.P, s.T, packed, s.ksize, s.dtype, stream_v));
        LBI_STEP(weight_gradient(b.g_in_proj, s.norm1_output, s.grad_in, packed, s.D));
    }
    LBI_STEP(product(b.g_in_proj, s.in_weight, b.g_norm1, rows, s.D, packed, LBI_PRODUCT_ROWS_BY_WEIGHT, 1, s.D));
    if (grads) {
        LBI_STEP(lbi_rmsnorm_weight_grad(b.g_norm1, s.norm1_input, b.small_grads + s.D, b.norm_ws, b.norm_bytes, rows, s.D, s.norm1_eps,
                                         s.dtype, s.norm1_dtype, stream_v));
        LBI_STEP(cast(b.small_grads, CastTargets{{s.grad_norm2, s.grad_norm1, s.grad_conv}, {s.D, 2 * s.D, 2 * s.D + packed * s.ksize}}, s.dtype,
                      stream));
    }
    return lbi_rmsnorm_pullback(b.g_norm1, s.norm1_input, s.norm1_weight, b.g_res2, s.g_input, s.g_input_branch, s.B, s.P, s.T, s.D,
                                s.norm1_eps, 0, s.dtype, s.norm1_dtype, stream_v);
}

}  // namespace
}  // namespace region_layer
}  // namespace lbi

extern "C" size_t lbi_region_layer_workspace_bytes(const struct lbi_region_layer* s) {
    using namespace lbi;
    clear_error();
    return region_layer::check(s) ? 0 : region_layer::lay_out(*s, nullptr).used;
}

extern "C" int lbi_region_layer_pullback(const struct lbi_region_layer* s, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace lbi;
    clear_error();
    if (int rc = region_layer::check(s)) return rc;
    const region_layer::Buffers b = region_layer::lay_out(*s, workspace);
    if (!workspace || workspace_bytes < b.used || reinterpret_cast<uintptr_t>(workspace) % 256 != 0)
        return fail(LBI_ERR_WORKSPACE, "lbi_region_layer_pullback: 256-byte aligned workspace of %zu bytes needed, %zu given", b.used,
                    workspace_bytes);
    return region_layer::run(*s, b, stream);
}
