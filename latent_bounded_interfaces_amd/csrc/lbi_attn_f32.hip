// The kernels of lbi_attn_f32_kernels.h for fp32 storage.
#include "lbi_attn_f32_kernels.h"

namespace lbi {
namespace attn_f32 {

int launch_float(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
                 float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream) {
    return launch_typed<float>(q, k, v, d_out, dq, dk, dv, workspace, B, H, T_len, dh, P, scale, causal, stream);
}

int launch(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
           float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, int dtype,
           hipStream_t stream) {
    const auto typed = dtype == LBI_F32 ? launch_float : dtype == LBI_F16 ? launch_half : launch_bf16;
    return typed(q, k, v, d_out, dq, dk, dv, workspace, B, H, T_len, dh, P, scale, causal, stream);
}

}  // namespace attn_f32
}  // namespace lbi
