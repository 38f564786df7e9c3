// The kernels of lbi_attn_f32_kernels.h for bf16 storage.
#include "lbi_attn_f32_kernels.h"

namespace lbi {
namespace attn_f32 {

int launch_bf16(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
                float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream) {
    return launch_typed<bf16_raw>(q, k, v, d_out, dq, dk, dv, workspace, B, H, T_len, dh, P, scale, causal, stream);
}

}  // namespace attn_f32
}  // namespace lbi
