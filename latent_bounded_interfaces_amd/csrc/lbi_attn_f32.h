// Attention input-pullback for fp32 storage on the fp32 matrix cores (lbi_attn_f32.hip).
#pragma once

#include "lbi_common.h"

namespace lbi {
namespace attn_f32 {

constexpr int MAX_DH = 128;

inline bool supports(int dh, int dtype) { return dtype == LBI_F32 && dh >= 1 && dh <= MAX_DH; }

// Workspace: lse2[B*H*T], delta[B*P*H*T], as for the scalar kernels.
int launch(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
           float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream);

}  // namespace attn_f32
}  // namespace lbi
