// Attention input-pullback for fp32 storage on the fp32 matrix cores (lbi_attn_f32.hip).
#pragma once

#include "lbi_common.h"

namespace lbi {
namespace attn_f32 {

constexpr int MAX_DH = 128;

inline bool supports(int dh, int dtype) { return dtype == LBI_F32 && dh >= 1 && dh <= MAX_DH; }

// Where the scalar kernels (lbi_attn_generic.h), whose tiles are 16 rows, are as fast or faster; both sides measured:
//  * up to 16 positions half of a 32-row tile is empty, and with few directions waves of a workgroup have no work (B=64
//    H=16 T=4 Dh=64 P=2: 58 us there, 111 here; P=8: 175 and 122); narrow heads in few workgroups gain from the shorter
//    chain of a tile here (B=4 H=8 T=16 Dh=32 P=4: 23 and 21 us);
//  * a call of few workgroups is as long as one of them, and a 32-row tile of very narrow heads, or one that is loaded
//    element by element, takes longer than two of 16 rows (B=4 H=8 T=48 Dh=8 P=2: 23 and 29 us; B=1 H=4 T=48 Dh=33 P=2: 43
//    and 51).
inline bool scalar_is_faster(int64_t B, int64_t H, int64_t T, int64_t dh, int64_t P, bool aligned) {
    const int64_t groups = B * H * P;
    if (groups > 65535) return false;  // more than they take
    if (T <= 16) {
        if (dh <= 32 && B * H < 512) return false;
        const bool busy = (P >= 8 && dh <= 96) || (P >= 4 && dh >= 64 && T > 8);  // enough work for the waves
        return !(aligned && busy && groups >= 1024);
    }
    return T <= 48 && groups < 256 && (aligned ? dh <= 16 && T > 32 : dh > 32);
}

// Workspace: lse2[B*H*T], delta[B*P*H*T], as for the scalar kernels.
int launch(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
           float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream);

}  // namespace attn_f32
}  // namespace lbi
