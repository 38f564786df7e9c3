// Attention input-pullback in fp32 on the fp32 matrix cores (lbi_attn_f32_kernels.h).
#pragma once

#include <initializer_list>

#include "lbi_common.h"

namespace lbi {
namespace attn_f32 {

constexpr int MAX_DH = 128;

// 16-bit calls of more than 65535 (batch, head, direction) triples stay refused by the scalar kernels.
inline bool supports(int dh, int dtype, int64_t groups) {
    return dh >= 1 && dh <= MAX_DH && (dtype == LBI_F32 || groups <= 65535);
}

// Loads of four elements at a time.
inline bool aligned(int64_t dh, size_t element_bytes, std::initializer_list<const void*> tensors) {
    uintptr_t bits = 0;
    for (const void* p : tensors) bits |= reinterpret_cast<uintptr_t>(p);
    return dh % 4 == 0 && bits % (4 * element_bytes) == 0;
}

// Where the scalar kernels (lbi_attn_generic.h), whose tiles are 16 rows, are as fast or faster; both sides measured:
//  * up to 16 positions half of a 32-row tile is empty, and with few directions waves of a workgroup have no work (B=64
//    H=16 T=4 Dh=64 P=2: 58 us there, 111 here; P=8: 175 and 122); heads of 17 ... 32 in few workgroups gain from the shorter
//    chain of a tile here (B=4 H=8 T=16 Dh=32 P=4: 23 and 21 us), narrower ones do not (Dh=8: 17.5 and 20.5, one launch
//    more), nor do many directions of heads wider than 96 (bf16 B=64 H=16 T=12 P=4, Dh=100: 230 and 277, Dh=96: 203 and 124);
//  * a call of few workgroups is as long as one of them, and a 32-row tile of very narrow heads, or one that is loaded
//    element by element, takes longer than two of 16 rows (B=4 H=8 T=48 Dh=8 P=2: 23 and 29 us; B=1 H=4 T=48 Dh=33 P=2: 43
//    and 51).
// One set of lines for every storage type: over T = 4 ... 56, Dh = 8 ... 128, P = 1 ... 8, B*H = 2 ... 1024 the side they name is the
// slower one by more than a tenth (and 2 us) in 69 of 1534 bf16 calls, by 1.53 at most (B=64 H=16 T=8 Dh=96 P=4: scalar 184, here
// 120), and in 9 of fp32's, by 1.22 at most.
inline bool scalar_is_faster(int64_t B, int64_t H, int64_t T, int64_t dh, int64_t P, bool aligned) {
    const int64_t groups = B * H * P;
    if (groups > 65535) return false;  // more than they take
    if (T <= 16) {
        if (dh > 16 && dh <= 32 && B * H < 512) return false;
        const bool busy = (P >= 8 && dh <= 96) || (P >= 4 && dh >= 64 && dh <= 96 && T > 8);  // enough work for the waves
        return !(aligned && busy && groups >= 1024);
    }
    return T <= 48 && groups < 256 && (aligned ? dh <= 16 && T > 32 : dh > 32);
}

// One storage type each, in a source of its own.
typedef int Launch(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
                   float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream);
Launch launch_float, launch_half, launch_bf16;

// Workspace: lse2[B*H*T], delta[B*P*H*T], as for the scalar kernels.
int launch(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
           float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, int dtype,
           hipStream_t stream);

}  // namespace attn_f32
}  // namespace lbi
