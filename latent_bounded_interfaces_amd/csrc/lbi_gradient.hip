// The weight gradient of a linear layer, C = A^T W: A [K, M] cotangent rows, W [K, N] the layer's input, both in one 16-bit type,
// K rows of tokens, C [M, N]; sums in fp32, rounded once.
//
// Such a product has few results and long sums: 768 x 3072 results are 144 tiles of 128 x 128, which leave 112 of the CUs idle, and
// each is a chain of 8192 terms.  So the sums are cut: a workgroup owns one tile and one range of K, its partial sums go to the
// workspace in the order in which the lanes hold them, and a second kernel adds those of a tile in order of K and rounds.
//
// A workgroup of four waves, 64 x 64 results each, takes 32 rows of both operands a step through LDS, in a ring of four, three
// steps ahead; two workgroups fit a CU.  The rows arrive by buffer_load ... lds (what lies past the end of an operand is zero) and leave
// through transposing LDS reads, the reduction index being the row of both.  Bound: alone on its CU a workgroup takes 0.3 us a step,
// which is latency (1.0 us for 64 rows with two buffers); all CUs together read 12.5 TB/s of tiles from the caches, 0.33 us for one
// step on each; the LDS would be full at 0.16.  A deeper ring changed nothing.
//
// bf16, M x N x K, the library's product (which does not cut the sums), lbi_small_product and this, us: 768 x 3072 x 8192 96, 100, 60; 768 x 768 x
// 8192 57, 39, 22; 2304 x 768 x 8192 73, 68, 45; 6144 x 768 x 8192 114, 168, 95; 6144 x 768 x 4096 61, 87, 51; 256 x 256 x 8192 48, 34, 16;
// 8192 x 1024 x 8192 154, 258, 141.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "lbi_attn_mfma.h"
#include "lbi_attn_dkdv128.h"

namespace lbi {
namespace gradient {
namespace {

using attn_mfma::Mma;
using attn_mfma::s16x4;
using attn_mfma::swz;
using attn_mfma::tile_off;
using attn_mfma::u32x2;
using attn_mfma::u32x4;

constexpr int TILE = 128, STEP = 32, RING = 4, AHEAD = RING - 1, NT = 256;
constexpr int SUB = STEP * 128, BUF = 4 * SUB;  // bytes: STEP rows x 64 columns; two of A, two of W
constexpr int LOADS = STEP / 8;                 // of a wave and step
constexpr int TILE_SUMS = TILE * TILE;

// lane (m, h) gets tile[k0 + 8h .. + 7][n0 + m]
__device__ __forceinline__ u32x4 frag_columns(const char* tile, int lane, int k0, int n0) {
    const int s = lane & 15, g1 = (lane >> 4) & 1, h = lane >> 5;
    const int row = k0 + 8 * h + (s >> 2);
    const int chunk = (n0 >> 3) + 2 * g1 + ((s & 3) >> 1);
    const int sub = (s & 1) << 3;
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + tile_off<64>(row, chunk) + sub));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + tile_off<64>(row + 4, chunk) + sub));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
}

template <typename T>
__device__ __forceinline__ void store4(T* out, int row, int col, int M, int N, f32x4 v) {
    if (row < M && col < N)
        *reinterpret_cast<u32x2*>(out + (size_t)row * N + col) = u32x2{Mma<T>::pack2(v[0], v[1]), Mma<T>::pack2(v[2], v[3])};
}

// Workgroup -> (range of K, tile).  Ids equal mod 8 share an L2: they get neighbouring tiles of the same rows.
__device__ __forceinline__ int place(int id, int count) {
    const int lot = count / 8, left = count % 8, x = id % 8;
    return x * lot + min(x, left) + id / 8;
}

template <typename T>
__global__ __launch_bounds__(NT, 2) void gradient_kernel(const T* __restrict__ a, const T* __restrict__ w, T* __restrict__ out,
                                                         f32x4* __restrict__ sums, int M, int N, int K, int n_tiles, int tiles,
                                                         int steps, int count) {
    __shared__ __align__(16) char lds[RING * BUF];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int at = place((int)blockIdx.x, count), range = at / tiles, tile = at - range * tiles;
    const int row0 = tile / n_tiles * TILE, col0 = tile % n_tiles * TILE;
    const int first = range * steps, last = min(first + steps, (K + STEP - 1) / STEP);
    // the wave's share of a step: one of the four pieces, eight rows a load; the lane's place in LDS is given, its source is swizzled
    const bool of_w = wave >= 2;
    const T* src = of_w ? w : a;
    const int width = of_w ? N : M, c0 = (of_w ? col0 : row0) + 64 * (wave & 1);
    const unsigned bytes = (unsigned)K * width * 2;
    unsigned off[2];  // rows 0 ... 7 and 8 ... 15
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int row = 8 * u + lane / 8, col = c0 + 8 * ((lane % 8) ^ swz<64>(row));
        off[u] = col < width ? (unsigned)(row * width + col) * 2 : 1u << 31;  // operands are smaller
    }
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds + wave * SUB;
    auto fetch = [&](int it, int slot) __attribute__((always_inline)) {  // past the last step: zeros
        const unsigned from = (unsigned)it * STEP * width * 2, to = lds0 + slot * BUF, end = it < last ? bytes : 0;
#pragma unroll
        for (int u = 0; u < LOADS; ++u)
            attn_mfma::dma_tile<true>(src, off[u & 1] + from + (unsigned)(u / 2 * 16 * width) * 2, end, to + u * 1024);
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(first + u, u);
    int slot = 0;
    for (int it = first; it < last; ++it) {
        // this wave's loads of the step have landed and its reads of the last one are done, and behind the barrier everyone's
        __builtin_amdgcn_s_waitcnt(attn_mfma::waitcnt_vm((AHEAD - 1) * LOADS));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        fetch(it + AHEAD, slot == 0 ? RING - 1 : slot - 1);
        const char* at_a = lds + slot * BUF + (wave >> 1) * SUB;
        const char* at_w = lds + slot * BUF + (2 + (wave & 1)) * SUB;
        slot = slot + 1 == RING ? 0 : slot + 1;
#pragma unroll
        for (int ks = 0; ks < STEP / 16; ++ks) {
            u32x4 af[2], wf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                af[i] = frag_columns(at_a, lane, 16 * ks, 32 * i);
                wf[i] = frag_columns(at_w, lane, 16 * ks, 32 * i);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = Mma<T>::mma(wf[j], af[i], acc[i][j]);
        }
    }
    __builtin_amdgcn_s_waitcnt(attn_mfma::waitcnt_vm(0));  // nothing is under way into LDS when the workgroup ends
    const int m = lane & 31, h = lane >> 5;
    f32x4* mine = sums + ((size_t)at * 4 + wave) * (TILE_SUMS / 16) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                if (count == tiles) store4(out, row0 + 64 * (wave >> 1) + 32 * i + m, col0 + 64 * (wave & 1) + 32 * j + 8 * g + 4 * h, M, N, v);
                else mine[((2 * i + j) * 4 + g) * 64] = v;
            }
}

// A workgroup adds a quarter of a tile, one wave's of the kernel above.
template <typename T>
__global__ __launch_bounds__(NT) void add_ranges_kernel(const f32x4* __restrict__ sums, T* __restrict__ out, int M, int N, int n_tiles,
                                                        int tiles, int ranges) {
    const int tile = blockIdx.x / 4, wave = blockIdx.x % 4, tid = threadIdx.x, lane = tid & 63, g = tid >> 6;
    const int row = tile / n_tiles * TILE + 64 * (wave >> 1) + (lane & 31), col = tile % n_tiles * TILE + 64 * (wave & 1) + 8 * g + 4 * (lane >> 5);
    const f32x4* at = sums + ((size_t)tile * 4 + wave) * (TILE_SUMS / 16) + tid;
    f32x4 total[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) total[u] = at[NT * u];
    #pragma unroll 2
    for (int r = 1; r < ranges; ++r) {
        at += (size_t)tiles * (TILE_SUMS / 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const f32x4 v = at[NT * u];
#pragma unroll
            for (int e = 0; e < 4; ++e) total[u][e] += v[e];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) store4(out, row + 32 * (u / 2), col + 32 * (u % 2), M, N, total[u]);
}

struct Plan {
    int n_tiles, tiles, steps, ranges;  // steps of a range
    double us;
};

// Into how many ranges the sums are cut, by what a call takes: the steps of a CU's workgroups one after another, those of all of them from the
// caches, and the partial sums once out and back.  The constants fit 47 calls of 256 ... 8192 x 256 ... 4096 results and sums of 700 ... 8192, each
// with 1 to 16 ranges: what is chosen is 1.02 times the best on average, 1.09 at most.
Plan plan_of(int64_t M, int64_t N, int64_t K) {
    const int m_tiles = (int)((M + TILE - 1) / TILE), n_tiles = (int)((N + TILE - 1) / TILE), tiles = m_tiles * n_tiles;
    const int all = (int)((K + STEP - 1) / STEP);
    const double cus = device_compute_units();
    Plan best{n_tiles, tiles, all, 1, 0.0};
    for (int s = 1; s <= 64 && (s == 1 || s * 8 <= all); ++s) {
        const int steps = (all + s - 1) / s, ranges = (all + steps - 1) / steps;
        if (ranges != s) continue;
        const double count = (double)tiles * s, deep = ceil(count / cus);
        const double chain = steps * (deep > 1.0 ? 0.33 * ceil(deep / 2.0) : 0.255), caches = count * steps * 0.28 / cus;
        const double us = std::max(chain, caches) + (s > 1 ? 3.7 + count * TILE_SUMS * 8.0 / 7.2e6 : 0.0);
        if (s == 1 || us < best.us) best = {n_tiles, tiles, steps, ranges, us};
    }
    return best;
}

// lbi_small_product takes 64 x 64 results a workgroup, uncut, 0.26 us for 64 terms until the workgroups fill the CUs.  It is the faster one
// for short sums: 768 x 768 x 700 8.3 us there, 10.6 here, 512 x 2048 x 1800 12.1 and 16.6, 512 x 512 x 1800 11.2 and 12.1; past the line 4096
// x 512 x 700 13.1 and 10.9, 768 x 3072 x 1800 25.2 and 21.4, 768 x 768 x 4096 19.5 and 18.8.
bool small_is_faster(const Plan& p, int64_t M, int64_t N, int64_t K) {
    const double tiles = (double)((M + 63) / 64) * (double)((N + 63) / 64), steps = (double)((K + 63) / 64);
    return steps * 0.26 * std::max(1.0, tiles / (0.83 * device_compute_units())) <= p.us + 1.0;
}

template <typename T>
int launch(const void* a, const void* w, void* out, void* sums, int M, int N, int K, const Plan& p, hipStream_t stream) {
    const int count = p.tiles * p.ranges;
    hipLaunchKernelGGL((gradient_kernel<T>), dim3((unsigned)count), dim3(NT), 0, stream, static_cast<const T*>(a),
                       static_cast<const T*>(w), static_cast<T*>(out), static_cast<f32x4*>(sums), M, N, K, p.n_tiles, p.tiles, p.steps, count);
    if (p.ranges > 1)
        hipLaunchKernelGGL((add_ranges_kernel<T>), dim3((unsigned)(4 * p.tiles)), dim3(NT), 0, stream, static_cast<const f32x4*>(sums),
                           static_cast<T*>(out), M, N, p.n_tiles, p.tiles, p.ranges);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

// what 32-bit offsets span, the steps asked for past the end included
bool takes(int64_t M, int64_t N, int64_t K) {
    constexpr int64_t most = 1 << 30;
    return M > 0 && N > 0 && K > 0 && M % 8 == 0 && N % 8 == 0 && M < most && N < most && K < most &&
           (K + (RING + 1) * STEP) * (M + TILE) < most && (K + (RING + 1) * STEP) * (N + TILE) < most && (M / TILE + 1) * (N / TILE + 1) < 1 << 20;
}

}  // namespace
}  // namespace gradient
}  // namespace lbi

extern "C" size_t lbi_weight_gradient_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    using namespace lbi::gradient;
    if (!takes(M, N, K)) return 0;
    const Plan p = plan_of(M, N, K);
    return p.ranges > 1 && !small_is_faster(p, M, N, K) ? (size_t)p.tiles * p.ranges * TILE_SUMS * sizeof(float) : 0;
}

extern "C" int lbi_weight_gradient(const void* a, const void* w, void* out, void* workspace, size_t workspace_bytes, int64_t M,
                                   int64_t N, int64_t K, int dtype, void* stream) {
    using namespace lbi;
    const bool ours = gradient::takes(M, N, K) && (dtype == LBI_F16 || dtype == LBI_BF16);
    const gradient::Plan p = ours ? gradient::plan_of(M, N, K) : gradient::Plan{};
    if (!ours || gradient::small_is_faster(p, M, N, K))
        return lbi_small_product(a, w, out, M, N, K, LBI_PRODUCT_GRADIENT, 1, N, dtype, stream);
    clear_error();
    if (!a || !w || !out) return fail(LBI_ERR_INVALID, "lbi_weight_gradient: null pointer");
    for (const void* ptr : {a, w, (const void*)out, (const void*)workspace})
        if (reinterpret_cast<uintptr_t>(ptr) % 16) return fail(LBI_ERR_INVALID, "lbi_weight_gradient: tensors must be 16-byte aligned");
    const size_t need = p.ranges > 1 ? (size_t)p.tiles * p.ranges * gradient::TILE_SUMS * sizeof(float) : 0;
    if (need && (!workspace || workspace_bytes < need))
        return fail(LBI_ERR_WORKSPACE, "lbi_weight_gradient: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    const auto typed = dtype == LBI_F16 ? gradient::launch<_Float16> : gradient::launch<bf16_raw>;
    return typed(a, w, out, workspace, (int)M, (int)N, (int)K, p, static_cast<hipStream_t>(stream));
}
