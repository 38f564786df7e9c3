// The small products of a linear layer, y = x weight^T, in one 16-bit type, sums in fp32, C rounded once:
//   ROWS_BY_WEIGHT  C = A W    the pullback: A [M, K] cotangent rows, W [K, N] the weight as it lies; C as [M, N] or, heads
//                              split, as [M / T, N / Dh, T, Dh]
//   GRADIENT        C = A^T W  the weight's gradient: A [K, M] cotangent rows, W [K, N] the layer's input
//   FORWARD         C = A W^T  the layer itself: A [M, K], W [N, K]
//
// A call of this size is a few microseconds of products on the part; what it costs is the call.  (A library product takes 18 us of
// host time, one here 7, and the layout that the next kernel wants takes no launch of its own.)
//
// A workgroup of four waves owns 32 WM rows x 32 WN columns; with fewer than four tiles of 32 x 32 the waves share the reduction
// of a tile, and their sums are added in wave order.  Operands pass through LDS in chunks of 64 k, two buffers, the
// next AHEAD chunks in registers: bound by the latency of those loads where K is long (0.2 us a chunk; 0.37 while the compiler
// waited for all of them at every chunk: 512 x 6144 x 768 35.7 -> 20.5 us, 2048 x 2048 x 256 13.9 -> 9.0).  The product is formed as C^T
// (lanes are rows of C), so that a lane ends up with four consecutive columns: 8-byte stores.  An operand whose reduction
// index is its row comes through transposing LDS reads, another through plain ones.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lbi_attn_mfma.h"

namespace lbi {
namespace product {
namespace {

using attn_mfma::Mma;
using attn_mfma::s16x4;
using attn_mfma::tile_off;
using attn_mfma::u32x2;
using attn_mfma::u32x4;

constexpr int CHUNK = 64, AHEAD = 3, RING = 2 * AHEAD;
template <int N> using At = std::integral_constant<int, N>;
constexpr unsigned PAST_END = 1u << 31;  // operands are smaller

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

// ROWS x 64 elements of a row-major matrix on their way to LDS; what lies past its end is zero.
template <int ROWS> struct Stage {
    static constexpr int PIECES = ROWS * 8 / 256;
    u32x4 reg[PIECES];
    __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t src, int row0, int col0, int cols, int tid) {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int id = tid + 256 * u, c = col0 + id % 8 * 8;
            const unsigned off = c < cols ? (unsigned)((row0 + id / 8) * cols + c) * 2 : PAST_END;
            reg[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, off, 0, 0));
        }
    }
    __device__ __forceinline__ void commit(char* tile, int tid) const {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int id = tid + 256 * u;
            *reinterpret_cast<u32x4*>(tile + tile_off<64>(id / 8, id % 8)) = reg[u];
        }
    }
};

// The tile of W is 64 columns wide.  FORM: how the operands lie.
constexpr int ROWS_BY_WEIGHT = LBI_PRODUCT_ROWS_BY_WEIGHT, GRADIENT = LBI_PRODUCT_GRADIENT, FORWARD = LBI_PRODUCT_FORWARD;
template <typename T, int WM, int FORM>
__global__ __launch_bounds__(256) void product_kernel(const T* __restrict__ a, const T* __restrict__ w, T* __restrict__ out,
                                                      int M, int N, int K, int T_len, int Dh, int n_tiles) {
    constexpr int KS = 2 / WM, STEPS = CHUNK / 16 / KS, ROWS = 32 * WM;
    constexpr int A_BYTES = ROWS * 128, BUF = A_BYTES + CHUNK * 128;
    __shared__ __align__(16) char lds[2 * BUF];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, wm = WM == 2 ? wave >> 1 : 0, kz = WM == 2 ? 0 : wave >> 1;
    const int row0 = (int)(blockIdx.x / n_tiles) * ROWS, col0 = (int)(blockIdx.x % n_tiles) * 64;
    const auto a_src = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a), 0, (unsigned)M * K * 2, 4 << 15);
    const auto w_src = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(w), 0, (unsigned)K * N * 2, 4 << 15);
    const int steps = (K + CHUNK - 1) / CHUNK;
    static_assert(FORM != GRADIENT || WM == 2, "a transposed tile of A has 64 columns");
    Stage<ROWS> as[AHEAD];
    Stage<CHUNK> ws[AHEAD];
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    auto fetch = [&](int slot, int it) __attribute__((always_inline)) {  // chunks past the last are all zero
        if constexpr (FORM == GRADIENT) as[slot].fetch(a_src, it * CHUNK, row0, M, tid);
        else as[slot].fetch(a_src, row0, it * CHUNK, K, tid);
        if constexpr (FORM == FORWARD) ws[slot].fetch(w_src, col0, it * CHUNK, K, tid);
        else ws[slot].fetch(w_src, it * CHUNK, col0, N, tid);
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(u, u);
    int base = 0;
    auto step = [&](auto place, bool more) __attribute__((always_inline)) {
        constexpr int u = decltype(place)::value;
        char* buf = lds + (u & 1) * BUF;
        as[u % AHEAD].commit(buf, tid);
        ws[u % AHEAD].commit(buf + A_BYTES, tid);
        if (more) fetch(u % AHEAD, base + u + AHEAD);
        // one barrier a chunk: the buffer written next was read before the barrier of the chunk in between
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) {
            const int k = kz * STEPS + ks;
            u32x4 af, wf;
            if constexpr (FORM == GRADIENT) af = frag_columns(buf, lane, 16 * k, 32 * wm);
            else af = *reinterpret_cast<const u32x4*>(buf + tile_off<64>(32 * wm + m, 2 * k + h));
            if constexpr (FORM == FORWARD) wf = *reinterpret_cast<const u32x4*>(buf + A_BYTES + tile_off<64>(32 * wn + m, 2 * k + h));
            else wf = frag_columns(buf + A_BYTES, lane, 16 * k, 32 * wn);
            acc = Mma<T>::mma(wf, af, acc);
        }
    };
    // Whole turns of the ring, then what is left, nested: a step that is left out in the middle would make the compiler wait for
    // every load under way at the join.
    auto turn = [&](auto... places) __attribute__((always_inline)) {
        static_assert(sizeof...(places) == RING);
        (step(places, true), ...);
    };
    for (; base + RING <= steps; base += RING) turn(At<0>{}, At<1>{}, At<2>{}, At<3>{}, At<4>{}, At<5>{});
    auto rest = [&](auto self, auto place) __attribute__((always_inline)) -> void {
        constexpr int u = decltype(place)::value;
        if constexpr (u < RING - 1)
            if (base + u < steps) {
                step(place, u + AHEAD < RING - 1);
                self(self, At<u + 1>{});
            }
    };
    rest(rest, At<0>{});
    if constexpr (KS == 2) {
        __syncthreads();
        f32x4* sums = reinterpret_cast<f32x4*>(lds) + wn * 256;
        if (kz == 1)
#pragma unroll
            for (int g = 0; g < 4; ++g) sums[64 * g + lane] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        __syncthreads();
        if (kz == 1) return;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 other = sums[64 * g + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * g + e] += other[e];
        }
    }
    const int row = row0 + 32 * wm + m;
    if (row >= M) return;
    const int n = row / T_len, t = row % T_len, heads = N / Dh;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int c = col0 + 32 * wn + 8 * g + 4 * h;
        if (c >= N) continue;
        const size_t at = (((size_t)n * heads + c / Dh) * T_len + t) * Dh + c % Dh;
        *reinterpret_cast<u32x2*>(out + at) = u32x2{Mma<T>::pack2(acc[4 * g], acc[4 * g + 1]), Mma<T>::pack2(acc[4 * g + 2], acc[4 * g + 3])};
    }
}

template <typename T>
int launch(const void* a, const void* w, void* out, int M, int N, int K, int form, int T_len, int Dh, hipStream_t stream) {
    const int n_tiles = (N + 63) / 64;
    // 64 rows of a workgroup where that gives every CU one, 32 otherwise
    const bool tall = form == GRADIENT || (long long)((M + 63) / 64) * n_tiles >= device_compute_units();
    const int m_tiles = tall ? (M + 63) / 64 : (M + 31) / 32;
    const auto kernel = form == GRADIENT ? product_kernel<T, 2, GRADIENT>
                        : form == FORWARD ? (tall ? product_kernel<T, 2, FORWARD> : product_kernel<T, 1, FORWARD>)
                                          : (tall ? product_kernel<T, 2, ROWS_BY_WEIGHT> : product_kernel<T, 1, ROWS_BY_WEIGHT>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(m_tiles * n_tiles)), dim3(256), 0, stream, static_cast<const T*>(a),
                       static_cast<const T*>(w), static_cast<T*>(out), M, N, K, T_len, Dh, n_tiles);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

}  // namespace
}  // namespace product
}  // namespace lbi

extern "C" int lbi_small_product(const void* a, const void* w, void* out, int64_t M, int64_t N, int64_t K, int form, int64_t T,
                                 int64_t Dh, int dtype, void* stream) {
    using namespace lbi;
    clear_error();
    if (M < 0 || N < 0 || K < 0 || T < 1 || Dh < 0)
        return fail(LBI_ERR_INVALID, "lbi_small_product: bad size (M=%lld N=%lld K=%lld T=%lld Dh=%lld)", (long long)M, (long long)N,
                    (long long)K, (long long)T, (long long)Dh);
    if (M == 0 || N == 0) return LBI_OK;
    if (!a || !w || !out) return fail(LBI_ERR_INVALID, "lbi_small_product: null pointer");
    if (form != LBI_PRODUCT_ROWS_BY_WEIGHT && form != LBI_PRODUCT_GRADIENT && form != LBI_PRODUCT_FORWARD)
        return fail(LBI_ERR_INVALID, "lbi_small_product: bad form %d", form);
    constexpr int64_t kMost = 1 << 30;  // elements of a matrix: offsets are 32 bits of bytes, and one bit says "past the end"
    const bool by_pieces = N % 8 == 0 && (form == LBI_PRODUCT_GRADIENT ? M : K) % 8 == 0;
    // what the tiles of the kernel span, the chunks that are asked for ahead included
    const bool fits = M < kMost && N < kMost && K < kMost && (M + 64) * (K + 256) < kMost && (K + 256) * (N + 64) < kMost &&
                      (M / 32 + 1) * (N / 64 + 1) < 1 << 24;
    if ((dtype != LBI_F16 && dtype != LBI_BF16) || K < 1 || !by_pieces || !fits)
        return fail(LBI_ERR_UNSUPPORTED, "lbi_small_product: needs half or bfloat16, rows of whole 16-byte pieces, operands below "
                                         "2 GiB, fewer than 2^24 tiles");
    if (Dh < 1 || Dh % 4 != 0 || N % Dh != 0 || M % T != 0)
        return fail(LBI_ERR_INVALID, "lbi_small_product: N must be heads of Dh (a multiple of 4), M sequences of T rows");
    for (const void* ptr : {a, w, (const void*)out})
        if (reinterpret_cast<uintptr_t>(ptr) % 16) return fail(LBI_ERR_INVALID, "lbi_small_product: tensors must be 16-byte aligned");
    const auto typed = dtype == LBI_F16 ? product::launch<_Float16> : product::launch<bf16_raw>;
    return typed(a, w, out, (int)M, (int)N, (int)K, form, (int)T, (int)Dh, static_cast<hipStream_t>(stream));
}
