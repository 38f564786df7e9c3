// Attention input-pullback in fp32 on the fp32 matrix cores: any T, head dim <= 128, any storage type, causal or not.
// 16-bit storage comes here where the 16-bit matrix-core kernels do not take the shape as it lies (long non-causal calls of
// ragged length above all): probabilities, dS and all sums stay fp32, as in the scalar kernels that took these calls
// before, and results round once.
//
// Bound: v_mfma_f32_32x32x2_f32 does 64 flop per cycle and SIMD (157 TFLOP/s on the part); a product is 64 cycles,
// so LDS, softmax and address work of a tile fit under its products and one wave per SIMD is enough.
//
// Operand layout of that instruction (lane = 32*h + m):
//   A (32 x 2): lane holds A[m][h]      B (2 x 32): lane holds B[h][m]
//   C (32 x 32): register i of the lane holds C[row(i)][m],  row(i) = 8*(i/4) + 4*h + i%4
// Which two k a product takes is free as long as A and B agree, which gives the two forms used here:
//   * reduction over the head dim ("dot" form): product t takes column t of the lower and of the upper half of the
//     head dim, so a lane's operand is one contiguous half row: 16-byte LDS reads, or registers for the operand
//     that stays with the wave;
//   * reduction over the rows of an accumulator tile ("chain" form): product t takes rows row(t) of both lane halves,
//     so register t of the tile IS the operand, and the other side is one 4-byte LDS read of row row(t), 32
//     consecutive columns per lane half.  P and dS never leave the registers.
//
// Four kernels per call, every output with one owner and a fixed summation order (no atomics, reruns bit-identical):
//   stats   lse2[b,h,i] (log2 domain)
//   delta   delta[b,p,h,i] = sum_j P dP
//   dq      a wave owns 32 queries x PB directions (S^T orientation: lanes are queries), as in stats and delta
//   dkdv    a wave owns 32 keys x PB directions (S orientation: lanes are keys)
// The streamed tiles pass through two LDS buffers (the next tile waits in registers during the products of the current
// one; one barrier per tile) and are shared by the four waves of a workgroup, which own different directions of the same
// rows as far as there are any: under the causal mask neighbouring row tiles end at different steps and the waves of the
// shorter ones wait (B=4 H=8 T=512 Dh=64 P=8: dq 145 -> 125 us, dkdv 189 -> 175 us against four row tiles).  Two
// directions per wave share one S tile, at one wave per SIMD; one direction at two waves per SIMD took 176 / 201 us.
// Whole call there: 5.41 ms on the scalar kernels (lbi_attn_generic.h), 0.355 ms here (50 TFLOP/s algorithmic), with the
// error of the scalar kernels: relative 2-norm against 64 bits 3.9e-7 / 6.0e-7 / 5.9e-7 in dQ / dK / dV, and 0.98 to 1.02
// times theirs over T = 24 ... 3000, head dims 16 ... 128, V with and without an offset.
// 16-bit storage, no mask, scalar kernels -> here: bf16 B=4 H=8 T=1000 Dh=64 P=8 26.2 -> 2.36 ms, B=1 H=2 T=333 Dh=64 P=3 388 ->
// 160 us, B=1 H=4 T=250 Dh=128 P=16 1005 -> 214 us; fp16 B=8 H=12 T=500 Dh=80 P=4 13.2 -> 1.67 ms; the same errors to three digits.
#pragma once

#include "lbi_attn_f32.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace lbi {
namespace attn_f32 {
namespace {

constexpr int NWAVE = 4, NT = 64 * NWAVE, TILE = 32;
constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ int acc_row(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }
__device__ __forceinline__ f32x16 mma(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// P of a score: the product is rounded before the subtraction, as in the statistics (a fused step would leave its rounding
// in P: with one visible key, P would not be exactly one).
__device__ __forceinline__ float prob_of(float score, float sc2, float lse) {
#pragma clang fp contract(off)
    const float x = score * sc2;
    return exp2f(x - lse);
}
__device__ __forceinline__ void store(float* p, float v) { *p = v; }
__device__ __forceinline__ void store(_Float16* p, float v) { *p = (_Float16)v; }
__device__ __forceinline__ void store(bf16_raw* p, float v) { p->bits = f32_to_bf16_bits(v); }
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.0f;
    return z;
}

// Products over the head dim: acc[p] += tile (32 rows in LDS) . own[p]^T.  The 16-byte LDS read of the next four products
// is issued ahead of the current ones (a wave has the SIMD to itself, nothing else would hide its latency), and
// `side(i)` for i = 0 .. 15, vector work that does not depend on these products, runs in their shadow.
template <int DH, int N, typename Side>
__device__ __forceinline__ void dot_form(f32x16 (&acc)[N], const float* lane_tile, const float (&own)[N][DH / 2],
                                         Side side) {
    constexpr int ROUNDS = DH / 8;
    f32x4 a[2];
    a[0] = *reinterpret_cast<const f32x4*>(lane_tile);
#pragma unroll
    for (int c = 0; c < ROUNDS; ++c) {
        if (c + 1 < ROUNDS) a[(c + 1) & 1] = *reinterpret_cast<const f32x4*>(lane_tile + 4 * (c + 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int p = 0; p < N; ++p) acc[p] = mma(a[c & 1][e], own[p][4 * c + e], acc[p]);
#pragma unroll
        for (int i = 16 * c / ROUNDS; i < 16 * (c + 1) / ROUNDS; ++i) side(i);
    }
}

// Products over the rows of accumulator tiles: acc[p][n] += x[p]^T . tile[:, 32n ...].
// `lane_tile` points at row 4h, column m of the tile.  `side(i)` runs in the shadow of the products of register i - 2
// (i = 0, 1: in front of them), so it may also form x[p][i].
template <int NB, int PITCH, int N, typename Side>
__device__ __forceinline__ void chain_form(f32x16 (&acc)[N][NB], const float* lane_tile, const f32x16 (&x)[N],
                                           Side side) {
    float b[2][2][NB];   // two rows per round, two rounds
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int n = 0; n < NB; ++n) b[0][u][n] = lane_tile[acc_row(u, 0) * PITCH + 32 * n];
        side(u);
    }
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
        if (i + 2 < 16)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int n = 0; n < NB; ++n) b[((i >> 1) + 1) & 1][u][n] = lane_tile[acc_row(i + 2 + u, 0) * PITCH + 32 * n];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    const float t = b[(i >> 1) & 1][u][n];
                    acc[p][n] = mma(x[p][i + u], t, acc[p][n]);
                }
        if (i + 2 < 16) {
            side(i + 2);
            side(i + 3);
        }
    }
}
constexpr auto nothing = [](int) __attribute__((always_inline)) {};

// The tile on the diagonal: rows that an output row may not see have x = 0, but zero times a value that is not finite is
// NaN.  If that has happened (acc, zero before the tile, holds something that is not finite), the products are repeated one
// tile row at a time and taken over only where `sees(output row, tile row)`.  `lane_tile` points at row 0, column m.
template <int NB, int PITCH, int N, typename Sees>
__device__ __forceinline__ void mend_diagonal(f32x16 (&acc)[N][NB], const float* lane_tile, const f32x16 (&x)[N], int h,
                                              Sees sees) {
    float probe = 0.0f;
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) probe = fmaf(acc[p][n][r], 0.0f, probe);
    if (!__any(probe != 0.0f)) return;
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[p][n] = zero16();
#pragma unroll 1
    for (int row = 0; row < TILE; ++row) {
        const int i = 4 * (row >> 3) + (row & 3);  // register and lane half that hold x of this row
        const bool mine = h == ((row >> 2) & 1);
        float b[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) b[n] = mine ? lane_tile[row * PITCH + 32 * n] : 0.0f;
#pragma unroll
        for (int p = 0; p < N; ++p) {
            float a = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) a = mine && e == i ? x[p][e] : a;
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const f32x16 sum = mma(a, b[n], acc[p][n]);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[p][n][r] = sees(acc_row(r, h), row) ? sum[r] : acc[p][n][r];
            }
        }
    }
}

// Four consecutive elements on their way from memory, as stored: widened where they are loaded, they would be waited for
// there.  One by one (no VEC) each has a register of its own, since packing two would wait as well.
template <typename T> struct Storage { typedef unsigned short Bits; };
template <> struct Storage<float> { typedef float Bits; };
template <typename T, bool VEC> struct RawOf { typedef unsigned Type __attribute__((ext_vector_type(4))); };
template <typename T> struct RawOf<T, true> { typedef u16x4 Type; };
template <bool VEC> struct RawOf<float, VEC> { typedef f32x4 Type; };
template <> struct RawOf<float, true> { typedef f32x4 Type; };
template <typename T, bool VEC> using Raw = typename RawOf<T, VEC>::Type;

// Four consecutive elements of a row-major [T, dh] matrix from (row, c), zero outside it.  The load itself is never
// predicated: it reads a clamped address and `keep` says whether the value counts, so that nothing waits for a load
// before its value is needed (a load under a branch is waited for at the join).  VEC: dh is a multiple of four and the
// matrix aligned to four elements.
template <typename T, bool VEC>
__device__ __forceinline__ Raw<T, VEC> load_piece(const T* __restrict__ src, int row, int c, int T_len, int dh) {
    const T* p = src + (size_t)min(row, T_len - 1) * dh;
    Raw<T, VEC> v;
    if constexpr (VEC) {
        v = *reinterpret_cast<const Raw<T, VEC>*>(p + min(c, dh - 4));
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_bit_cast(typename Storage<T>::Bits, p[min(c + e, dh - 1)]);
    }
    return v;
}
template <typename T, typename R>
__device__ __forceinline__ f32x4 keep(const R& raw, bool row_ok, int c, int dh) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const typename Storage<T>::Bits bits = raw[e];
        v[e] = row_ok && c + e < dh ? to_f32(__builtin_bit_cast(T, bits)) : 0.0f;
    }
    return v;
}

// A 32 x DH tile on its way from memory to LDS (pitch DH + 4 floats: the half-row reads of a lane group spread over all
// banks).  Rows past `rows_end` and columns past dh become zero.
template <typename T, int DH, bool VEC>
struct TileStage {
    static constexpr int PITCH = DH + 4, PIECES = TILE * DH / 4 / NT;
    Raw<T, VEC> reg[PIECES];
    __device__ __forceinline__ void fetch(const T* __restrict__ src, int row0, int T_len, int dh, int tid) {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int piece = tid + NT * u;
            reg[u] = load_piece<T, VEC>(src, row0 + piece / (DH / 4), 4 * (piece % (DH / 4)), T_len, dh);
        }
    }
    __device__ __forceinline__ void commit(float* lds, int row0, int rows_end, int dh, int tid) const {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int piece = tid + NT * u, row = piece / (DH / 4), c = 4 * (piece % (DH / 4));
            *reinterpret_cast<f32x4*>(lds + row * PITCH + c) = keep<T>(reg[u], row0 + row < rows_end, c, dh);
        }
    }
};

// The lane's half row (columns h*DH/2 ...) of row `row`, zero outside the matrix.
template <typename T, int DH, bool VEC>
__device__ __forceinline__ void load_half_row(float (&dst)[DH / 2], const T* __restrict__ src, int row, int h,
                                              int T_len, int dh, bool live = true) {
#pragma unroll
    for (int q = 0; q < DH / 8; ++q) {
        const int c = h * (DH / 2) + 4 * q;
        const f32x4 v = keep<T>(load_piece<T, VEC>(src, row, c, T_len, dh), live && row < T_len, c, dh);
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[4 * q + e] = v[e];
    }
}

// Workgroup -> (row tile, group).  The groups lie along x, which is dealt first, and the row tiles along y and z: all
// groups of the longest row tile come first, so that the short tiles of a causal call fill the end of the launch.  Only the first
// `turned` workgroups, one for every CU, come shortest first: where a CU holds two of them, the longest of the second lot joins the
// shortest of the first (B=4 H=8 T=512 Dh=64 P=8, all four kernels: 393 us with both lots longest first, 360 so).  A grid
// may hold fewer than 2^32 threads along x and 65535 workgroups along y and z, so neither lies along x alone.
struct Place {
    int tile, group;
};
__device__ __forceinline__ Place place(bool last_first, int tiles, int turned) {
    int t = (int)(blockIdx.z * gridDim.y + blockIdx.y), group = (int)blockIdx.x;  // past `tiles` in the last row of z: no work
    const long long id = (long long)t * gridDim.x + group;
    if (id < turned) {
        const unsigned from_end = (unsigned)turned - 1 - (unsigned)id;
        t = (int)(from_end / gridDim.x);
        group = (int)(from_end - (unsigned)t * gridDim.x);
    }
    return {last_first ? tiles - 1 - t : t, group};
}
// the workgroups that come shortest first
inline int turned_of(int tiles, int groups) {
    const long long all = (long long)tiles * groups, cus = device_compute_units();
    return (int)(all < cus ? all : cus);
}
inline dim3 grid_of(int tiles, int groups) {
    const int rows = tiles < 65535 ? tiles : 65535;
    return dim3((unsigned)groups, (unsigned)rows, (unsigned)((tiles + rows - 1) / rows));
}

// N matrices streamed through LDS in tiles of 32 rows, STEP +1 from the first to the last, -1 backwards: two buffers of N
// tiles, the next tile in registers during the products of the current one, one barrier per tile.
template <typename T, int DH, bool VEC, int N, int STEP = 1>
struct TileStream {
    using Stage = TileStage<T, DH, VEC>;
    static constexpr int MAT = TILE * Stage::PITCH, BUF = N * MAT;
    static constexpr size_t LDS_BYTES = 2 * BUF * sizeof(float);
    const T* src[N];
    float* lds;
    int T_len, dh, tid, steps;
    Stage stage[N];
    __device__ __forceinline__ void fetch(int it) {
#pragma unroll
        for (int n = 0; n < N; ++n) stage[n].fetch(src[n], it * TILE, T_len, dh, tid);
    }
    __device__ __forceinline__ void commit(int it) {
#pragma unroll
        for (int n = 0; n < N; ++n) stage[n].commit(lds + (it & 1) * BUF + n * MAT, it * TILE, T_len, dh, tid);
    }
    __device__ __forceinline__ void start() {
        const int it = STEP > 0 ? 0 : steps - 1;
        fetch(it);
        commit(it);
        __syncthreads();
    }
    __device__ __forceinline__ bool more(int it) const { return STEP > 0 ? it + 1 < steps : it > 0; }
    __device__ __forceinline__ void begin(int it) {  // the next tile sets out
        if (more(it)) fetch(it + STEP);
    }
    __device__ __forceinline__ void finish(int it) {
        if (more(it)) commit(it + STEP);
        __syncthreads();
    }
    __device__ __forceinline__ const float* tile(int it, int n) const { return lds + (it & 1) * BUF + n * MAT; }
};

__device__ __forceinline__ float sum16(const f32x16& x) {
    float t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = (x[i] + x[i + 4]) + (x[i + 8] + x[i + 12]);
    return (t[0] + t[1]) + (t[2] + t[3]);
}

// The largest score (log2 domain) of a query so far and the sum of 2^(score - largest); the two lanes of a query share `top`.
struct RowSums {
    float top = -INFINITY, sum = 0.0f;
    __device__ __forceinline__ void add(f32x16& s, int j0, int h, int last_key, float sc2) {
        float most = top;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = j0 + acc_row(i, h) <= last_key ? s[i] * sc2 : -INFINITY;
            most = fmaxf(most, s[i]);
        }
        most = fmaxf(most, __shfl_xor(most, 32, 64));
        const float base = most == -INFINITY ? 0.0f : most;  // scores of -inf only so far: their terms are 0
        const float alpha = exp2f(top - base);
        top = most;
        // the terms of a tile in a tree of their own: the running sum rounds once per tile
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = exp2f(s[i] - base);
        sum = sum * alpha + sum16(s);
    }
};

template <typename T, int DH, bool VEC>
__global__ __launch_bounds__(NT) void stats_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                   float* __restrict__ lse2, int T_len, int dh, float scale, int causal,
                                                   int tiles, int turned) {
    constexpr int ROWS = NWAVE * TILE, PITCH = TileStage<T, DH, VEC>::PITCH;
    extern __shared__ __align__(16) float lds[];  // [2][K tile]
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5, wave = tid >> 6;
    const Place at = place(causal, tiles, turned);
    if (at.tile < 0 || at.tile >= tiles) return;
    const size_t base = (size_t)at.group * T_len * dh;
    const int q0 = at.tile * ROWS + wave * TILE, query = q0 + m;
    float qf[1][DH / 2];
    load_half_row<T, DH, VEC>(qf[0], q + base, query, h, T_len, dh);
    RowSums run;
    const float sc2 = scale * LOG2E;
    const int end = causal ? min(T_len, (at.tile + 1) * ROWS) : T_len;
    TileStream<T, DH, VEC, 1> keys{{k + base}, lds, T_len, dh, tid, (end + TILE - 1) / TILE};
    keys.start();
    // this wave's own tiles first, then the rest of the workgroup's (no branch around the products: the accumulators
    // would be copied at its join on every step)
    const int mine = q0 >= T_len ? 0 : causal ? min(keys.steps, q0 / TILE + 1) : keys.steps;
    for (int it = 0; it < mine; ++it) {
        const int j0 = it * TILE;
        keys.begin(it);
        f32x16 ss[1] = {zero16()};
        f32x16& s = ss[0];
        dot_form<DH, 1>(ss, keys.tile(it, 0) + m * PITCH + h * (DH / 2), qf, nothing);
        run.add(s, j0, h, causal ? min(query, T_len - 1) : T_len - 1, sc2);
        keys.finish(it);
    }
    for (int it = mine; it < keys.steps; ++it) {
        keys.begin(it);
        keys.finish(it);
    }
    if (query >= T_len) return;
    const float l_all = run.sum + __shfl_xor(run.sum, 32, 64);
    if (h == 0) lse2[(size_t)at.group * T_len + query] = run.top + log2f(l_all);
}

// The statistics of few rows: a workgroup owns 32 queries and its waves every fourth tile of their keys, each read straight into the
// operand registers, a tile ahead; the four sums of a query meet at the end.  (The kernel above has a workgroup for every 128
// queries, as long as the last of them: a whole call of B=4 H=8 T=512 Dh=64 P=8 370 -> 355 us, B=2 H=8 T=1000 Dh=64 P=4 448 ->
// 415, B=2 H=4 T=512 Dh=128 P=4 387 -> 369.)
template <typename T, int DH, bool VEC>
__global__ __launch_bounds__(NT) void stats_split_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                         float* __restrict__ lse2, int T_len, int dh, float scale, int causal,
                                                         int tiles, int turned) {
    __shared__ float part[NWAVE][2][TILE];  // largest score and sum, by wave
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Place at = place(causal, tiles, turned);
    if (at.tile < 0 || at.tile >= tiles) return;
    const size_t base = (size_t)at.group * T_len * dh;
    const int query = at.tile * TILE + m;
    float qf[1][DH / 2];
    load_half_row<T, DH, VEC>(qf[0], q + base, query, h, T_len, dh);
    const int last_key = causal ? min(query, T_len - 1) : T_len - 1, steps = causal ? at.tile + 1 : tiles;
    const float sc2 = scale * LOG2E;
    RowSums run;
    Raw<T, VEC> next[DH / 8];
    auto fetch = [&](int it) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < DH / 8; ++c) next[c] = load_piece<T, VEC>(k + base, it * TILE + m, h * (DH / 2) + 4 * c, T_len, dh);
    };
    if (wave < steps) fetch(wave);
    for (int it = wave; it < steps; it += NWAVE) {
        f32x4 key[DH / 8];
#pragma unroll
        for (int c = 0; c < DH / 8; ++c) key[c] = keep<T>(next[c], it * TILE + m < T_len, h * (DH / 2) + 4 * c, dh);
        fetch(min(it + NWAVE, steps - 1));
        f32x16 s = zero16();
#pragma unroll
        for (int c = 0; c < DH / 8; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) s = mma(key[c][e], qf[0][4 * c + e], s);
        run.add(s, it * TILE, h, last_key, sc2);
    }
    const float sum = run.sum + __shfl_xor(run.sum, 32, 64);
    if (h == 0) {
        part[wave][0][m] = run.top;
        part[wave][1][m] = sum;
    }
    __syncthreads();
    if (tid >= TILE || query >= T_len) return;
    float top = part[0][0][m];
#pragma unroll
    for (int w = 1; w < NWAVE; ++w) top = fmaxf(top, part[w][0][m]);
    const float base2 = top == -INFINITY ? 0.0f : top;
    float terms[NWAVE];
#pragma unroll
    for (int w = 0; w < NWAVE; ++w) terms[w] = part[w][1][m] * exp2f(part[w][0][m] - base2);
    lse2[(size_t)at.group * T_len + query] = top + log2f((terms[0] + terms[1]) + (terms[2] + terms[3]));
}

// The wave's share of a dq or delta launch.  DW of the four waves own different direction groups of the same rows, 4 / DW
// different row tiles.  A group of the launch is (b, DW * PB directions, head); directions past P in the last group compute
// on zeros and store nothing.
template <int PB, int DW> struct QueryShare {
    int head, b, p0, q0;
    size_t kv;  // first row of (b, head) in units of rows
    __device__ __forceinline__ QueryShare(const Place& at, int wave, int H, int P, int T_len) {
        const int pgroups = (P + DW * PB - 1) / (DW * PB);
        head = at.group % H;
        b = at.group / (H * pgroups);
        p0 = ((at.group / H) % pgroups * DW + wave % DW) * PB;  // the wave's first direction
        kv = ((size_t)b * H + head) * T_len;
        q0 = at.tile * (NWAVE / DW * TILE) + wave / DW * TILE;
    }
    __device__ __forceinline__ size_t row_of(int p, int H, int P, int T_len) const {  // first row of (b, direction, head)
        return (((size_t)b * P + min(p0 + p, P - 1)) * H + head) * T_len;
    }
};

// delta[b,p,h,i] = sum_j P_ij dP_ij from the very P and dP that the next two kernels subtract it from, so that their
// rounding cancels as far as it can (one visible key: dS is exactly zero).  Taken as d_out . O, with O from the statistics
// kernel, it saves these products (the whole call above 0.330 ms), but the error of dQ is 1.04 to 1.14 times as large, and
// with an offset in V up to 1.9 times.
// Two directions per wave at two waves per SIMD, as many as in dq: four at one wave per SIMD share S but hide less, 0.403
// against 0.391 ms for the whole causal call (0.616 and 0.631 without the mask).  The matrix cores are at work for 58 % of its time (47 with
// both lots of workgroups longest first; 61 and 58 in dq and dkdv, one wave per SIMD).
template <typename T, int DH, int PB, int DW, bool VEC>
__global__ __launch_bounds__(NT) void delta_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                   const T* __restrict__ v, const T* __restrict__ d_out,
                                                   const float* __restrict__ lse2, float* __restrict__ delta, int H, int P,
                                                   int T_len, int dh, float scale, int causal, int tiles, int turned) {
    constexpr int ROWS = NWAVE / DW * TILE, PITCH = TileStage<T, DH, VEC>::PITCH;
    extern __shared__ __align__(16) float lds[];  // [2][K tile, V tile]
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Place at = place(causal, tiles, turned);
    if (at.tile < 0 || at.tile >= tiles) return;
    const QueryShare<PB, DW> own(at, wave, H, P, T_len);
    const int query = own.q0 + m;
    float qf[1][DH / 2], gf[PB][DH / 2], sum[PB];
    load_half_row<T, DH, VEC>(qf[0], q + own.kv * dh, query, h, T_len, dh);
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        load_half_row<T, DH, VEC>(gf[p], d_out + own.row_of(p, H, P, T_len) * dh, query, h, T_len, dh, own.p0 + p < P);
        sum[p] = 0.0f;
    }
    const float my_lse = query < T_len ? lse2[own.kv + query] : INFINITY;
    const float sc2 = scale * LOG2E;
    const int end = causal ? min(T_len, (at.tile + 1) * ROWS) : T_len;
    TileStream<T, DH, VEC, 2> keys{{k + own.kv * dh, v + own.kv * dh}, lds, T_len, dh, tid, (end + TILE - 1) / TILE};
    keys.start();
    const int mine = own.q0 >= T_len ? 0 : causal ? min(keys.steps, own.q0 / TILE + 1) : keys.steps;
    const int last_key = causal ? min(query, T_len - 1) : T_len - 1;
    for (int it = 0; it < mine; ++it) {
        keys.begin(it);
        f32x16 ss[1] = {zero16()}, dp[PB];
#pragma unroll
        for (int p = 0; p < PB; ++p) dp[p] = zero16();
        dot_form<DH, 1>(ss, keys.tile(it, 0) + m * PITCH + h * (DH / 2), qf, nothing);
        f32x16& prob = ss[0];
        dot_form<DH, PB>(dp, keys.tile(it, 1) + m * PITCH + h * (DH / 2), gf, [&](int i) __attribute__((always_inline)) {
            prob[i] = prob_of(prob[i], sc2, my_lse);
        });
#pragma unroll
        for (int p = 0; p < PB; ++p) {
#pragma unroll
            for (int i = 0; i < 16; ++i) dp[p][i] = it * TILE + acc_row(i, h) <= last_key ? prob[i] * dp[p][i] : 0.0f;
            sum[p] += sum16(dp[p]);
        }
        keys.finish(it);
    }
    for (int it = mine; it < keys.steps; ++it) {
        keys.begin(it);
        keys.finish(it);
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        const float all = sum[p] + __shfl_xor(sum[p], 32, 64);
        if (own.p0 + p < P && h == 0 && query < T_len) delta[own.row_of(p, H, P, T_len) + query] = all;
    }
}

template <typename T, int DH, int PB, int DW, bool VEC>
__global__ __launch_bounds__(NT) void dq_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                const T* __restrict__ v, const T* __restrict__ d_out,
                                                const float* __restrict__ lse2, const float* __restrict__ delta,
                                                T* __restrict__ dq, int H, int P, int T_len, int dh, float scale,
                                                int causal, int tiles, int turned) {
    constexpr int ROWS = NWAVE / DW * TILE, PITCH = TileStage<T, DH, VEC>::PITCH, NB = DH / 32;
    extern __shared__ __align__(16) float lds[];  // [2][K tile, V tile]
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Place at = place(causal, tiles, turned);
    if (at.tile < 0 || at.tile >= tiles) return;
    const QueryShare<PB, DW> own(at, wave, H, P, T_len);
    const int q0 = own.q0, query = q0 + m;
    float qf[1][DH / 2], gf[PB][DH / 2], dl[PB];
    load_half_row<T, DH, VEC>(qf[0], q + own.kv * dh, query, h, T_len, dh);
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        const size_t row = own.row_of(p, H, P, T_len);
        load_half_row<T, DH, VEC>(gf[p], d_out + row * dh, query, h, T_len, dh, own.p0 + p < P);
        dl[p] = delta[row + min(query, T_len - 1)];
    }
    const float my_lse = query < T_len ? lse2[own.kv + query] : INFINITY;  // P = 0 past the end
    f32x16 acc[PB][NB];
#pragma unroll
    for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[p][n] = zero16();
    const float sc2 = scale * LOG2E;
    const int end = causal ? min(T_len, (at.tile + 1) * ROWS) : T_len;
    // from the diagonal backwards: the one tile with keys that some query may not see comes first, on empty sums
    TileStream<T, DH, VEC, 2, -1> keys{{k + own.kv * dh, v + own.kv * dh}, lds, T_len, dh, tid, (end + TILE - 1) / TILE};
    keys.start();
    auto step = [&](int it, auto first) __attribute__((always_inline)) {
        keys.begin(it);
        const float* kt = keys.tile(it, 0);
        f32x16 ss[1] = {zero16()}, dp[PB];
#pragma unroll
        for (int p = 0; p < PB; ++p) dp[p] = zero16();
        dot_form<DH, 1>(ss, kt + m * PITCH + h * (DH / 2), qf, nothing);
        f32x16& prob = ss[0];
        dot_form<DH, PB>(dp, keys.tile(it, 1) + m * PITCH + h * (DH / 2), gf, [&](int i) __attribute__((always_inline)) {
            prob[i] = prob_of(prob[i], sc2, my_lse);
        });
        const int last_key = (causal ? min(query, T_len - 1) : T_len - 1) - it * TILE;
        chain_form<NB, PITCH, PB>(acc, kt + 4 * h * PITCH + m, dp, [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < PB; ++p) {
                dp[p][i] = prob[i] * (dp[p][i] - dl[p]);
                if (first.value && acc_row(i, h) > last_key) dp[p][i] = 0.0f;
            }
        });
        if (first.value && causal)
            mend_diagonal<NB, PITCH, PB>(acc, kt + m, dp, h, [&](int r, int row) __attribute__((always_inline)) {
                return q0 + r >= it * TILE + row;
            });
        keys.finish(it);
    };
    // the steps of the workgroup's later queries first, then this wave's own (no branch around the products: the
    // accumulators would be copied at its join on every step)
    const int top = q0 >= T_len ? -1 : causal ? q0 / TILE : keys.steps - 1;
    for (int it = keys.steps - 1; it > top; --it) {
        keys.begin(it);
        keys.finish(it);
    }
    if (top >= 0) {
        step(top, std::true_type{});
        for (int it = top - 1; it >= 0; --it) step(it, std::false_type{});
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        if (own.p0 + p >= P) break;
        T* out = dq + own.row_of(p, H, P, T_len) * dh;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int row = q0 + acc_row(i, h), c = 32 * n + m;
                if (row < T_len && c < dh) store(out + (size_t)row * dh + c, acc[p][n][i] * scale);
            }
    }
}

template <typename T, int DH, int PB, int DW, bool VEC>
__global__ __launch_bounds__(NT) void dkdv_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                  const T* __restrict__ v, const T* __restrict__ d_out,
                                                  const float* __restrict__ lse2, const float* __restrict__ delta,
                                                  T* __restrict__ dk, T* __restrict__ dv, int H, int P,
                                                  int T_len, int dh, float scale, int causal, int tiles, int turned) {
    using Stage = TileStage<T, DH, VEC>;
    constexpr int PITCH = Stage::PITCH, NB = DH / 32, ROWS = NWAVE / DW * TILE;
    constexpr int ND = DW * PB;  // directions of the workgroup
    constexpr int MATS = (1 + ND) * TILE * PITCH, BUF = MATS + 2 * NT;
    extern __shared__ __align__(16) float lds[];  // [2][Q tile, ND d_out tiles, lse of the rows, ND deltas of the rows]
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Place at = place(false, tiles, turned);  // the first keys see the most queries
    if (at.tile >= tiles) return;
    const int pgroups = (P + ND - 1) / ND;
    const int head = at.group % H, b = at.group / (H * pgroups);
    const int dir0 = (at.group / H) % pgroups * ND;                   // the workgroup's first direction
    const int d0 = wave % DW * PB;                                    // the wave's first one behind it
    const size_t rows = (size_t)T_len, bh = (size_t)b * H + head, kv_base = bh * rows * dh;
    const int k0 = at.tile * ROWS + wave / DW * TILE, key = k0 + m;
    float kf[1][DH / 2], vf[1][DH / 2];
    load_half_row<T, DH, VEC>(kf[0], k + kv_base, key, h, T_len, dh);
    load_half_row<T, DH, VEC>(vf[0], v + kv_base, key, h, T_len, dh);
    f32x16 acc_k[PB][1][NB], acc_v[PB][1][NB];
#pragma unroll
    for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc_k[p][0][n] = acc_v[p][0][n] = zero16();
    const float sc2 = scale * LOG2E;
    const int first = causal ? at.tile * (ROWS / TILE) : 0;
    const int steps = (T_len + TILE - 1) / TILE;
    Stage qs, gs[ND];
    float row_value[2];  // lse and deltas of the next tile's rows, one or two per thread
    auto fetch = [&](int it) {
        const int i0 = it * TILE;
        qs.fetch(q + kv_base, i0, T_len, dh, tid);
#pragma unroll
        for (int p = 0; p < ND; ++p) {
            const size_t bph = ((size_t)b * P + min(dir0 + p, P - 1)) * H + head;
            gs[p].fetch(d_out + bph * rows * dh, i0, T_len, dh, tid);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int which = min((tid + NT * u) / TILE, ND), row = min(i0 + tid % TILE, T_len - 1);
            const int p = min(dir0 + which - 1, P - 1);
            row_value[u] = *(which == 0 ? lse2 + bh * rows + row : delta + (((size_t)b * P + p) * H + head) * rows + row);
        }
    };
    auto commit = [&](int it) {
        const int i0 = it * TILE;
        float* dst = lds + (it & 1) * BUF;
        qs.commit(dst, i0, T_len, dh, tid);
#pragma unroll
        for (int p = 0; p < ND; ++p)
            gs[p].commit(dst + (1 + p) * TILE * PITCH, i0, dir0 + p < P ? T_len : 0, dh, tid);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            dst[MATS + tid + NT * u] = i0 + tid % TILE < T_len ? row_value[u] : 0.0f;
    };
    fetch(first);
    commit(first);
    __syncthreads();
    // the steps of the workgroup's earlier keys first, then this wave's own (no branch around the products: the
    // accumulators would be copied at its join on every step)
    const int own = k0 >= T_len ? steps : causal ? k0 / TILE : first;
    for (int it = first; it < own; ++it) {
        if (it + 1 < steps) fetch(it + 1);
        if (it + 1 < steps) commit(it + 1);
        __syncthreads();
    }
    auto step = [&](int it, auto diagonal) __attribute__((always_inline)) {
        const int i0 = it * TILE;
        if (it + 1 < steps) fetch(it + 1);
        const float* qt = lds + (it & 1) * BUF;
        const float* stat = qt + MATS;
        f32x16 ss[1] = {zero16()};
        f32x16& s = ss[0];
        dot_form<DH, 1>(ss, qt + m * PITCH + h * (DH / 2), kf, nothing);
        // queries of the tile that see the lane's key and exist
        const int from = causal ? key - i0 : 0, to = T_len - i0;
        auto sees = [&](int r) __attribute__((always_inline)) { return r < to && (!diagonal.value || r >= from); };
        f32x4 lse4[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) lse4[g] = *reinterpret_cast<const f32x4*>(stat + 8 * g + 4 * h);
        f32x16 dps[PB][1];
        auto mend = [&](int p) __attribute__((always_inline)) {
            auto seen = [&](int r, int row) __attribute__((always_inline)) { return i0 + row >= k0 + r; };
            mend_diagonal<NB, PITCH, 1>(acc_v[p], qt + (1 + d0 + p) * TILE * PITCH + m, ss, h, seen);
            mend_diagonal<NB, PITCH, 1>(acc_k[p], qt + m, dps[p], h, seen);
        };
#pragma unroll
        for (int p = 0; p < PB; ++p) {
            const float* gt = qt + (1 + d0 + p) * TILE * PITCH;
            f32x16& dp = dps[p][0];
            dp = zero16();
            if (p == 0)
                dot_form<DH, 1>(dps[p], gt + m * PITCH + h * (DH / 2), vf, [&](int i) __attribute__((always_inline)) {
                    s[i] = sees(acc_row(i, h)) ? prob_of(s[i], sc2, lse4[i >> 2][i & 3]) : 0.0f;
                });
            else
                dot_form<DH, 1>(dps[p], gt + m * PITCH + h * (DH / 2), vf, nothing);
            f32x4 d4[4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
                d4[g] = *reinterpret_cast<const f32x4*>(stat + (1 + d0 + p) * TILE + 8 * g + 4 * h);
            chain_form<NB, PITCH, 1>(acc_v[p], gt + 4 * h * PITCH + m, ss, [&](int i) __attribute__((always_inline)) {
                dp[i] = sees(acc_row(i, h)) ? s[i] * (dp[i] - d4[i >> 2][i & 3]) : 0.0f;
            });
            chain_form<NB, PITCH, 1>(acc_k[p], qt + 4 * h * PITCH + m, dps[p], nothing);
            if (diagonal.value && causal && p + 1 < PB) mend(p);
        }
        if (it + 1 < steps) commit(it + 1);
        if (diagonal.value && causal) mend(PB - 1);  // the registers of the next tile are free again
        __syncthreads();
    };
    if (own < steps) {
        step(own, std::true_type{});
        for (int it = own + 1; it < steps; ++it) step(it, std::false_type{});
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
        if (dir0 + d0 + p >= P) break;
        const size_t base = (((size_t)b * P + dir0 + d0 + p) * H + head) * rows * dh;
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int row = k0 + acc_row(i, h), c = 32 * n + m;
                if (row < T_len && c < dh) {
                    store(dk + base + (size_t)row * dh + c, acc_k[p][0][n][i] * scale);
                    store(dv + base + (size_t)row * dh + c, acc_v[p][0][n][i]);
                }
            }
    }
}

template <typename T> struct Args {
    const T *q, *k, *v, *d_out;
    T *dq, *dk, *dv;
    float *lse2, *delta;
    int B, H, T_len, dh, P, causal;
    float scale;
    hipStream_t stream;
};

template <int DH, int PB, int DW, bool VEC, typename T>
int launch_with(const Args<T>& a) {
    constexpr int PITCH = TileStage<T, DH, VEC>::PITCH, ROWS = NWAVE / DW * TILE, ND = DW * PB;
    constexpr size_t k_bytes = TileStream<T, DH, VEC, 1>::LDS_BYTES, kv_bytes = TileStream<T, DH, VEC, 2>::LDS_BYTES;
    constexpr size_t qg_bytes = (size_t)2 * ((1 + ND) * TILE * PITCH + 2 * NT) * sizeof(float);
    static_assert(qg_bytes <= 160 * 1024 && (1 + ND) * TILE <= 2 * NT, "LDS budget");
    const int heads = a.B * a.H, groups = heads * ((a.P + ND - 1) / ND);
    const int tiles = (a.T_len + ROWS - 1) / ROWS, stat_tiles = (a.T_len + NWAVE * TILE - 1) / (NWAVE * TILE);
    if ((long long)groups * NT >= 1LL << 32)  // before the first launch: a refused call writes nothing
        return fail(LBI_ERR_UNSUPPORTED, "lbi_attn_pullback: too many (batch, head, direction) groups for one launch");
    if (int rc = ensure_dynamic_lds<&stats_kernel<T, DH, VEC>>(k_bytes)) return rc;
    if (int rc = ensure_dynamic_lds<&delta_kernel<T, DH, PB, DW, VEC>>(kv_bytes)) return rc;
    if (int rc = ensure_dynamic_lds<&dq_kernel<T, DH, PB, DW, VEC>>(kv_bytes)) return rc;
    if (int rc = ensure_dynamic_lds<&dkdv_kernel<T, DH, PB, DW, VEC>>(qg_bytes)) return rc;
    const int key_tiles = (a.T_len + TILE - 1) / TILE, turned = turned_of(tiles, groups);
    // the largest number of workgroups of the other statistics kernel at which this one was as fast or faster: B=8 H=8 T=512 P=1 224 -> 217 us
    // with a mask (256), 223 -> 226 without; B=4 H=8 T=2048 Dh=128 (512) 1579 -> 1610 and 2841 -> 2924.  One tile of keys has nothing to split (B H=28 T=21
    // Dh=128 P=15 48 -> 49)
    if (key_tiles > 1 && 4LL * stat_tiles * heads <= (a.causal ? 4LL : 3LL) * device_compute_units())
        hipLaunchKernelGGL((stats_split_kernel<T, DH, VEC>), grid_of(key_tiles, heads), dim3(NT), 0, a.stream, a.q, a.k, a.lse2,
                           a.T_len, a.dh, a.scale, a.causal, key_tiles, turned_of(key_tiles, heads));
    else
        hipLaunchKernelGGL((stats_kernel<T, DH, VEC>), grid_of(stat_tiles, heads), dim3(NT), k_bytes, a.stream, a.q, a.k,
                           a.lse2, a.T_len, a.dh, a.scale, a.causal, stat_tiles, turned_of(stat_tiles, heads));
    hipLaunchKernelGGL((delta_kernel<T, DH, PB, DW, VEC>), grid_of(tiles, groups), dim3(NT), kv_bytes, a.stream, a.q, a.k, a.v,
                       a.d_out, a.lse2, a.delta, a.H, a.P, a.T_len, a.dh, a.scale, a.causal, tiles, turned);
    hipLaunchKernelGGL((dq_kernel<T, DH, PB, DW, VEC>), grid_of(tiles, groups), dim3(NT), kv_bytes, a.stream, a.q, a.k, a.v,
                       a.d_out, a.lse2, a.delta, a.dq, a.H, a.P, a.T_len, a.dh, a.scale, a.causal, tiles, turned);
    hipLaunchKernelGGL((dkdv_kernel<T, DH, PB, DW, VEC>), grid_of(tiles, groups), dim3(NT), qg_bytes, a.stream,
                       a.q, a.k, a.v, a.d_out, a.lse2, a.delta, a.dk, a.dv, a.H, a.P, a.T_len, a.dh, a.scale, a.causal,
                       tiles, turned);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

// How many waves of a workgroup take different directions: as many as there are direction groups (MAX at most: what the
// d_out tiles leave of the LDS), fewer where that leaves fewer waves without a direction.  One where few workgroups of one
// or two row tiles leave half of the CUs idle anyway: a tile of one direction is loaded sooner (B=4 H=8 T=32 Dh=33 P=4:
// 39 -> 33 us; with a workgroup for every CU or more it takes up to twice as long).
template <int PB, int MAX, typename T> int waves_apart(const Args<T>& a) {
    const int pgroups = (a.P + PB - 1) / PB;
    auto padded = [&](int dw) { return (pgroups + dw - 1) / dw * dw; };
    if (a.T_len <= 2 * TILE && (long long)a.B * a.H * pgroups <= device_compute_units() / 2) return 1;
    if (MAX >= 4 && padded(4) == padded(2) && pgroups > 2) return 4;
    return padded(2) == pgroups || pgroups > 2 ? 2 : 1;
}

template <int DH, int PB, int MAX, bool VEC, typename T> int launch_directions(const Args<T>& a) {
    const int dw = waves_apart<PB, MAX>(a);
    if constexpr (MAX >= 4)
        if (dw == 4) return launch_with<DH, PB, 4, VEC>(a);
    return dw == 2 ? launch_with<DH, PB, 2, VEC>(a) : launch_with<DH, PB, 1, VEC>(a);
}

// Tiles that a CU goes through at PB directions per wave, one workgroup after another: those of the longest one at least.
template <int PB, typename T> double steps_of_a_cu(const Args<T>& a) {
    const int dw = waves_apart<PB, 4>(a), rows = NWAVE / dw, nd = dw * PB;
    const double steps = (a.T_len + TILE - 1) / TILE, tiles = (a.T_len + rows * TILE - 1) / (rows * TILE);
    const double cus = device_compute_units(), groups = (double)a.B * a.H * ((a.P + nd - 1) / nd);
    if (!a.causal || tiles == 1.0) return steps * ceil(groups * tiles / cus);
    return std::max(steps, groups * tiles * (steps + rows) / (2 * cus));
}

// Two directions per wave share S: 15 products for the two and not 18.  One makes for twice the workgroups, half as long: taken
// where few long ones leave CUs idle.  The line lies at 3 / 2, below 5 / 3, since a wave does less well with one (us, with one and
// with two): B=1 H=2 T=1000 Dh=64 P=8 430 and 637, B=4 H=8 T=512 P=2 226 and 329, B=2 H=8 T=1000 P=4 417 and 591, B=5 H=1 T=1761 Dh=32
// P=8 430 and 589; B=4 H=8 T=512 Dh=64 P=8 427 and 354, B=8 H=5 T=320 P=8 248 and 215.  Where a row tile is all there is, workgroups are alike, and whole
// rounds of them count under the mask, too: B H=100 T=21 Dh=64 P=9 45 and 67, 54 T=62 P=18 79 and 118.
template <typename T> bool two_directions(const Args<T>& a) {
    return a.P >= 2 && 1.5 * steps_of_a_cu<2>(a) <= steps_of_a_cu<1>(a);
}

template <typename T>
int launch_typed(const void* q, const void* k, const void* v, const void* d_out, void* dq, void* dk, void* dv,
                 float* workspace, int B, int H, int T_len, int dh, int P, float scale, int causal, hipStream_t stream) {
    const Args<T> a{static_cast<const T*>(q), static_cast<const T*>(k), static_cast<const T*>(v),
                    static_cast<const T*>(d_out), static_cast<T*>(dq), static_cast<T*>(dk), static_cast<T*>(dv),
                    workspace, workspace + (size_t)B * H * T_len, B, H, T_len, dh, P, causal, scale, stream};
    if (!aligned(dh, sizeof(T), {q, k, v, d_out})) {
        if (dh <= 32) return launch_directions<32, 1, 4, false>(a);
        if (dh <= 64) return launch_directions<64, 1, 4, false>(a);
        return dh <= 96 ? launch_directions<96, 1, 4, false>(a) : launch_directions<128, 1, 2, false>(a);
    }
    if (dh <= 32) return two_directions(a) ? launch_directions<32, 2, 4, true>(a) : launch_directions<32, 1, 4, true>(a);
    if (dh <= 64) return two_directions(a) ? launch_directions<64, 2, 4, true>(a) : launch_directions<64, 1, 4, true>(a);
    if (dh <= 96) return launch_directions<96, 1, 4, true>(a);
    return launch_directions<128, 1, 2, true>(a);
}

}  // namespace
}  // namespace attn_f32
}  // namespace lbi
