// Suffix scan of narrow matrices (widths up to 128) on the fp32 matrix cores, in 16 x 16 tiles.
//
// What bounds a narrow scan is the length of a step, not the chip: B column-block chains of K dependent products, each of a few
// hundred cycles of matrix work.  A wave therefore owns ONE row tile of 16 (v_mfma_f32_16x16x4_f32: 32 cycles for four k, the
// rate of the 32 x 32 form at a quarter of its tile), a workgroup all NT row tiles of 16 CT columns.  Against waves of 32 x 32 tiles
// a step has a quarter of the dependent matrix work at CT = 1, and twice the workgroups share it.
//  * Operand layout (lane = 16 q + m): A: A[m][k(q)], B: B[k(q)][m], C: register i holds C[4 q + i][m].  Which k feeds which
//    slot is free, so a lane brings four CONSECUTIVE k of its row, 16 t + 4 q + [0, 4), to four products (one 16-byte load; four
//    lanes cover 64 bytes of a row).  The suffix block is kept transposed in LDS, St[col][k], so the matching B values are one
//    16-byte read and a result one 16-byte write (pitch 16 NT + 4 floats: the 16 lanes of either meet all 64 banks).
//  * The k of the wave's own rows come first: their B values ARE the accumulators of the step before, so four products run
//    while the other waves' rows arrive.  One barrier a step.
//  * The matrices do not depend on the chain: each slot of a register ring is refilled, right after its use, with the same tile
//    AHEAD steps further down.  A narrow step takes less time than a load.
//  * Sums are blocked: the products of two k tiles (32) in an accumulator of their own, those of the wave's own rows, which hold the
//    diagonal, in four.  The matrices of this scan are the identity and a small update: the sum of all else meets the large term once.
//  * The cotangent chain is a workgroup of its own per chain: a column block that holds the vector in one column.  It costs
//    the matrix blocks nothing and takes no longer than they do.
// The chunk phases of ScanPlan (1, 2, 3) are the same loop from another start state; the vector rides on the last chunk of phase 1 and
// on phase 3, where it starts from the finished boundary product applied to g.
// Rows come straight into registers up to 48 columns.  Beyond that each lane loading another row would be what bounds a step: sixteen
// 64-byte pieces an instruction come at 35 GB/s per CU (d = 128 1.85 us a step, 1.06 without the loads).  They go through LDS there, by
// 16-byte transfers into a ring of the wave's own, four lanes to 64 bytes of a row (1.23 us).
// A step takes (fp32, B = 1, K = 256 less K = 56) 0.15 / 0.24 / 0.42 / 0.98 / 1.30 us at d = 16 / 32 / 64 / 96 / 128, of which 0.06 / 0.11 / 0.23 / 0.7 /
// 0.9 are the fp32 products at the rate of the matrix cores.  Whole calls, old (scalar or 32 x 32 tiles) -> here, us, matrices and cotangents,
// inputs from memory: fp32 B = 17 K = 73 d = 16 133 -> 14; B = 18 K = 101 d = 64 86 -> 47; B = 3 K = 10 d = 128 36 -> 17; B = 64 K = 45 d = 128
// 176 -> 145.  Error against fp64 (2-norm, identity plus update), over 400 random calls: 0.54 of before (matrices), 0.68 (cotangents).
#pragma once

#include <type_traits>

#include "lbi_scan_narrow.h"
#include "lbi_scan_planes.h"

namespace lbi {
namespace scan_narrow {

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Four elements of a row as they are stored.  They are widened where they are used: at the load, the compiler would wait for it.
template <typename Tin> struct Row4 {
    typedef unsigned int type __attribute__((ext_vector_type(2)));
    typedef unsigned int type_at __attribute__((ext_vector_type(2), aligned(2)));
    static __device__ __forceinline__ f32x4 widen(type w) {
        f32x4 x;
        const u16x4 v = __builtin_bit_cast(u16x4, w);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned short one = v[i];
            x[i] = to_f32(__builtin_bit_cast(Tin, one));
        }
        return x;
    }
};
template <> struct Row4<float> {
    typedef f32x4 type;
    typedef float type_at __attribute__((ext_vector_type(4), aligned(4)));
    static __device__ __forceinline__ f32x4 widen(f32x4 w) { return w; }
};

// f(integral_constant<int, i>) for i = FROM ... TO - 1.
template <int FROM, int TO, typename F> __device__ __forceinline__ void for_each(F&& f) {
    if constexpr (FROM < TO) {
        f(std::integral_constant<int, FROM>{});
        for_each<FROM + 1, TO>(f);
    }
}

// Steps that a row tile is requested ahead of its use: about 96 registers of rows in flight.
constexpr int ahead(int NT) { return NT <= 2 ? 8 : NT <= 4 ? 6 : NT <= 6 ? 4 : 3; }

// RAGGED: d < 16 NT, any alignment of single elements; rows and columns past the end are zero on chip.
// RING: rows come straight into registers (0), or through LDS, RING steps ahead.
template <typename Tin, int NT, int CT, bool RAGGED, int RING>
__global__ __launch_bounds__(64 * NT, 2) void scan_narrow_kernel(const Tin* __restrict__ mats, float* __restrict__ out,
                                                              const float* __restrict__ g, float* __restrict__ cot, int B, int K,
                                                              int d_rt, int carry, ScanPlan plan) {
    constexpr int D = 16 * NT, CB = 16 * CT, NB = (NT + CT - 1) / CT, PITCH = D + 4, AHEAD = ahead(NT);
    const int d = RAGGED ? d_rt : D;
    const size_t dd = (size_t)d * d;
    constexpr int TPS = RING > 0 && sizeof(Tin) == 2 ? 2 : 1;   // k tiles in a slot of the ring: 64 bytes of 16 rows
    constexpr int SPS = NT / TPS;                               // slots of a step
    static_assert(RING == 0 || (NT >= 4 && NT % TPS == 0), "whole slots, and three tiles within two steps");
    extern __shared__ __align__(16) char smem[];                // [2][CB][PITCH] floats, (CT > 1) [2][D], [NT] rings
    float* st = reinterpret_cast<float*>(smem);

    // A launch covers E chains of NBX column blocks, dealt so that the blocks of one chain share an XCD (ids equal mod 8).
    const int phase = plan.phase;
    const int nseg = phase == 1 || phase == 3 ? plan.C - 1 : 1;
    const bool carried = CT > 1 && carry && cot;   // the first column block carries the vector, too
    const bool alone = !out;                       // the cotangent chain without the matrices
    const int nbx = alone ? 1 : NB + (cot && !carried ? 1 : 0);
    const int E = B * nseg;
    const int id = blockIdx.x;
    int e, block;
    if (E >= 8) {
        const int slot = id >> 3;
        e = (slot / nbx) * 8 + (id & 7);
        block = slot % nbx;
    } else {
        e = id / nbx;
        block = id % nbx;
    }
    if (e >= E) return;
    const bool chain = alone || block == NB;
    const int c0 = block * CB;
    const int b = e / nseg, seg = e - b * nseg;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, m = lane & 15, q = lane >> 4;
    const int row0 = 16 * wave, row = row0 + 4 * q;   // the rows of this lane's results: row ... row + 3

    // Steps r = r_top ... r_lo multiply a_base[r a_stride] onto the running block (see ScanPlan); it starts as `init_a` (storage
    // type) or `init_s` (fp32, a product computed earlier).
    float* out_b = out + (size_t)b * (K + 1) * dd;
    const Tin* a_base = mats + (size_t)b * K * dd;
    float* o_base = out_b;
    const Tin* init_a = nullptr;
    const float* init_s = nullptr;
    int r_top, r_lo = 0;
    bool write_tail = false, store_all = true;
    size_t stride = dd;
    if (phase == 0) {
        init_a = a_base + (size_t)(K - 1) * dd;
        r_top = K - 2;
        write_tail = true;
    } else if (phase == 1) {
        const int c = seg + 1;
        const bool last = c == plan.C - 1;
        if (chain && !last) return;
        const int end = last ? K : (c + 1) * plan.L - plan.s;
        init_a = a_base + (size_t)(end - 1) * dd;
        r_top = end - 2;
        r_lo = c * plan.L - plan.s;
        write_tail = last;
        store_all = last;
    } else if (phase == 2) {
        // the totals, each parked one slot above the first matrix of its chunk (Tin is float here)
        a_base = reinterpret_cast<const Tin*>(out_b + (size_t)(plan.L - plan.s + 1) * dd);
        o_base = out_b + (size_t)(plan.L - plan.s) * dd;
        stride = (size_t)plan.L * dd;
        init_s = out_b + (size_t)((plan.C - 1) * plan.L - plan.s) * dd;
        r_top = plan.C - 3;
    } else {
        const int c = seg;
        init_s = out_b + (size_t)((c + 1) * plan.L - plan.s) * dd;
        r_top = (c + 1) * plan.L - plan.s - 1;
        r_lo = c == 0 ? 0 : c * plan.L - plan.s + 1;
    }

    // This lane's 4 elements of row row0 + m in the k tile that its wave takes j-th.
    const unsigned a_row = RAGGED && row0 + m >= d ? 0u : (unsigned)((row0 + m) * d);
    auto tile_of = [&](int j) __attribute__((always_inline)) {
        if constexpr (TPS == 2) {   // its own tile, the other one of that slot, then the other slots
            if (j < 2) return wave ^ j;
            const int pair = (wave >> 1) + j / 2;
            return 2 * (pair < SPS ? pair : pair - SPS) + j % 2;
        }
        return wave + j < NT ? wave + j : wave + j - NT;
    };
    unsigned a_at[NT];            // byte offsets from a matrix
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const unsigned k = 16 * tile_of(j) + 4 * q;
        a_at[j] = (a_row + (!RAGGED || k < (unsigned)d ? k : 0)) * (unsigned)sizeof(Tin);
    }
    auto load_tile = [&](const Tin* mat, int j) __attribute__((always_inline)) {
        using Stored = Row4<Tin>;
        const char* p = reinterpret_cast<const char*>(mat) + a_at[j];
        if constexpr (RAGGED) return (typename Stored::type)*reinterpret_cast<const typename Stored::type_at*>(p);
        else return *reinterpret_cast<const typename Stored::type*>(p);
    };
    // The start state's elements are requested first and used once the first rows are on their way: what is requested last is
    // waited for with all that came before it.
    f32x4 own[CT];
    f32x4 val[NT], vec[NT];
    const float* g_b = g + (size_t)b * d;
    const bool vector = chain || (carried && block == 0 && (phase != 1 || seg + 1 == plan.C - 1));
    if (vector) {
        // (nothing past the end of a row: there may be nothing behind the last matrix)
        auto elements = [&](const auto* p, bool there, int k) __attribute__((always_inline)) {
            using T = typename std::remove_cv<typename std::remove_reference<decltype(*p)>::type>::type;
            if (!RAGGED || (there && k + 3 < d)) return Row4<T>::widen((typename Row4<T>::type)*reinterpret_cast<const typename Row4<T>::type_at*>(p + k));
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (there && k + x < d) v[x] = to_f32(p[k + x]);
            return v;
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int k = 16 * t + 4 * q;
            val[t] = phase != 3 ? elements(init_a + a_row, row0 + m < d, k) : elements(init_s + a_row, row0 + m < d, k);
            vec[t] = elements(g_b, true, k);
        }
    }
    if (!chain) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int col = c0 + 16 * c + m;
                const bool there = row + x < d && col < d;
                const unsigned off = there ? (unsigned)((row + x) * d + col) : 0u;
                own[c][x] = phase < 2 ? to_f32(init_a[off]) : init_s[off];
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    constexpr int FRAGS = 4, RA = FRAGS - 1;   // the ring in LDS: tiles in registers, and how far ahead they are read
    typename Row4<Tin>::type ring[RING > 0 ? FRAGS : AHEAD][RING > 0 ? 1 : NT];
    constexpr unsigned kNowhere = 0x80000000u;
    // The ring in LDS: slots in the order of their use.  16-byte piece p of row i lies at p ^ (i / 4) % 4 (the 16 lanes of a read meet
    // all banks).
    constexpr unsigned SLOT = 1024, RING_BYTES = (RING > 0 ? RING : 1) * SPS * SLOT;
    const unsigned ring0 = (NT > 1 ? 2 * CB * PITCH * 4 : 0) + (CT > 1 ? 2 * D * 4 : 0) + wave * RING_BYTES;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
    const int dma_row = row0 + (lane >> 2);
    const unsigned dma_lane = !RAGGED || dma_row < d
        ? (unsigned)(dma_row * d) * (unsigned)sizeof(Tin) + (((lane & 3) ^ ((lane >> 4) & 3)) << 4) : kNowhere;
    const unsigned stored_bytes = (unsigned)(dd * sizeof(Tin));
    auto request = [&](const Tin* mat, int j, unsigned slot) __attribute__((always_inline)) {
        scan_planes::dma16(scan_planes::rows(mat, stored_bytes), dma_lane, (unsigned)(tile_of(j) / TPS) * 64u, lds0 + slot);
    };
    if (r_top >= r_lo) {
        if constexpr (RING > 0) {
#pragma unroll
            for (int u = 0; u < RING; ++u) {
                const int rr = r_top - u;
#pragma unroll
                for (int i = 0; i < SPS; ++i)
                    request(a_base + (size_t)(rr > r_lo ? rr : r_lo) * stride, i * TPS, ring0 + (u * SPS + i) * SLOT);
            }
        } else {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int rr = r_top - u;
                if (rr < r_lo) break;   // (rows that nothing uses: bf16 B = 32 K = 2, d = 65 9.6 -> 7.2 us without, d = 113 11.2 -> 8.2)
#pragma unroll
                for (int j = 0; j < NT; ++j) ring[u][j] = load_tile(a_base + (size_t)rr * stride, j);
                __builtin_amdgcn_sched_barrier(0);   // in the order in which they are used
            }
        }
    }
    // Start state.  The vector's block keeps it in column 0; what the other columns hold is never looked at.
    unsigned at[CT];              // byte offset of this lane's first result; past everything where there is none
    unsigned row_bytes = (unsigned)d * 4, result_bytes = (unsigned)dd * 4;
    size_t o_stride = stride;
    float* cot_b = cot ? cot + (size_t)b * (K + 1) * d : nullptr;
    float sum = 0.0f;             // of row row0 + m of the vector
    if (vector) {
        const bool from_a = phase != 3;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float part = 0.0f;
#pragma unroll
            for (int x = 0; x < 4; ++x) part = fmaf(val[t][x], vec[t][x], part);
            sum += part;
        }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        // its own place: behind the last chunk's matrices, or the boundary (phase 1 has written the last one's)
        const int place = from_a ? K - 1 : r_top + 1;
        if ((from_a || seg + 1 < plan.C - 1) && q == 0 && row0 + m < d) {
            cot_b[(size_t)place * d + row0 + m] = sum;
            if (from_a) cot_b[(size_t)K * d + row0 + m] = g_b[row0 + m];
        }
    }
    if (chain) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const float v = __shfl(sum, 4 * q + x, 64);
            own[0][x] = m == 0 ? v : 0.0f;
        }
#pragma unroll
        for (int c = 1; c < CT; ++c) own[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < CT; ++c) at[c] = c == 0 && m == 0 ? (unsigned)row * 4 : kNowhere;
        row_bytes = 4;
        result_bytes = (unsigned)d * 4;
        o_base = cot_b;
        o_stride = d;
        store_all = true;
    } else {
        float* o_last = out_b + (size_t)(K - 1) * dd;
        float* o_eye = out_b + (size_t)K * dd;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int col = c0 + 16 * c + m;
            at[c] = col < d ? (unsigned)(row * d + col) * 4 : kNowhere;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                own[c][x] = row + x < d && col < d ? own[c][x] : 0.0f;
            }
        }
        if (write_tail) {
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const int col = c0 + 16 * c + m;
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    if (row + x < d && col < d) {
                        o_last[(size_t)(row + x) * d + col] = own[c][x];
                        o_eye[(size_t)(row + x) * d + col] = row + x == col ? 1.0f : 0.0f;
                    }
            }
        }
    }
    if (r_top < r_lo) return;

    unsigned b_at[NT];            // this lane's 4 rows of the j-th tile in the block
#pragma unroll
    for (int j = 0; j < NT; ++j) b_at[j] = (unsigned)(m * PITCH + 16 * tile_of(j) + 4 * q);
    auto publish = [&](int buffer) __attribute__((always_inline)) {
        if constexpr (NT > 1) {
#pragma unroll
            for (int c = 0; c < CT; ++c) *reinterpret_cast<f32x4*>(st + (buffer * CB + 16 * c) * PITCH + m * PITCH + row) = own[c];
        }
    };
    publish(0);
    float* const vbuf = st + 2 * CB * PITCH;   // [2][D], where the first column block carries the vector
    if (CT > 1 && vector && !chain && q == 0) vbuf[row0 + m] = sum;

    // The matrix to request in this step (and, while a tile of the step before is still to come, the one before it).
    constexpr int FAR = RING > 0 ? RING + (RA + NT - 1 - TPS) / NT : AHEAD;
    auto matrix = [&](int r) __attribute__((always_inline)) { return a_base + (size_t)(r > r_lo ? r : r_lo) * stride; };
    const Tin* next = matrix(r_top - FAR);
    const Tin* before = matrix(r_top - FAR + 1);
    // The ring in LDS: the slot that is read next, and the one that is requested next, which has been read.
    unsigned slot = ring0, slot_read = ring0;
    auto past = [&](unsigned at_slot) __attribute__((always_inline)) { return at_slot + SLOT == ring0 + RING_BYTES ? ring0 : at_slot + SLOT; };
    unsigned piece[2], first_piece[2];   // this lane's elements of an even and an odd tile in a slot
#pragma unroll
    for (int t = 0; t < 2; ++t)
        piece[t] = TPS == 1 ? (unsigned)(m * 64 + ((q ^ (m >> 2)) << 4)) : (unsigned)(m * 64 + (((2 * t + (q >> 1)) ^ (m >> 2)) << 4) + 8 * (q & 1));
    first_piece[0] = wave & 1 ? piece[1] : piece[0];
    first_piece[1] = wave & 1 ? piece[0] : piece[1];
    auto read_tile = [&](int j) __attribute__((always_inline)) {
        const unsigned at_piece = TPS == 1 ? piece[0] : j < 2 ? first_piece[j & 1] : piece[j & 1];
        const auto v = *reinterpret_cast<const typename Row4<Tin>::type*>(smem + slot_read + at_piece);
        if (TPS == 1 || j % 2 == 1) slot_read = past(slot_read);
        return v;
    };
    // Tile i of the chain (k tile i % NT of step i / NT) moves on: the tile read before it is in its registers, so its slot takes
    // the tile RING NT further down, and tile i is read, once its slot is there (`younger` operations are).
    auto advance = [&](auto i_tag, const Tin* mat, auto younger) __attribute__((always_inline)) {
        constexpr int i = decltype(i_tag)::value, last = (i + FRAGS - 1) % FRAGS;
        if constexpr (i % TPS == 0 && i > 0) {
            asm volatile("" : "+v"(ring[last][0]));
            if constexpr (TPS == 2) asm volatile("" : "+v"(ring[(last + FRAGS - 1) % FRAGS][0]));
            request(mat, (i + NT - TPS) % NT, slot);
            slot = past(slot);
        }
        if constexpr (i % TPS == 0) scan_planes::wait_vm<decltype(younger)::value>();
        ring[i % FRAGS][0] = read_tile(i % NT);
    };
    if constexpr (RING > 0) {
        for_each<0, RA>([&](auto i) __attribute__((always_inline)) {
            constexpr int ahead_of = RING + (decltype(i)::value + NT - TPS) / NT - 1;   // steps down of the tile that is requested
            advance(i, matrix(r_top - ahead_of), std::integral_constant<int, RING * SPS - 1>{});
        });
        // as many as the stores of the steps that the first waits count
        const __amdgpu_buffer_rsrc_t nothing = scan_planes::rows(out, 0);
#pragma unroll
        for (int x = 0; x < 4 * CT * RING; ++x) __builtin_amdgcn_raw_buffer_store_b32(0u, nothing, 0, 0, 0);
    }
    // One step on the first TILES column tiles, the u-th of a trip; CARRY: with the vector, whose rows are dot products of the same
    // elements beside the matrix products.
    auto step = [&](auto u_tag, int r, auto tiles, auto carry_tag) __attribute__((always_inline)) {
        constexpr int TILES = decltype(tiles)::value, U = decltype(u_tag)::value, buffer = U & 1;
        constexpr bool CARRY = decltype(carry_tag)::value;
        f32x4 first = {0.0f, 0.0f, 0.0f, 0.0f};
        float total = 0.0f, near_total = 0.0f;
        auto dot = [&](f32x4 a, int j) __attribute__((always_inline)) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(vbuf + buffer * D + 16 * tile_of(j) + 4 * q);
            float one = a[0] * v[0];
#pragma unroll
            for (int x = 1; x < 4; ++x) one = fmaf(a[x], v[x], one);
            (j == 0 ? near_total : total) += one;
        };
        f32x4 near[TILES][4], part[TILES][NT / 2 + 1];
        f32x4 other[TILES][NT];
        auto products = [&](auto j_tag) __attribute__((always_inline)) {
            constexpr int j = decltype(j_tag)::value;
            auto& stored = RING > 0 ? ring[(U * NT + j) % FRAGS][0] : ring[RING > 0 ? 0 : U % AHEAD][RING > 0 ? 0 : j];
            asm volatile("" : "+v"(stored));   // not before here
            f32x4 a = Row4<Tin>::widen(stored);
            if constexpr (RAGGED) {   // what a row's last tile holds past its end
                const int there = d - 16 * tile_of(j) - 4 * q;
#pragma unroll
                for (int x = 0; x < 4; ++x) a[x] = x < there ? a[x] : 0.0f;
            }
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int c = 0; c < TILES; ++c) {
                    if constexpr (j == 0) near[c][x] = mma(a[x], own[c][x], zero);
                    else part[c][(j - 1) / 2] = mma(a[x], other[c][j][x], j % 2 == 1 && x == 0 ? zero : part[c][(j - 1) / 2]);
                }
            if constexpr (j == 1 || NT == 1) {   // (under the products just issued)
#pragma unroll
                for (int c = 0; c < TILES; ++c) {
                    near[c][0] = (near[c][0] + near[c][1]) + (near[c][2] + near[c][3]);
                    if constexpr (NT > 1) asm volatile("" : "+v"(near[c][0]));
                }
            }
            if constexpr (CARRY) {
                if constexpr (j == 0) first = a;   // (its vector is there behind the barrier)
                else dot(a, j);
            }
            if constexpr (RING == 0) {
                if constexpr (j > 0) stored = load_tile(next, j);
            } else {
                // requested with it so far, besides the tiles: the stores of the steps since
                constexpr int n = U * NT + j, steps = RING - (j + TPS >= NT ? 1 : 0);
                advance(std::integral_constant<int, n + RA>{}, RING + (j + RA - TPS) / NT < FAR ? before : next,
                        std::integral_constant<int, RING * SPS - 1 + 4 * TILES * steps>{});
            }
        };
        products(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);   // under the wait for the other waves
        if constexpr (NT > 1) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int j = 1; j < NT; ++j)
#pragma unroll
                for (int c = 0; c < TILES; ++c)
                    other[c][j] = *reinterpret_cast<const f32x4*>(st + (buffer * CB + 16 * c) * PITCH + b_at[j]);
        }
        if constexpr (CARRY) dot(first, 0);
        if constexpr (RING == 0) ring[U % AHEAD][0] = load_tile(next, 0);
        for_each<1, NT>(products);
#pragma unroll
        for (int c = 0; c < TILES; ++c) {
            f32x4 sum = near[c][0];
            if constexpr (NT > 1) {
                f32x4 rest = part[c][0];
#pragma unroll
                for (int p = 1; p < NT / 2; ++p) rest += part[c][p];
                sum += rest;
            }
            if (RAGGED) {
#pragma unroll
                for (int x = 0; x < 4; ++x) sum[x] = row + x < d ? sum[x] : 0.0f;
            }
            own[c] = sum;
        }
        publish(buffer ^ 1);
        if constexpr (CARRY) {
            total += __shfl_xor(total, 16, 64);
            near_total += __shfl_xor(near_total, 16, 64);
            total += __shfl_xor(total, 32, 64);
            near_total += __shfl_xor(near_total, 32, 64);
            total += near_total;
            if (RAGGED && row0 + m >= d) total = 0.0f;
            if (q == 0) {
                vbuf[(buffer ^ 1) * D + row0 + m] = total;
                if (!RAGGED || row0 + m < d) cot_b[(size_t)r * d + row0 + m] = total;
            }
        }
        // a chunk that only forms its total parks it one slot above its first matrix
        const __amdgpu_buffer_rsrc_t o_r =
            scan_planes::rows(o_base + (size_t)(store_all ? r : r + 1) * o_stride, store_all || r == r_lo ? result_bytes : 0);
#pragma unroll
        for (int c = 0; c < TILES; ++c)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const float v = own[c][x];
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), o_r, at[c] + x * row_bytes, 0, 0);
            }
        before = next;
        next -= r - FAR > r_lo ? stride : 0;
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run = [&](auto tiles, auto carry_tag) __attribute__((always_inline)) {
        // the register ring, the four tiles read ahead and the two buffers of the block: all at compile-time places
        constexpr int TRIP = RING > 0 ? 4 : AHEAD % 2 == 0 ? AHEAD : 2 * AHEAD;
        int r = r_top;
        if constexpr (RING > 0) {
            for (bool more = true; more; r -= TRIP)
                for_each<0, TRIP>([&](auto u) __attribute__((always_inline)) {
                    if (!more) return;
                    step(u, r - decltype(u)::value, tiles, carry_tag);
                    more = r - decltype(u)::value > r_lo;
                });
        } else {
            // (whole trips without a way out between their steps: at one, the compiler would wait for all that it has requested)
            for (; r - r_lo >= TRIP - 1; r -= TRIP)
                for_each<0, TRIP>([&](auto u) __attribute__((always_inline)) { step(u, r - decltype(u)::value, tiles, carry_tag); });
            for_each<0, TRIP - 1>([&](auto u) __attribute__((always_inline)) {
                if (r - decltype(u)::value >= r_lo) step(u, r - decltype(u)::value, tiles, carry_tag);
            });
        }
        if constexpr (RING > 0) scan_planes::wait_vm<0>();   // no transfer into LDS outlives the workgroup
    };
    if constexpr (CT > 1) {
        if (chain) run(std::integral_constant<int, 1>{}, std::false_type{});
        else if (vector) run(std::integral_constant<int, CT>{}, std::true_type{});
        else run(std::integral_constant<int, CT>{}, std::false_type{});
    } else {
        run(std::integral_constant<int, CT>{}, std::false_type{});
    }
}

// Steps ahead of the ring in LDS: what leaves room for two workgroups per CU up to 80 columns, what fits beyond.
constexpr int ring_steps(int NT, int CT, int size) {
    return NT < 4 ? 0 : NT == 4 ? 4 : NT == 5 ? 3 : size == 2 ? (NT < 8 ? 4 : 3) : NT == 6 ? 3 : NT == 7 || CT == 1 ? 2 : 1;
}

template <typename Tin, int NT, int CT, bool RAGGED, int RING>
int launch_one(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, bool carry, ScanPlan plan, hipStream_t stream) {
    constexpr int NB = (NT + CT - 1) / CT;
    constexpr size_t bytes = (NT > 1 ? (size_t)2 * 16 * CT * (16 * NT + 4) * 4 : 0) + (CT > 1 ? 2 * 16 * NT * 4 : 0) + (size_t)RING * NT * NT * 256 * sizeof(Tin);
    static_assert(bytes <= 160 * 1024, "LDS budget");
    if (int rc = ensure_dynamic_lds<&scan_narrow_kernel<Tin, NT, CT, RAGGED, RING>>(bytes)) return rc;
    const int64_t chains = (int64_t)B * (plan.phase == 1 || plan.phase == 3 ? plan.C - 1 : 1);
    const int64_t blocks = (chains >= 8 ? (chains + 7) / 8 * 8 : chains) * (out ? NB + (cot && !(CT > 1 && carry) ? 1 : 0) : 1);
    hipLaunchKernelGGL((scan_narrow_kernel<Tin, NT, CT, RAGGED, RING>), dim3((unsigned)blocks), dim3(64 * NT), bytes, stream,
                       static_cast<const Tin*>(mats), static_cast<float*>(out), static_cast<const float*>(g),
                       static_cast<float*>(cot), B, K, d, (int)carry, plan);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

// One launch (a whole chain, or a phase of the plan) on blocks of 16 `tiles` columns.
template <typename Tin, int NT>
int launch_width(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, int tiles, bool carry,
                 ScanPlan plan, hipStream_t stream) {
    auto run = [&](auto ct) {
        constexpr int CT = decltype(ct)::value, RING = ring_steps(NT, CT, sizeof(Tin));
        // transfers into LDS move whole 4-byte words: 16-bit rows of an odd width or start come straight into registers
        if constexpr (sizeof(Tin) == 2)
            if (d % 2 != 0 || reinterpret_cast<uintptr_t>(mats) % 4 != 0)
                return launch_one<Tin, NT, CT, true, 0>(mats, out, g, cot, B, K, d, carry, plan, stream);
        if (d == 16 * NT) return launch_one<Tin, NT, CT, false, RING>(mats, out, g, cot, B, K, d, carry, plan, stream);
        return launch_one<Tin, NT, CT, true, RING>(mats, out, g, cot, B, K, d, carry, plan, stream);
    };
    if constexpr (NT > 1)
        if (tiles == 2) return run(std::integral_constant<int, 2>{});
    return run(std::integral_constant<int, 1>{});
}

template <typename Tin>
int launch_type(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, int tiles, bool carry,
                const ScanPlan& plan, hipStream_t stream) {
    const int nt = row_tiles(d, sizeof(Tin) == 4 ? LBI_F32 : LBI_F16);
    switch (nt) {
        case 1: return launch_width<Tin, 1>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case 2: return launch_width<Tin, 2>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case 3: return launch_width<Tin, 3>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case 4: return launch_width<Tin, 4>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case 6: return launch_width<Tin, 6>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case 8: return launch_width<Tin, 8>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        default: break;
    }
    if constexpr (sizeof(Tin) == 4) {
        if (nt == 5) return launch_width<Tin, 5>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        return launch_width<Tin, 7>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
    }
    return LBI_ERR_UNSUPPORTED;
}

}  // namespace scan_narrow
}  // namespace lbi
