// Suffix scan on the 16-bit matrix cores with fp32 products (widths 129 ... 256; every storage type, but for bf16 at 256
// where the batch fills the chip).
//
// The bf16 rate of gfx950's matrix cores is sixteen times their fp32 rate.  An fp32 number is the sum of three bf16
// numbers, hi + mid + lo, exactly, so a product of two of them is nine bf16 products, of which the six above 2^-24 of the
// whole are formed: 6 against 16.  (fp16 elements have two planes: 5 of 6 products, mid x lo left out, which lies below 2^-27 of
// the whole as what fp32 ones leave out does; bf16 elements one: all 3.)
//
// Accuracy.  v_mfma_f32_32x32x16_bf16 adds the products of eight k to each other first, cut off at the last place of the largest
// among them, and the two sums to the accumulator with one rounding each.  What would suffer is a row with one
// large element among small ones, and the matrices that this scan multiplies are of that kind: the identity and a small
// update.  The diagonal is therefore taken out of the rows and multiplied in fp32, by one fused multiply-add onto the sum of all
// the rest; the hi x hi products and the smaller ones are summed apart.  Relative error against fp64 (2-norm over K = 128 products
// at d = 256, B = 64; products of fp32 MFMAs with blocked sums -> here): identity plus update 9.6e-7 -> 2.3e-7, random
// orthogonal-like 9.2e-7 -> 7.3e-7; the cotangents 1.7e-6 -> 3.9e-7 and 1.7e-6.
// Range.  bf16 ends where fp32 does, so the lower planes of a number near 2^-126 would fall below it.  The planes are those of the
// number times 2^23: every bit of an fp32 number, down to the last of its subnormals, is then a normal number of bf16, and what
// underflows in a product lies below 2^-172, out of sight of fp32 results.  (fp16 elements need no factor, bf16 ones are their
// own plane, which the products take subnormal too.)  Products end at 2^81 instead, those of 16-bit elements at 2^104.  A wave whose tile holds such a
// number, an infinity or NaN forms it again with fp32 products, and the block enters the next step in fp32: the workgroup
// goes on like that until every tile is back in range.  The error of an element is that of fp32 arithmetic,
// against the sizes of its own terms.  (B=64 K=128 d=256, a chain above 2^81 all the way 3.4 ms, fp32 MFMAs 2.3; one below 2^-100 1.8, random
// matrices that shrink by 0.4 a step 1.8, that grow by 1.7 to 2^98 2.1, fp32 MFMAs 2.2-2.3 each.)
//
// A workgroup owns CB columns of one batch element and keeps that block of the running suffix S in LDS as three planes,
// transposed; a wave owns 32 rows.  What a step costs was found by timing it without one thing after the other (d = 256, CB =
// 64, us of 13.8): the products alone 6, the splitting 1.6, bringing the rows in 2.6, the results' stores 1.7, handing the block on
// 2.5; the part runs it at 1.9 GHz, where the products alone reach 2.3.  Hence:
//  * Rows come by 16-byte transfers into a ring in LDS, four lanes to 64 bytes of a row.  Loaded straight into the registers
//    that the products want them in, each lane another row, they come at 36 GB/s per CU however many are in flight; like
//    this at 61, contiguous at 72.
//  * What is left of a number after a plane is one v_dot2_f32_bf16: 7 instead of 11 instructions for a pair.  (The factor of
//    2^23 is two more: B=64 K=128 d=256 1.77 -> 1.81 ms, B=1 122 -> 126 us; 16-bit elements 0-1 %.)
//  * The vector work of a product step (the next step's split, the stores of the product before) is written between its
//    products, one or two instructions' groups to each.
//  * A step begins with the k of the wave's own rows, so that the barrier behind the handing on sits 12 products later, and
//    ends column tile by column tile, so that one is added up and split under the products of the other.
//  * The two waves of a SIMD do not wait for each other's age: whoever is behind in the step has the higher priority.
// Measured (K = 128, start of this form in brackets: fp32 MFMAs): d = 256 B = 64 fp32 with cotangents 1.8-1.9 ms (2.25-2.4),
// B = 1 126 us (146); d = 192 B = 64 1.1 ms (1.6); d = 200 B = 64, read as it lies instead of padded to 256: 0.45-0.65 of the time.
#pragma once

#include "lbi_common.h"

namespace lbi {

// Which part of the chain a workgroup runs.  `phase` 0 is the whole chain of a batch element (K - 1 dependent
// steps).  Phases 1-3 are the K-parallel form for batches too small to fill the chip with one chain per column
// block: the chain is cut into C chunks; chunk c >= 1 starts at matrix b_c = cL - s and has L matrices (the last
// one what is left), chunk 0 has the first L - s (s = 1: every chunk then has L - 1 steps in phase 3, where chunk 0,
// which has no boundary product of its own to skip, would otherwise run one step longer than the rest), and
//   phase 1  every chunk c >= 1 multiplies its own matrices (L - 1 steps, all chunks side by side): the last chunk's
//            products are final results and are stored as in phase 0; a middle chunk keeps only its total
//            T_c = mats[b_c] ... mats[b_c + L - 1], parked in out[b_c + 1], a slot phase 3 rewrites;
//   phase 2  one chain over the totals (C - 2 steps): out[b_c] = T_c @ out[b_c + L] for c = C-2 ... 1, which are the
//            final suffix products at the chunk boundaries (the kernel runs it with mats = the parked totals);
//   phase 3  every chunk c <= C-2 restarts the chain from out[b_{c+1}] through its own matrices (L - 1 steps, all
//            chunks side by side), storing each product.
// The cotangents, if asked for, are then the finished products applied to g (suffix_apply_kernel) above 128 columns; up to 128 the vector rides on the
// last chunk of phase 1 and on phase 3 (scan_narrow).
// About twice the products, a dependent depth of 2L + C - 4 instead of K - 1, no scratch memory, no atomics; the
// summation order is fixed by (K, L), so reruns are bit-identical.
struct ScanPlan {
    int phase;  // 0: whole chain; 1, 2, 3: see above
    int L;      // matrices per chunk (>= 2)
    int C;      // chunks (>= 3)
    // One level of the log-depth form of phase 2 (MODE 3): element c = 1 .. C-2 lives in slot out[b_c + rd], the
    // last element is out[b_{C-1}]; the level writes elem[c] @ elem[c + off] (or elem[c] itself where c + off is
    // past the last element) to out[b_c + wr].
    int off, rd, wr;
    int s;      // chunk boundaries b_c = cL - s (0 or 1)
};

namespace scan_planes {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));  // v_cvt_pk_bf16_f32, RNE
}
__device__ __forceinline__ float bf16_lo(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(unsigned w) { return __uint_as_float(w & 0xffff0000u); }

// Splits pairs of fp32 numbers into packed bf16 planes, hi + mid + lo == x exactly for multiples of 2^-126 below 2^127.  What is left of a
// number after a plane is one v_dot2_f32_bf16 with (-1, 0) or (0, -1), which are kept in registers: as literals the
// compiler would encode them as inline constants, whose value this instruction takes in another format.
struct Splitter {
    unsigned first, second;
    __device__ __forceinline__ Splitter() {
        asm volatile("s_mov_b32 %0, 0x0000bf80" : "=s"(first));
        asm volatile("s_mov_b32 %0, 0xbf800000" : "=s"(second));
    }
    __device__ __forceinline__ void rest(unsigned plane, float& x0, float& x1) const {
        x0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, plane), __builtin_bit_cast(bf16x2, first), x0, false);
        x1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, plane), __builtin_bit_cast(bf16x2, second), x1, false);
    }
    template <int N>
    __device__ __forceinline__ void split(float x0, float x1, unsigned (&w)[N]) const {
#pragma unroll
        for (int p = 0; p < N; ++p) {
            w[p] = pack_bf16(x0, x1);
            if (p + 1 < N) rest(w[p], x0, x1);
        }
    }
};

// Planes of a stored element, what they are of it, and 16-byte words of the 8 elements a lane brings to a product step.
constexpr float kScale = 0x1p23f;         // of the suffix block's planes
template <typename Tin> struct Storage;
template <> struct Storage<float> { static constexpr int NA = 3, WORDS = 2; static constexpr float SCALE = kScale; };
template <> struct Storage<_Float16> { static constexpr int NA = 2, WORDS = 1; static constexpr float SCALE = 1.0f; };
template <> struct Storage<bf16_raw> { static constexpr int NA = 1, WORDS = 1; static constexpr float SCALE = 1.0f; };

// Four consecutive elements, aligned as single ones are.
__device__ __forceinline__ f32x4 load4_at(const float* p) {
    typedef float f32x4_at __attribute__((ext_vector_type(4), aligned(4)));
    return *reinterpret_cast<const f32x4_at*>(p);
}
template <typename Tin> __device__ __forceinline__ f32x4 load4_at(const Tin* p) {
    typedef unsigned short u16x4_at __attribute__((ext_vector_type(4), aligned(2)));
    const u16x4_at w = *reinterpret_cast<const u16x4_at*>(p);
    f32x4 v;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const unsigned short one = w[x];
        v[x] = to_f32(__builtin_bit_cast(Tin, one));
    }
    return v;
}

__device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows(const void* p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// At most N vector memory operations of the wave are still under way.
template <int N> __device__ __forceinline__ void wait_vm() {
    constexpr int n = N < 63 ? N : 63;
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

// As many as BASE + n PER, n <= MOST known once the loops are unrolled.
template <int BASE, int PER, int MOST> __device__ __forceinline__ void wait_younger(int n) {
    if constexpr (MOST == 0) wait_vm<BASE>();
    else if (n == MOST) wait_vm<BASE + MOST * PER>();
    else wait_younger<BASE, PER, MOST - 1>(n);
}

__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t src, unsigned lane_offset, unsigned offset, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(lane_offset), "s"(src), "s"(offset)
                 : "memory");
}

// LDS of a workgroup: three planes of the suffix block, the waves' rings of rows (slots of 32 rows x 64 bytes), two copies of
// the diagonal and (with the chain) of the vector, two flags.
constexpr int kSlotBytes = 2048;
// Slots of a wave's ring.  Three where the planes leave no room for more (64 columns of 256) or where two workgroups share a
// CU; six in the short steps of 32 columns of 256, which one workgroup per CU takes, and in the launches of a single step.
constexpr int ring_slots(int D, int CB, int MODE) { return CB == 32 && (D == 256 || MODE == 3) ? 6 : 3; }
constexpr size_t lds_bytes(int D, int CB, bool chain, int MODE) {
    return (size_t)3 * CB * (D + 8) * 2 + (size_t)(D / 32) * ring_slots(D, CB, MODE) * kSlotBytes + (size_t)(chain ? 4 : 2) * D * 4 + 16;
}

template <typename Tin, int D, int RT, int CB, bool COT, int MODE>
__global__ __launch_bounds__(64 * (D / RT)) void scan_planes_kernel(
    const Tin* __restrict__ mats, float* __restrict__ out, const float* __restrict__ g,
    float* __restrict__ cot, int B, int K, int d, ScanPlan plan) {
    constexpr int NW = D / RT, RTILES = RT / 32, CTILES = CB / 32, NB = D / CB;
    constexpr int NA = Storage<Tin>::NA, WORDS = Storage<Tin>::WORDS, NP = 3;
    constexpr float SCALE = Storage<Tin>::SCALE, PRODUCT_SCALE = SCALE * kScale;
    constexpr int PITCH = D + 8;                    // bf16 elements of a column of a plane
    constexpr int PLANE = CB * PITCH;
    constexpr int WPITCH = D + 4;                   // floats of a column of the block kept in fp32
    constexpr int HALVES = D / 16;                  // product steps (16 k) of a suffix step
    constexpr int kSlots = ring_slots(D, CB, MODE);
    constexpr int HPS = WORDS == 2 ? 1 : 2;         // product steps a ring slot holds: 64 bytes of 32 rows
    const size_t dd = (size_t)d * d;

    extern __shared__ __align__(16) char smem[];    // [NP][CB][PITCH] bf16 (or [CB][WPITCH] fp32), [2][D] diagonal, (COT) [2][D], [2] flags
    unsigned short* planes = reinterpret_cast<unsigned short*>(smem);
    float* wide_s = reinterpret_cast<float*>(smem);
    constexpr unsigned RING_AT = (unsigned)NP * PLANE * 2;
    float* diag = reinterpret_cast<float*>(smem + RING_AT + (size_t)NW * RTILES * kSlots * kSlotBytes);
    float* vbuf = diag + 2 * D;
    volatile int* flags = reinterpret_cast<int*>(diag + 2 * D + (COT ? 2 * D : 0));

    // A launch covers E = B * (segments per batch element) chains.  With at least 8 of them the workgroups are
    // dealt round-robin to the 8 XCDs so that all column blocks of one chain get ids that are equal mod 8 and
    // share one L2; smaller launches are sized exactly.
    const int nseg = MODE == 1 ? plan.C - 1 : MODE == 3 ? plan.C - 2 : 1;
    const int E = B * nseg;
    const int id = blockIdx.x;
    int e, c0;
    if (E >= 8) {
        const int slot = id >> 3;
        e = (slot / NB) * 8 + (id & 7);
        c0 = (slot % NB) * CB;
    } else {
        e = id / NB;
        c0 = (id % NB) * CB;
    }
    if (e >= E || c0 >= d) return;
    const int b = e / nseg;
    const int seg = e - b * nseg;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, m = lane & 31, h = lane >> 5;
    const int row0 = wave * RT;

    float* out_b = out + (size_t)b * (K + 1) * dd;
    // The chain of this workgroup: steps r = r_top ... r_lo multiply a_base[r * a_stride] onto the running suffix
    // and store it at o_base[r * o_stride]; the suffix starts as the matrix `init_a` (storage type) or `init_s`
    // (fp32, a product computed earlier).
    const Tin* a_base = mats + (size_t)b * K * dd;
    float* o_base = out_b;
    const Tin* init_a = nullptr;
    const float* init_s = nullptr;
    int r_top, r_lo = 0;
    bool write_tail = false;   // the start matrix and the identity behind it are results (out[K - 1], out[K])
    bool store_all = true;     // every step's product is a result
    // the cotangent chain rides on the whole-chain form only; the chunk phases share no chain to carry it
    static_assert(MODE == 0 || !COT, "chunk phases carry no cotangent chain");
    size_t stride_rt = dd;
    if constexpr (MODE == 0) {
        init_a = a_base + (size_t)(K - 1) * dd;
        r_top = K - 2;
        write_tail = true;
    } else if constexpr (MODE == 1) {
        if (plan.phase == 1) {
            const int c = seg + 1;
            const bool last = c == plan.C - 1;
            const int end = last ? K : (c + 1) * plan.L - plan.s;
            init_a = a_base + (size_t)(end - 1) * dd;
            r_top = end - 2;
            r_lo = c * plan.L - plan.s;
            write_tail = last;
            store_all = last;
        } else {
            const int c = seg;
            init_s = out_b + (size_t)((c + 1) * plan.L - plan.s) * dd;
            r_top = (c + 1) * plan.L - plan.s - 1;
            r_lo = c == 0 ? 0 : c * plan.L - plan.s + 1;   // the chunk's first product is a phase 2 result already
        }
    } else if constexpr (MODE == 3) {
        const int c = seg + 1;
        const float* left = out_b + (size_t)(c * plan.L - plan.s + plan.rd) * dd;
        float* dst = out_b + (size_t)(c * plan.L - plan.s + plan.wr) * dd;
        const int partner = c + plan.off;
        if (partner > plan.C - 1) {
            // nothing to the right at this distance: the element is complete, it moves to the level's output slot
            const int cols = d - c0 < CB ? d - c0 : CB;
            for (int idx = tid; idx < d * CB; idx += 64 * NW) {
                const int row = idx / CB, q = idx % CB;
                if (q < cols) dst[(size_t)row * d + c0 + q] = left[(size_t)row * d + c0 + q];
            }
            return;
        }
        a_base = reinterpret_cast<const Tin*>(left);
        o_base = dst;
        init_s = partner == plan.C - 1 ? out_b + (size_t)((plan.C - 1) * plan.L - plan.s) * dd
                                       : out_b + (size_t)(partner * plan.L - plan.s + plan.rd) * dd;
        r_top = 0;
    } else {
        // step j multiplies the total parked one slot above the first matrix of chunk j + 1 and stores that first slot
        a_base = reinterpret_cast<const Tin*>(out_b + (size_t)(plan.L - plan.s + 1) * dd);
        o_base = out_b + (size_t)(plan.L - plan.s) * dd;
        stride_rt = (size_t)plan.L * dd;
        init_s = out_b + (size_t)((plan.C - 1) * plan.L - plan.s) * dd;
        r_top = plan.C - 3;
    }
    const bool from_a = MODE == 0 || (MODE == 1 && plan.phase == 1);   // start state: init_a, else init_s
    // distance between the matrices (and the results) of consecutive steps
    const size_t a_stride = MODE == 2 ? stride_rt : dd;
    const size_t o_stride = a_stride;

    const Splitter splitter;
    auto lds_barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // This wave's RT x CB tile: the newest finished product, and of the next one the sum of the hi x hi products and that
    // of all others (the diagonal's apart).  The product is kept as it comes out, times PRODUCT_SCALE, unless it is past that
    // range: `down` takes it to what it is.
    f32x16 tot[RTILES][CTILES], top[RTILES][CTILES], fine[RTILES][CTILES];
    float down = 1.0f;
    auto row_of = [&](int i, int e) __attribute__((always_inline)) { return row0 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3); };

    // Results and start states by element: a descriptor over the matrix, past whose end nothing is read or written, an offset
    // per lane and column tile (past everything where the column is not there) and one per row.  (Both in the lane's offset:
    // a scalar offset larger than the descriptor would leave the range check to an underflow.)
    constexpr unsigned kNowhere = 0x80000000u;
    unsigned lane_col[CTILES];
#pragma unroll
    for (int j = 0; j < CTILES; ++j) {
        const int c = c0 + 32 * j + m;
        lane_col[j] = c < d ? (unsigned)(4 * h * d + c) * 4 : kNowhere;
    }
    int row_elements = d;
    auto row_bytes = [&](int i, int q, int e) __attribute__((always_inline)) { return (unsigned)((row0 + 32 * i + 8 * q + e) * row_elements) * 4; };
    const unsigned matrix_bytes = (unsigned)dd * 4;
    // element n of the tile, n = 0 ... 16 RTILES CTILES - 1, of the finished product
    auto store_element = [&](__amdgpu_buffer_rsrc_t o_r, int n) __attribute__((always_inline)) {
        const int i = n / (16 * CTILES), j = n / 16 % CTILES, q = n % 16 / 4, e = n % 4;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(tot[i][j][4 * q + e] * down), o_r, lane_col[j] + row_bytes(i, q, e), 0, 0);
    };
    constexpr int NEL = 16 * RTILES * CTILES;

    // One step (or, from the planes, its repetition) on the fp32 matrix cores: any values, one product at a time.
    // The planes keep the 16 k of a product step in the order of the lane halves that bring them: rows 4 h + [0, 4) and
    // 8 + 4 h + [0, 4), which is how the accumulators hold a column, so that a lane writes and reads 16 bytes at a time.
    auto place = [](int k) { return (k & ~15) | ((k >> 2) & 1) << 3 | ((k >> 3) & 1) << 2 | (k & 3); };
    auto wide_tile = [&](const Tin* a_r, bool from_planes, bool chain, float (&vdot)[RTILES], const float* v_old) __attribute__((always_inline)) {
        down = 1.0f;
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int j = 0; j < CTILES; ++j)
#pragma unroll
                for (int x = 0; x < 16; ++x) tot[i][j][x] = 0.0f;
        // lane half h brings k = 8 k8 + 4 h + [0, 4) of its row to four products (what lies behind a row's end is of the next row
        // or matrix: the last matrix is no left operand)
#pragma unroll 1
        for (int k8 = 0; k8 < D / 8; ++k8) {
            const int k = 8 * k8 + 4 * h;
            f32x4 a[RTILES];
#pragma unroll
            for (int i = 0; i < RTILES; ++i) {
                const int row = row0 + 32 * i + m;
                a[i] = load4_at(a_r + (size_t)(row < d ? row : 0) * d + (k < d ? k : 0));
#pragma unroll
                for (int x = 0; x < 4; ++x) a[i][x] = row < d && k + x < d ? a[i][x] : 0.0f;
            }
            if (chain) {
                const f32x4 v4 = *reinterpret_cast<const f32x4*>(v_old + k);
#pragma unroll
                for (int i = 0; i < RTILES; ++i)
#pragma unroll
                    for (int x = 0; x < 4; ++x) vdot[i] = fmaf(a[i][x], v4[x], vdot[i]);
            }
#pragma unroll
            for (int j = 0; j < CTILES; ++j) {
                f32x4 s;
                if (from_planes) {
                    const int at = (32 * j + m) * PITCH + place(k);
                    s = (load4(reinterpret_cast<const bf16_raw*>(planes) + at) + load4(reinterpret_cast<const bf16_raw*>(planes) + PLANE + at)) +
                        load4(reinterpret_cast<const bf16_raw*>(planes) + 2 * PLANE + at);
                    s *= 1.0f / kScale;
                } else {
                    s = *reinterpret_cast<const f32x4*>(wide_s + (32 * j + m) * WPITCH + k);
                }
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int i = 0; i < RTILES; ++i) tot[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][x], s[x], tot[i][j], 0, 0, 0);
            }
        }
    };
    // Whether the tile, kept as it is or scaled, holds what planes and products do not.
    auto out_of_range = [&](float limit) __attribute__((always_inline)) {
        float high = 0.0f;
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int j = 0; j < CTILES; ++j)
#pragma unroll
                for (int x = 0; x < 16; x += 2)
                    high = __builtin_elementwise_maximum(high, __builtin_elementwise_maximum(__builtin_fabsf(tot[i][j][x]), __builtin_fabsf(tot[i][j][x + 1])));
        return __builtin_amdgcn_ballot_w64(!(high < limit)) != 0;
    };
    // A tile that is kept as it is goes on in scale, if it can.
    auto scale_up = [&]() __attribute__((always_inline)) {
        const bool bad = out_of_range(0x1p127f / PRODUCT_SCALE);
        if (!bad) {
#pragma unroll
            for (int i = 0; i < RTILES; ++i)
#pragma unroll
                for (int j = 0; j < CTILES; ++j)
#pragma unroll
                    for (int x = 0; x < 16; ++x) tot[i][j][x] *= PRODUCT_SCALE;
            down = 1.0f / PRODUCT_SCALE;
        }
        return bad;
    };

    int parity = 0;
    unsigned words[RTILES][CTILES][4][NP][2];   // the finished tile as planes
    auto split_tile = [&](int i, int j, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            unsigned w[NP];
            splitter.split<NP>(tot[i][j][4 * q + 2 * u] * (1.0f / SCALE), tot[i][j][4 * q + 2 * u + 1] * (1.0f / SCALE), w);
#pragma unroll
            for (int p = 0; p < NP; ++p) words[i][j][q][p][u] = w[p];
        }
    };
    // Hands the tile to the next step, once nobody reads the block before any more.
    auto publish = [&](bool bad) __attribute__((always_inline)) {
        parity ^= 1;
        if (bad && lane == 0) flags[parity] = 1;
        lds_barrier();
        if (tid == 0) flags[parity ^ 1] = 0;
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int j = 0; j < CTILES; ++j)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        *reinterpret_cast<u32x4*>(planes + p * PLANE + (32 * j + m) * PITCH + row0 + 32 * i + 16 * x + 8 * h) =
                            u32x4{words[i][j][2 * x][p][0], words[i][j][2 * x][p][1], words[i][j][2 * x + 1][p][0], words[i][j][2 * x + 1][p][1]};
    };
    // Whether the block must be taken in fp32 (valid behind a barrier that follows publish).
    auto asked_wide = [&]() __attribute__((always_inline)) { return flags[parity]; };
    auto write_wide = [&]() __attribute__((always_inline)) {
        lds_barrier();
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int j = 0; j < CTILES; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4*>(wide_s + (32 * j + m) * WPITCH + row_of(i, 4 * q)) =
                        f32x4{tot[i][j][4 * q], tot[i][j][4 * q + 1], tot[i][j][4 * q + 2], tot[i][j][4 * q + 3]} * down;
        lds_barrier();
    };
    auto split_all = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int j = 0; j < CTILES; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) split_tile(i, j, q);
    };

    // Rows of mats[r] come through LDS: a wave's ring of slots (32 rows x 64 bytes per row tile; 16-byte piece p of row i at
    // p ^ (i / 4) % 4, so that the 16 lanes of a read meet all banks).  Product step s of the wave's order takes k =
    // first_k(s) + 4 h + {0 ... 3, 8 ... 11}; the order begins with the k of its own rows.
    auto first_k = [&](int s) __attribute__((always_inline)) {
        const int k = 32 * wave * RTILES + 16 * s;
        return k < D ? k : k - D;
    };
    const unsigned ring0 = RING_AT + (unsigned)wave * RTILES * kSlots * kSlotBytes;
    unsigned dma_lane[RTILES][2];
#pragma unroll
    for (int i = 0; i < RTILES; ++i)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int local = 16 * x + (lane >> 2), row = row0 + 32 * i + local;
            dma_lane[i][x] = row < d ? (unsigned)(row * d) * (unsigned)sizeof(Tin) + (((lane & 3) ^ ((local >> 2) & 3)) << 4) : kNowhere;
        }
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
    unsigned slot_at[kSlots];               // ring order from now on: the slot read next first
#pragma unroll
    for (int x = 0; x < kSlots; ++x) slot_at[x] = ring0 + x * RTILES * kSlotBytes;
    // requests the slot of product steps s ... s + HPS - 1 (past the end: of the steps that follow)
    auto request = [&](unsigned slot, int r, int s) __attribute__((always_inline)) {
        const int rr = r - s / HALVES;
        // The last row's pieces end up to 15 elements past the matrix.  Those of mats are the next matrix there (the last one is no
        // left operand); a parked total's are cut, element by element, at its end: the slot behind it may hold anything.
        const __amdgpu_buffer_rsrc_t src = rows(a_base + (size_t)(rr > r_lo ? rr : r_lo) * a_stride,
                                                (unsigned)(dd * sizeof(Tin)) + (MODE >= 2 ? 0 : 64));
        const unsigned k = (unsigned)first_k(s % HALVES) * (unsigned)sizeof(Tin);
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int x = 0; x < 2; ++x) dma16(src, dma_lane[i][x], k, lds0 + slot + i * kSlotBytes + x * 1024);
    };
    // the first rows travel while the start state is made
    if (r_top >= r_lo) {
#pragma unroll
        for (int x = 0; x < kSlots; ++x) request(slot_at[x], r_top, x * HPS);
    }
    bool requested = true;

    if (tid == 0) flags[0] = flags[1] = 0;
    // Start state
#pragma unroll
    for (int i = 0; i < RTILES; ++i)
#pragma unroll
        for (int j = 0; j < CTILES; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    if (from_a) {
                        constexpr int F = 4 / (int)sizeof(Tin);
                        if constexpr (sizeof(Tin) == 4)
                            tot[i][j][4 * q + x] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                                rows(init_a, matrix_bytes), lane_col[j] + row_bytes(i, q, x), 0, 0));
                        else
                            tot[i][j][4 * q + x] = to_f32(__builtin_bit_cast(Tin, __builtin_amdgcn_raw_buffer_load_b16(
                                rows(init_a, matrix_bytes / F), (lane_col[j] + row_bytes(i, q, x)) / F, 0, 0)));
                    } else {
                        tot[i][j][4 * q + x] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                            rows(init_s, matrix_bytes), lane_col[j] + row_bytes(i, q, x), 0, 0));
                    }
                }
    if (write_tail) {
        const __amdgpu_buffer_rsrc_t o_last = rows(out_b + (size_t)(K - 1) * dd, matrix_bytes);
        const __amdgpu_buffer_rsrc_t o_eye = rows(out_b + (size_t)K * dd, matrix_bytes);
#pragma unroll
        for (int n = 0; n < NEL; ++n) store_element(o_last, n);
#pragma unroll
        for (int n = 0; n < NEL; ++n) {
            const int i = n / (16 * CTILES), j = n / 16 % CTILES, q = n % 16 / 4, x = n % 4;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(row_of(i, 4 * q + x) == c0 + 32 * j + m ? 1.0f : 0.0f), o_eye,
                                                  lane_col[j] + row_bytes(i, q, x), 0, 0);
        }
    }
    if (COT) {
        // first vector of the chain: (start state) @ g, one row per thread, once per kernel
        const float* g_b = g + (size_t)b * d;
        float* cot_b = cot + (size_t)b * (K + 1) * d;
        for (int row = tid; row < D; row += 64 * NW) {
            float sum = 0.0f;
            if (row < d) {
                const Tin* a_row = init_a + (size_t)row * d;
#pragma unroll 8
                for (int k = 0; k < d; ++k) sum = fmaf(to_f32(a_row[k]), g_b[k], sum);
                if (c0 == 0) {
                    cot_b[(size_t)K * d + row] = g_b[row];
                    cot_b[(size_t)(K - 1) * d + row] = sum;
                }
            }
            vbuf[row] = sum;
        }
    }
    if (r_top < r_lo) return;
    lds_barrier();   // the flags are zero
    const bool past = scale_up();
    split_all();
    publish(past);
    bool wide = false;

    u32x4 raw[RTILES][WORDS];               // this lane's elements of the product step that is split next
    u32x4 afr[2][NA][RTILES];               // [parity of the product step][plane][tile]
    u32x4 bfr[NP][CTILES];
    float vdot[RTILES];
    f32x4 vvec[2];                          // the 8 entries of the vector that raw meets
    const unsigned piece0 = (unsigned)(m * 64), piece_swz = (unsigned)((m >> 2) & 3);
    auto read_raw = [&](unsigned slot, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RTILES; ++i)
#pragma unroll
            for (int w = 0; w < WORDS; ++w) {
                if constexpr (WORDS == 2) {
                    raw[i][w] = *reinterpret_cast<const u32x4*>(smem + slot + i * kSlotBytes + piece0 + 16 * ((2 * w + h) ^ piece_swz));
                } else {
                    const u32x2 a = *reinterpret_cast<const u32x2*>(smem + slot + i * kSlotBytes + piece0 + 16 * ((2 * t) ^ piece_swz) + 8 * h);
                    const u32x2 c = *reinterpret_cast<const u32x2*>(smem + slot + i * kSlotBytes + piece0 + 16 * ((2 * t + 1) ^ piece_swz) + 8 * h);
                    raw[i][w] = u32x4{a[0], a[1], c[0], c[1]};
                }
            }
    };
    auto element_pair = [&](int i, int w, float& x0, float& x1) __attribute__((always_inline)) {
        if constexpr (WORDS == 2) {
            x0 = __uint_as_float(raw[i][w >> 1][2 * (w & 1)]);
            x1 = __uint_as_float(raw[i][w >> 1][2 * (w & 1) + 1]);
        } else if constexpr (NA == 2) {
            typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
            const unsigned word = raw[i][0][w];
            const f16x2 v = __builtin_bit_cast(f16x2, word);
            x0 = (float)v[0];
            x1 = (float)v[1];
        } else {
            x0 = bf16_lo(raw[i][0][w]);
            x1 = bf16_hi(raw[i][0][w]);
        }
    };
    // The diagonal's elements leave the matrix before it is split: the row of lane m of tile i meets them in chunk i of its
    // wave's order, product step 2 i + m / 16, lane half (m / 4) % 2.
    auto take_diagonal = [&](int s, int buffer) __attribute__((always_inline)) {
        const int i = s / 2;
        if (i >= RTILES) return;
        const bool mine = m >> 4 == s % 2 && ((m >> 2) & 1) == h;
        const int at = (m & 3) + 4 * ((m >> 3) & 1);
        float value = 0.0f;
#pragma unroll
        for (int x = 0; x < 8; ++x)
            if (mine && at == x) {
                if constexpr (WORDS == 2) {
                    value = __uint_as_float(raw[i][x >> 2][x & 3]);
                    raw[i][x >> 2][x & 3] = 0;
                } else {
                    const unsigned w = raw[i][0][x >> 1];
                    value = to_f32(__builtin_bit_cast(Tin, (unsigned short)((x & 1) ? w >> 16 : w & 0xffffu)));
                    raw[i][0][x >> 1] = w & ((x & 1) ? 0xffffu : 0xffff0000u);
                }
            }
        if (mine) diag[buffer * D + row0 + 32 * i + m] = value;
    };
    // The cotangents of 16-bit elements are summed by product steps, then over them (error against fp64 on random matrices, bf16 B=32
    // K=20 d=240: 7.0e-7 as one running sum, 4.3e-7 in the chain waves of the kernel these widths were padded to; here 4.4e-7).
    // fp32 ones were one running sum in the kernel before, too, and B=64 K=128 d=256 takes 1.84 ms like that, 1.87 by steps.
    constexpr bool SUM_BY_STEPS = NA < 3;
    // The vector work of a product step in units: unit n takes pair w of the next step's elements one plane further.
    float left0[RTILES][4], left1[RTILES][4], part[RTILES];
    constexpr int UNITS = 4 * NA * RTILES;
    auto unit = [&](int n, int par, bool chain) __attribute__((always_inline)) {
        const int i = n / (4 * NA), p = n % (4 * NA) / 4, w = n % 4;
        if (p == 0) {
            element_pair(i, w, left0[i][w], left1[i][w]);
            if (COT && chain) {
                if constexpr (SUM_BY_STEPS) {
                    part[i] = w == 0 ? left0[i][w] * vvec[0][0] : fmaf(left0[i][w], vvec[w >> 1][2 * (w & 1)], part[i]);
                    part[i] = fmaf(left1[i][w], vvec[w >> 1][2 * (w & 1) + 1], part[i]);
                    if (w == 3) vdot[i] += part[i];
                    asm volatile("" : "+v"(part[i]), "+v"(vdot[i]));   // the sums stay here: sunk to their use they would keep the rows alive
                } else {
                    vdot[i] = fmaf(left0[i][w], vvec[w >> 1][2 * (w & 1)], vdot[i]);
                    vdot[i] = fmaf(left1[i][w], vvec[w >> 1][2 * (w & 1) + 1], vdot[i]);
                    asm volatile("" : "+v"(vdot[i]));
                }
            }
            if constexpr (SCALE != 1.0f) {
                left0[i][w] *= SCALE;
                left1[i][w] *= SCALE;
            }
        }
        if constexpr (NA == 1) {
            afr[par][0][i][w] = raw[i][0][w];
        } else {
            afr[par][p][i][w] = pack_bf16(left0[i][w], left1[i][w]);
            if (p + 1 < NA) splitter.rest(afr[par][p][i][w], left0[i][w], left1[i][w]);
        }
    };
    const char* b_lane = smem + (size_t)(m * PITCH + h * 8) * 2;
    auto load_b = [&](int p, int s) __attribute__((always_inline)) {       // the fragments of one plane for product step s
#pragma unroll
        for (int j = 0; j < CTILES; ++j)
            bfr[p][j] = *reinterpret_cast<const u32x4*>(b_lane + first_k(s) * 2 + (p * PLANE + j * 32 * PITCH) * 2);
    };

    constexpr int NPROD = NA == 3 ? 6 : NA == 2 ? 5 : 3, MFMAS = NPROD * RTILES * CTILES;
    constexpr int STORE_STEPS = HALVES < 8 ? HALVES : 8;   // the product before is stored under the first product steps
    int cur = 0;
    int r = r_top;
    bool primed = false;
    bool pending = false;                   // tot is a result that is not stored yet (it goes to o_base[(r + 1) * o_stride])
    // `apart`: the diagonal's elements were taken out of the rows
    auto chain_out = [&](bool apart) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RTILES; ++i) {
            const int row = row0 + 32 * i + m;
            float total = vdot[i] + __shfl_xor(vdot[i], 32, 64);   // the two k halves of a row
            if (apart) total = fmaf(diag[cur * D + row], vbuf[cur * D + row], total);
            if (apart && __builtin_amdgcn_ballot_w64(!(__builtin_fabsf(total) <= 0x1.fffffep127f))) {
                // The rows are taken again as they lie: the first product step meets the vector with the sums of its elements'
                // planes, which are not the elements where those are not finite or round to infinity; and an element behind the
                // end of a row that is not finite must not meet the zeros the vector ends in.
                total = 0.0f;
                if (row < d) {
                    const Tin* a_row = a_base + (size_t)r * a_stride + (size_t)row * d;
#pragma unroll 8
                    for (int k = 0; k < d; ++k) total = fmaf(to_f32(a_row[k]), vbuf[cur * D + k], total);
                }
            }
            if (row >= d) total = 0.0f;   // (zero rows times an infinite vector)
            if (h == 0) {
                vbuf[(cur ^ 1) * D + row] = total;
                if (c0 == 0 && row < d) cot[((size_t)b * (K + 1) + r) * d + row] = total;
            }
        }
    };
    auto load_v = [&](int s) __attribute__((always_inline)) {
        const float* v = vbuf + cur * D + 4 * h + first_k(s);
        vvec[0] = *reinterpret_cast<const f32x4*>(v);
        vvec[1] = *reinterpret_cast<const f32x4*>(v + 8);
    };
    auto store_now = [&]() __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t o_r = rows(o_base + (size_t)(store_all ? r : r + 1) * o_stride, matrix_bytes);
#pragma unroll
        for (int n = 0; n < NEL; ++n) store_element(o_r, n);
    };
    while (true) {
        if (__builtin_expect(wide, 0)) {
            write_wide();
            if (pending) {
                ++r;
                store_now();
                --r;
            }
#pragma unroll
            for (int i = 0; i < RTILES; ++i) vdot[i] = 0.0f;
            wide_tile(a_base + (size_t)r * a_stride, false, COT, vdot, vbuf + cur * D);
            primed = false;
            pending = false;
            if (store_all || r == r_lo) store_now();
            if (COT) chain_out(false);
            cur ^= 1;
            if (r == r_lo) {
                wait_vm<0>();   // no transfer into LDS outlives the workgroup
                return;
            }
            const bool past = scale_up();
            split_all();
            publish(past);
            lds_barrier();
            wide = __builtin_amdgcn_readfirstlane(asked_wide()) != 0;
            --r;
            continue;
        }
        if (!primed) {
            if (__builtin_expect(!requested, 0)) {
                wait_vm<0>();
#pragma unroll
                for (int x = 0; x < kSlots; ++x) request(slot_at[x], r, x * HPS);
            }
            requested = false;
            wait_vm<0>();
            read_raw(slot_at[0], 0);
            take_diagonal(0, cur);
#pragma unroll
            for (int n = 0; n < UNITS; ++n) unit(n, 0, false);
            if constexpr (HPS == 1) {
                read_raw(slot_at[1], 0);
                asm volatile("" : : "v"(raw[0][0]) : "memory");
                request(slot_at[0], r, kSlots);
                const unsigned first = slot_at[0];
#pragma unroll
                for (int x = 0; x + 1 < kSlots; ++x) slot_at[x] = slot_at[x + 1];
                slot_at[kSlots - 1] = first;
            } else {
                read_raw(slot_at[0], 1);
            }
            primed = true;
        }
        const __amdgpu_buffer_rsrc_t o_prev = rows(o_base + (size_t)(r + 1) * o_stride, pending ? matrix_bytes : 0);
#pragma unroll
        for (int i = 0; i < RTILES; ++i) vdot[i] = 0.0f;
        // The step begins with the k of the wave's own rows, which need no barrier.
#pragma unroll
        for (int p = NP - 1; p >= 0; --p) load_b(p, 0);
        if (COT) load_v(1);
        asm volatile("" : "+s"(row_elements));   // row offsets are cheaper formed again than kept
        int asked = 0;
        f32x4 dg[RTILES][4];
        // four rows of a tile: the sums come together, with the diagonal's product, and are split
        auto finish = [&](int i, int j, int q) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 4; ++x)
                tot[i][j][4 * q + x] = fmaf(dg[i][q][x], tot[i][j][4 * q + x], top[i][j][4 * q + x] + fine[i][j][4 * q + x]);
            split_tile(i, j, q);
        };
        auto product_step = [&](const int s) __attribute__((always_inline)) {
            const int par = s & 1;
            const bool chain_next = s + 1 < HALVES;
            // The two waves of a SIMD would take turns by age, one idle while the other ends its step: whoever is behind goes first.
            if constexpr (HALVES == 16) {
                if (s == 0) __builtin_amdgcn_s_setprio(3);
                else if (s == 8) __builtin_amdgcn_s_setprio(2);
                else if (s == 12) __builtin_amdgcn_s_setprio(1);
                else if (s == 14) __builtin_amdgcn_s_setprio(0);
            }
            if (s == 1 && COT && HALVES > 2) load_v(2);
            // raw holds the elements of product step s + 1.  Its slot (the older step pair's, for 16-bit storage) is free.
            if (HPS == 1 || par == 0) {
#pragma unroll
                for (int i = 0; i < RTILES; ++i)
#pragma unroll
                    for (int w = 0; w < WORDS; ++w) asm volatile("" : "+v"(raw[i][w]));
                request(slot_at[0], r, HPS == 1 ? s + 1 + kSlots : s + 2 * kSlots);
                const unsigned first = slot_at[0];
#pragma unroll
                for (int x = 0; x + 1 < kSlots; ++x) slot_at[x] = slot_at[x + 1];
                slot_at[kSlots - 1] = first;
            }
            take_diagonal((s + 1) % HALVES, s + 1 < HALVES ? cur : cur ^ 1);
            if (s == HALVES - 1) {
#pragma unroll
                for (int i = 0; i < RTILES; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) dg[i][q] = *reinterpret_cast<const f32x4*>(diag + cur * D + row_of(i, 4 * q));
            }
            int y = 0, done = 0, finished = 0;
            // one product and the share of the vector work that goes under it
            auto product = [&](int sp, int ap, int i, int j) __attribute__((always_inline)) {
                f32x16 zero;
#pragma unroll
                for (int x = 0; x < 16; ++x) zero[x] = 0.0f;
                if (ap + sp) fine[i][j] = mma(afr[par][ap][i], bfr[sp][j], s == 0 && sp == NP - 1 ? zero : fine[i][j]);
                else top[i][j] = mma(afr[par][ap][i], bfr[sp][j], s == 0 ? zero : top[i][j]);
                ++y;
                const int before = done;
#pragma unroll
                for (; done < y * UNITS / MFMAS; ++done) unit(done, par ^ 1, chain_next);
                if (s < STORE_STEPS) {
                    const int from = (s * MFMAS + y - 1) * NEL / (STORE_STEPS * MFMAS), to = (s * MFMAS + y) * NEL / (STORE_STEPS * MFMAS);
#pragma unroll
                    for (int n = from; n < to; ++n) store_element(o_prev, n);
                }
                // the last unit that looks at raw has run: the elements of product step s + 2
                constexpr int LAST = UNITS - 4 * NA + 3;
                if (before <= LAST && done > LAST) {
                    if (COT && s > 0 && s + 2 < HALVES) load_v(s + 2);
                    if constexpr (HPS == 1) {
                        // its slot was requested at the start of step s + 1 - kSlots; younger: the requests since and the stores
                        // of the product steps between
                        constexpr int PER_STEP = NEL / STORE_STEPS;
                        int stores = 0;
#pragma unroll
                        for (int back = 1; back < kSlots; ++back) stores += s >= back && s - back < STORE_STEPS;
                        wait_younger<2 * RTILES * (kSlots - 1), PER_STEP, kSlots - 1>(stores);
                        read_raw(slot_at[0], 0);
                    } else {
                        // of a pair of steps; younger: the requests of the pairs since
                        if (par == 0) wait_vm<2 * RTILES * (kSlots - 1)>();
                        read_raw(slot_at[0], par);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            if (s + 1 < HALVES) {
#pragma unroll
                for (int sp = NP - 1; sp >= 0; --sp) {
#pragma unroll
                    for (int ap = NA - 1; ap >= 0; --ap) {
                        if (ap + sp > 2) continue;
#pragma unroll
                        for (int i = 0; i < RTILES; ++i)
#pragma unroll
                            for (int j = 0; j < CTILES; ++j) product(sp, ap, i, j);
                    }
                    load_b(sp, s + 1);      // a plane is next wanted after the products of the other two
                }
            } else {
                // the last product step takes one column tile after the other: a finished one is split under the next one's products
#pragma unroll
                for (int j = 0; j < CTILES; ++j) {
                    int n = 0;
#pragma unroll
                    for (int sp = NP - 1; sp >= 0; --sp)
#pragma unroll
                        for (int ap = NA - 1; ap >= 0; --ap) {
                            if (ap + sp > 2) continue;
#pragma unroll
                            for (int i = 0; i < RTILES; ++i) {
                                product(sp, ap, i, j);
                                ++n;
                                // (from the second product on: the last one's result takes two products' time)
                                constexpr int PER_COLUMN = MFMAS / CTILES;
                                if (j > 0 && n >= 2) {
#pragma unroll
                                    for (; finished < 4 * RTILES * (j - 1) + 4 * RTILES * (n - 1) / (PER_COLUMN - 1); ++finished)
                                        finish(finished / 4 % RTILES, finished / (4 * RTILES), finished % 4);
                                    __builtin_amdgcn_sched_barrier(0);
                                }
                            }
                        }
                }
#pragma unroll
                for (; finished < 4 * RTILES * CTILES; ++finished) finish(finished / 4 % RTILES, finished / (4 * RTILES), finished % 4);
            }
            if (COT && s == 0) {
                // the first elements of the step were split before its vector was there: they are the sum of their planes
                const float* v = vbuf + cur * D + 4 * h + first_k(0);
#pragma unroll
                for (int i = 0; i < RTILES; ++i) {
                    float first = 0.0f;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        float x0 = 0.0f, x1 = 0.0f;
#pragma unroll
                        for (int p = NA - 1; p >= 0; --p) {
                            x0 += bf16_lo(afr[0][p][i][w]);
                            x1 += bf16_hi(afr[0][p][i][w]);
                        }
                        first = fmaf(x0 * (1.0f / SCALE), v[2 * w + (w >= 2 ? 4 : 0)], first);
                        first = fmaf(x1 * (1.0f / SCALE), v[2 * w + (w >= 2 ? 4 : 0) + 1], first);
                    }
                    vdot[i] += first;
                }
            }
        };
        product_step(0);
        lds_barrier();                      // the other rows of the block are there
        asked = asked_wide();
        if constexpr (HALVES > 2) product_step(1);
        wide = __builtin_amdgcn_readfirstlane(asked) != 0;
        if (__builtin_expect(wide, 0)) continue;                 // (nothing but raw and the planes of the rows has changed: both are made again)
        if constexpr (HALVES == 2) product_step(1);
#pragma unroll
        for (int s = 2; s < HALVES; ++s) product_step(s);
        const bool bad = out_of_range(0x1p127f);
        if (__builtin_expect(bad, 0)) {
            float none[RTILES];
            wide_tile(a_base + (size_t)r * a_stride, true, false, none, nullptr);
        }
        if (COT) chain_out(true);
        cur ^= 1;
        if (r == r_lo) {
            store_now();
            wait_vm<0>();
            return;
        }
        pending = store_all;
        publish(bad);
        --r;
    }
}

template <typename Tin, int D, int CB, bool COT, int MODE>
int launch_mode(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, hipStream_t stream, ScanPlan plan) {
    constexpr int NB = D / CB;
    constexpr size_t bytes = lds_bytes(D, CB, COT, MODE);
    static_assert(bytes <= 160 * 1024, "LDS budget");
    if (int rc = ensure_dynamic_lds<&scan_planes_kernel<Tin, D, 32, CB, COT, MODE>>(bytes)) return rc;
    // chains in this launch (the kernel derives the same number from the plan)
    const int chains = B * (MODE == 1 ? plan.C - 1 : MODE == 3 ? plan.C - 2 : 1);
    const dim3 grid(chains >= 8 ? ((chains + 7) / 8) * 8 * NB : chains * NB);
    hipLaunchKernelGGL((scan_planes_kernel<Tin, D, 32, CB, COT, MODE>), grid, dim3(2 * D), bytes, stream,
                       static_cast<const Tin*>(mats), static_cast<float*>(out), static_cast<const float*>(g),
                       static_cast<float*>(cot), B, K, d, plan);
    LBI_HIP_CHECK(hipGetLastError());
    return LBI_OK;
}

// The whole chain in one launch, with the cotangent chain where `cot` is given.
template <typename Tin, int D, int CB>
int launch(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, hipStream_t stream) {
    const ScanPlan whole{0, 0, 0, 0, 0, 0, 0};
    return cot ? launch_mode<Tin, D, CB, true, 0>(mats, out, g, cot, B, K, d, stream, whole)
               : launch_mode<Tin, D, CB, false, 0>(mats, out, nullptr, nullptr, B, K, d, stream, whole);
}

}  // namespace scan_planes
}  // namespace lbi
