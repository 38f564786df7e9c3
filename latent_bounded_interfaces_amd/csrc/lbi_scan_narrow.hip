// Suffix scan of narrow matrices: which form a call takes, and its launches (kernel: lbi_scan_narrow_kernel.h).
#include "lbi_scan_narrow.h"

#include "lbi_scan_planes.h"

namespace lbi {
namespace scan_narrow {

// One launch, a whole chain (plan.phase 0) or a phase of the plan, on blocks of 16 `tiles` columns (1 or 2); `carry`: the vector of a whole
// chain beside the first block of 32.  An instance per storage type in a source of its own.
template <typename Tin>
int launch_type(const void* mats, void* out, const void* g, void* cot, int B, int K, int d, int tiles, bool carry,
                const ScanPlan& plan, hipStream_t stream);
extern template int launch_type<float>(const void*, void*, const void*, void*, int, int, int, int, bool, const ScanPlan&, hipStream_t);
extern template int launch_type<_Float16>(const void*, void*, const void*, void*, int, int, int, int, bool, const ScanPlan&, hipStream_t);
extern template int launch_type<bf16_raw>(const void*, void*, const void*, void*, int, int, int, int, bool, const ScanPlan&, hipStream_t);

int launch(const void* mats, int in_dtype, void* out, const void* g, void* cot, int B, int K, int d, int tiles, bool carry,
           const ScanPlan& plan, hipStream_t stream) {
    switch (in_dtype) {
        case LBI_F32: return launch_type<float>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        case LBI_F16: return launch_type<_Float16>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
        default: return launch_type<bf16_raw>(mats, out, g, cot, B, K, d, tiles, carry, plan, stream);
    }
}

// Compute units of the smallest partition of the part.
constexpr int kLeastCus = 32;

// us of a step on blocks of 16 `tiles` columns: of workgroups that have a CU to themselves (fp32, fitted with the other constants, up to a tenth below
// the 0.15 ... 1.30 that a step alone takes), and how much longer it takes
// where `groups` workgroups share the chip: up to 48 columns several run on a CU side by side, at 64 two, beyond one (the rings), and what
// they read then counts, too (d = 128 B = 16 K = 74, inputs from memory: 1.9).
float step_us(int nt, int tiles, int64_t groups, int cus) {
    static constexpr float alone[8] = {0.14f, 0.24f, 0.31f, 0.41f, 0.77f, 0.88f, 1.05f, 1.22f};
    const float full = (float)groups / (float)cus, rounds = (float)((groups + cus - 1) / cus);
    float share = 1.0f;
    if (nt > 4) share = rounds * (1.0f + (nt > 6 ? 1.5f : 0.6f) * full / (rounds * (float)tiles));
    else if (groups > cus) share = nt < 4 ? 1.0f + 0.5f * (full - 1.0f) : 1.8f * (float)((groups + 2 * cus - 1) / (2 * cus));
    return alone[nt - 1] * share * (tiles == 2 ? 1.8f : 1.0f);
}

// Chains are dealt to the eight XCDs, so it is the fullest one that counts.
int64_t dealt(int64_t chains) { return chains >= 8 ? (chains + 7) / 8 * 8 : chains; }

// Chunks of L matrices (0: the plain chain), their phases 1 and 3 on blocks of 16 `tiles` columns.
struct Chunks { int L, tiles; };

// The form with the least estimated time: chunks are three launches instead of one and about twice the products, but 2 L + C - 4
// dependent steps instead of K - 1; blocks of 32 columns, the vector beside the first, take 1.8 times as long for a step of half as
// many workgroups.  Room is left for the vector whether it is asked for or not: the matrices are the same bits with and without.  K = 128, fp32,
// matrices, us, plain -> chunks: d = 16 B = 1 18 -> 12; d = 32 B = 4 31 -> 17, B = 64 32 -> 32; d = 64 B = 4 52 -> 23, B = 32 54 (59 in
// chunks, not taken); d = 128 B = 1 156 -> 49, B = 4 154 -> 61; B = 7 K = 120, inputs from memory,
// in chunks 122 on 16 columns, 92 on 32.
Chunks chunks(int B, int K, int nt, bool half, int cus) {
    const int forced = scan_forced_chunk();
    if (forced == 0 || K < 12) return {0, 1};
    if (forced > 0) {
        const int L = forced < 2 ? 2 : forced;
        return {(K + L) / L >= 4 ? L : 0, 1};
    }
    // Beyond 64 columns a plain chain whose blocks of 16 don't find a CU each runs on 32, and chunks have never been the better form then (13 widths,
    // B = 8 ... 768, K = 13 ... 100: 253 calls 1.18 times as long in chunks).
    if (nt > 4 && dealt(B) * nt > cus) return {0, 1};
    const float plain = 5.0f + (float)(K - 1) * step_us(nt, 1, dealt(B) * nt, cus);
    float best = plain;
    int64_t groups = 0;
    Chunks form{0, 1};
    for (int L = 2; (K + L) / L >= 4; L += 1 + L / 16) {
        const int C = (K + L) / L;
        const int64_t chains = dealt((int64_t)B * (C - 1));
        const float between = 12.0f + (float)(C - 2) * step_us(nt, 1, dealt(B) * nt, cus);
        for (int tiles = 1; tiles <= (nt > 3 ? 2 : 1); ++tiles) {
            const int64_t blocks = chains * (tiles == 2 ? (nt + 1) / 2 : nt + 1);
            const float cost = between + (float)(2 * L - 2) * step_us(nt, tiles, blocks, cus);
            if (cost < best) {
                best = cost;
                groups = blocks;
                form = {L, tiles};
            }
        }
    }
    // The estimate is good to a tenth, and what it misses where chunks fill the CUs is the same for calls alike (measured / estimated part of the plain chain): 7 and 8
    // row tiles 1.17 / 0.91 (bf16 d = 128 B = 16 K = 24), 0.90 / 0.90 (B = 8 K = 24); 5 and 6 1.13 / 0.99 (bf16 d = 80 B = 24 K = 50), 0.80 / 0.93 (B = 8 K =
    // 24); fp32 at 4 1.19 / 0.97 (d = 64 B = 32 K = 100); at 3, ten workgroups a CU, 1.29 / 0.94 (d = 33 B = 40 K = 100).
    const bool crowd = !half && nt == 3 && groups >= 8 * (int64_t)cus;
    const float full = nt > 7 ? 0.905f : nt > 6 ? 0.93f : nt > 4 ? 0.97f : crowd ? 0.85f : nt == 4 && !half ? 0.95f : 1.0f;
    return best < (5 * groups >= 4 * (int64_t)cus ? full : 1.0f) * plain ? form : Chunks{0, 1};
}

// 16-bit rows that are no whole 4-byte words come straight into registers at all widths.
static bool in_words(const void* mats, int d, int in_dtype) {
    return in_dtype == LBI_F32 || (d % 2 == 0 && reinterpret_cast<uintptr_t>(mats) % 4 == 0);
}

// Where the chip has several workgroups for every CU to run one after the other, a step's length no longer counts, and 32 x 32
// tiles move half the operands.  The matrices are the same bits with the cotangents and without, so it is one rule for both, and its lines lie where
// the two together begin to take longer here (15492 calls: 14 widths, three types, B = 8 ... 2048, K = 2 ... 100, inputs from memory
// and from the caches).  us, 32 x 32 tiles -> here, matrices / with the cotangents:
//  * up to 32 columns several small workgroups share a CU: fp32 d = 32 B = 1024 K = 50 150 -> 150 / 173 -> 169, B = 1536 K = 24 118 -> 145 / 133 -> 154.
//  * 33 ... 48, and 49 ... 64 where 16-bit rows come through LDS: bf16 d = 64 B = 768 K = 24 136 -> 98 / 149 -> 120.  In registers at most one
//    workgroup of 32 columns a CU twice over: fp32 d = 49 B = 256 K = 24 46 -> 35 / 57 -> 46, B = 288 47 -> 52 / 57 -> 66.
//  * beyond 64 columns while a step's blocks of 32 find a CU each: fp32 d = 81 B = 80 K = 24 56 -> 57 / 70 -> 63, B = 96 58 -> 71 / 72 -> 83; d = 128 B = 64
//    K = 100 319 -> 293 / 350 -> 315, B = 72 323 -> 353 / 352 -> 381; three quarters of them for 16-bit rows of 97 ... 127.  Odd 16-bit widths, whose
//    rows come straight into registers, take them in chains of eight matrices and more: bf16 d = 81 B = 64 K = 4 11 -> 15 / 19 -> 15, K = 8 20 -> 22 / 28 -> 24.
bool takes(const void* mats, int B, int K, int d, int in_dtype) {
    if (d < 2 || d > 128) return false;
    if (d <= 16 || scan_forced_chunk() > 0) return true;   // the others take whole chains of more than 16 columns
    const int nt = row_tiles(d, in_dtype);
    if (dealt(B) * nt <= kLeastCus) return true;           // on any device: small calls do without asking the runtime
    const int64_t cus = device_compute_units();
    const bool words = in_words(mats, d, in_dtype), half = in_dtype != LBI_F32, whole = d == 16 * nt;
    if (nt <= 2) return B <= (whole || K >= 24 ? 4 : 2) * cus;
    if (nt == 3 || (nt == 4 && half && words)) return B <= (K < (whole ? 4 : 8) ? 1 : 3) * cus;
    if (nt == 4) return 2 * B <= (whole || K >= 8 ? 2 : 1) * cus;
    if (!words && K < 8) return dealt(B) * nt <= cus;
    return 4 * dealt(B) * ((nt + 1) / 2) <= (half && nt == 8 && !whole ? 3 : 4) * cus;
}

// A chain of vectors is its vector's block of a scan (15 of the 16 columns are empty: a step is as long as the fp32 products of one tile
// column). The kernels for whole 16-byte pieces of rows (fold of a staged copy) and for other rows (a row a lane group) take 0.6 to 3 us a
// step for d = 16 ... 128; they move more a step, which counts where the chains fill the chip. us, those -> this, fp32 / bf16: B = 64 K = 128
// d = 32 86 / 74 -> 35 / 39; d = 64 140 / 112 -> 66 / 69; d = 96 265 / 191 -> 142 / 141; d = 128 B = 40 K = 90 295 -> 168, B = 64 K = 128 232 -> 188
// (bf16).  d < 17 (scalar before unless in whole pieces): B = 64 K = 128 d = 12 fp16 550 -> 28; fp32 B = 4096 K = 64 d = 16 310 -> 64; but a chain of
// one to four matrices of two to four columns is less than a workgroup's start here: fp32 B = 65536 d = 2 K = 1 17 -> 30, K = 4 45 -> 49, K = 6 69 -> 59; d = 3
// K = 2 39 -> 44, K = 3 52 -> 47.  Past the other lines: B = 512 K = 20 d = 80 bf16 32 -> 55, d = 101 B = 64 K = 128 150 / 123 -> 219 / 240, d = 112
// fp16 B = 16 K = 90 154 -> 156, B = 64 K = 12 d = 47 bf16 9.5 -> 10.3, d = 72 fp16 B = 64 K = 8 12 -> 14 (six row tiles for five), d = 56 fp32 B = 512
// K = 4 9 -> 11, d = 128 bf16 B = 256 K = 4 11 -> 13, d = 31 B = 1024 K = 2 7 -> 10; 16-bit matrices that start off the 4-byte grid (their rows would not come
// through LDS here), bf16 B = 16 K = 20, d = 64 19.8 -> 25.3, d = 128 42.6 -> 82.7.
bool takes_chain(const void* mats, int B, int K, int d, int in_dtype) {
    if (d < 2 || d > 128) return false;
    const bool pieces = d % (in_dtype == LBI_F32 ? 4 : 8) == 0 && reinterpret_cast<uintptr_t>(mats) % 4 == 0;
    if (d <= 16) return pieces || (int64_t)K * d * d > 18 || B <= 16 * (int64_t)device_compute_units();
    if (!pieces && (d > 48 || (d > 32 && K < 20))) return false;
    const bool half = in_dtype != LBI_F32;
    if (half && ((d > 96 && d != 128) || (d > 64 && d <= 80 && K < 24))) return false;
    const int64_t cus = device_compute_units();
    if (d <= 48) return B <= (K < 4 ? 3 : 4) * cus;
    if (d <= 64) return B <= (K >= 13 && (half || d == 64) ? 4 : 1) * cus;
    return 4 * B <= (half && d == 128 && K < 8 ? 1 : 4) * cus;
}

int chain(const void* mats, int in_dtype, const void* g, void* cot, int B, int K, int d, hipStream_t stream) {
    return launch(mats, in_dtype, nullptr, g, cot, B, K, d, 1, false, ScanPlan{0, 0, 0, 0, 0, 0, 0}, stream);
}

int scan(const void* mats, int in_dtype, void* out, const void* g, void* cot, int B, int K, int d, hipStream_t stream) {
    ScanPlan plan{0, 0, 0, 0, 0, 0, 0};
    const int nt = row_tiles(d, in_dtype);
    if (K < 12 && dealt(B) * (nt + 1) <= kLeastCus) return launch(mats, in_dtype, out, g, cot, B, K, d, 1, false, plan, stream);
    const int cus = device_compute_units();
    if (const Chunks form = chunks(B, K, nt, in_dtype != LBI_F32, cus); form.L) {
        plan.L = form.L;
        plan.C = (K + form.L) / form.L;
        plan.s = 1;
        for (plan.phase = 1; plan.phase <= 3; ++plan.phase) {
            const bool totals = plan.phase == 2;   // operands and results are fp32 products inside `out`
            if (int rc = launch(totals ? out : mats, totals ? LBI_F32 : in_dtype, out, g, totals ? nullptr : cot, B, K, d,
                                totals ? 1 : form.tiles, form.tiles == 2 && !totals, plan, stream))
                return rc;
        }
        return LBI_OK;
    }
    // 16 columns a workgroup while every workgroup finds room at once, 32 beyond (a step of those takes 1.5-1.9 times as long); the vector
    // in a workgroup of its own while that does.  fp32 K = 128 with cotangents, us, 16 / 32 / 32 with the vector beside: d = 64 B = 32
    // 54 / 90 / -, B = 64 131 / 99 / 126; d = 128 B = 32 402 / 303 / 325, B = 64 709 / 610 / 377.
    const int64_t room = nt <= 3 ? 8 * cus / nt : cus, more = cot ? 1 : 0;
    const int tiles = nt > 1 && dealt(B) * (nt + more) > room ? 2 : 1;
    const bool carry = tiles == 2 && cot && dealt(B) * ((nt + 1) / 2 + 1) > room;
    return launch(mats, in_dtype, out, g, cot, B, K, d, tiles, carry, plan, stream);
}

}  // namespace scan_narrow
}  // namespace lbi
