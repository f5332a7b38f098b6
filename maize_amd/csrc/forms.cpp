#include "forms.hpp"

#include <cmath>
#include <cstdio>
#include <cstring>

#include "dispatch.hpp"

namespace maize {
namespace {

inline uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }
inline uint64_t cdiv64(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// ---- maize_tile_*: tiles of 32 x 128, 64 x 64, 64 x 128 and (but for fp64) 128 x 128 (kernels/gemm_tile.hpp) -------------
enum Tile : uint32_t { T32x128, T64x64, T64x128, T64x64W, T128x128, kTiles };     // W: 8-bit operands widened to bf16
constexpr const char* const kOperands[8] = {"bf16", "f16", "e4m3", "e5m2", "e4m3e5m2", "e5m2e4m3", "f32", "f64"};   // maize_in_type_t's order
constexpr uint32_t kTileForms = 8u * 2u * kTiles;
static_assert(kTileForms <= kMaxForms, "the context's table of functions");
bool tile_exists(uint32_t in_type, uint32_t tile) {
    const bool wide = in_type >= MAIZE_IN_F32;
    return tile == T64x64W ? !wide && in_type >= MAIZE_IN_E4M3 : tile == T128x128 ? in_type != MAIZE_IN_F64 : true;
}
struct Names {
    char name[kTileForms][40];
    Names() {
        static const char* const kShape[kTiles] = {"32x128", "64x64", "64x128", "64x64w", "128x128"};
        for (uint32_t i = 0; i < kTileForms; ++i) {
            const uint32_t t = i % kTiles, nt = i / kTiles % 2u, op = i / kTiles / 2u;
            if (!tile_exists(op, t)) name[i][0] = 0;
            else std::snprintf(name[i], sizeof name[i], "maize_tile_%s_%s_%s", kOperands[op], nt ? "nt" : "nn", kShape[t]);
        }
    }
};
const Names& names() {
    static const Names n;
    return n;
}

// What a launch costs, in microseconds, fitted to 3800 timings of 600 products (operands cycled through three sets, so that
// what does not fit the memory-side cache comes from HBM; residuals 8-14 %):
//   t0 + core + [K tail] tail + [K ranges] (r0 + r1 * ranges)
// core: `one` per K tile where a compute unit has one workgroup, `many` per K tile and workgroup where it has several (what
// bounds them is the rate at which a compute unit's LDS is filled: 75-100 GB/s) and `turn` for each workgroup after the first;
// rows of A (B) that are no 16-byte material make the requests longer by ua (ub), transposing reads by nn, 8-bit
// operands by e8; at least bytes / bw.
struct TileCost { uint32_t bm, bn; double t0, one, many, turn, r0, r1, ua, ub, nn, bw, tail, e8; };
// 128 x 128 has a compute unit to itself and half of the LDS fill per product of 64 x 128: where its tiles make up one round or
// few (129 to 256: 1024 x 3072 x 1999 into bf16 30.1 -> 24.5 us, 4499 x 520 x 3644 51.1 -> 35.8; below, K ranges of smaller tiles
// keep the chip busier).  Fitted to 110 timings, residuals 7 % where it is a candidate.
constexpr TileCost kTileCost[kTiles] = {
    {32, 128, 3.62, 0.215, 0.371, 0.0, 1.63, 0.14, 0.18, 0.36, 0.0, 6.55, 0.55, 0.07},
    {64, 64, 3.97, 0.167, 0.177, 1.06, 1.82, 0.19, 0.11, 0.40, 0.14, 6.88, 0.30, 0.10},
    {64, 128, 4.10, 0.278, 0.292, 1.49, 1.33, 0.54, 0.24, 0.25, 0.04, 6.03, 0.29, 0.09},
    {64, 64, 3.57, 0.329, 0.276, 1.27, 2.20, 0.22, 0.12, 0.15, 0.10, 5.21, 0.65, -0.04},
    {128, 128, 4.42, 0.527, 0.527, 5.42, 0.0, 0.0, 0.14, 0.16, -0.05, 4.00, 1.50, -0.01},
};
// fp32 and fp64 operands: bound by the matrix instructions (a K tile of 64 x 64 is 1024 of their cycles, 0.43 us), so alignment
// and layout cost next to nothing.  Fitted to 18600 timings of 1977 products, residuals 5-6 %.
constexpr TileCost kFullCost[2][kTiles] = {
    {{32, 128, 3.48, 0.548, 0.560, 1.82, 2.22, 0.22, 0.0, 0.0, 0.0, 6.49, 0.30, 0.0},
     {64, 64, 3.50, 0.541, 0.489, 1.90, 2.26, 0.23, 0.0, 0.0, 0.0, 8.34, 0.27, 0.0},
     {64, 128, 4.12, 1.006, 0.905, 2.83, 1.28, 0.59, 0.0, 0.0, 0.03, 7.19, 0.27, 0.0},
     {},
     {128, 128, 4.24, 2.129, 1.876, 3.89, 0.0, 0.0, 0.0, 0.0, 0.0, 4.00, 0.41, 0.0}},
    {{32, 128, 4.05, 0.532, 0.558, 2.43, 1.71, 0.46, 0.0, 0.0, 0.0, 6.43, 0.29, 0.0},
     {64, 64, 4.20, 0.524, 0.477, 2.72, 1.55, 0.52, 0.0, 0.0, 0.0, 8.58, 0.11, 0.0},
     {64, 128, 5.28, 0.968, 0.893, 4.59, 1.42, 1.03, 0.0, 0.0, 0.03, 6.77, 0.17, 0.0}},
};
// The longer of two times that overlap, smoothly (their 4-norm).
inline double longer(double a, double b) {
    const double a2 = a * a, b2 = b * b;
    return std::sqrt(std::sqrt(a2 * a2 + b2 * b2));
}
struct Problem {
    Dims s;
    uint32_t batch, esz, bke, steps, cus;    // bytes per element of A and B; elements and number of K tiles
    bool rows_a, rows_b, tail;               // rows that are 16-byte material; a ragged last K tile
    double bytes;                            // each operand once
};
double tile_cost(const TileCost& c, const Problem& p, uint64_t tiles, uint32_t ks) {
    const uint32_t per = cdiv(p.steps, ks);
    const double items = (double)(tiles * ks), each = (p.rows_a ? 1.0 : 1.0 + c.ua) * (p.rows_b ? 1.0 : 1.0 + c.ub) * (p.s.nt ? 1.0 : 1.0 + c.nn) * (p.esz == 1u ? 1.0 + c.e8 : 1.0);
    const uint64_t n = cdiv64(tiles * ks, p.cus);
    const double core = n <= 1u ? per * c.one * each : per * c.many * each * (n > 6u ? items / p.cus : (double)n) + c.turn * (double)(n - 1u);
    return c.t0 + longer(core, p.bytes / (c.bw * 1e6)) + (p.tail ? c.tail : 0.0) + (ks > 1u ? c.r0 + c.r1 * ks : 0.0);
}

// The registry's kernels, by what their time depends on.  The same fit, of the time of the call (kernel, copies and reduce
// pass) on the same products: one coefficient set per family, residuals 8-23 %.
enum Family : uint32_t { kSkinnyNN, kSkinnyNT, kCopies, kT128, kH128, kH128R3, kMT256, kH128Split, kMT256Split, kAnyShape, kWide };
Family family_of(const char* name) {
    if (std::strstr(name, "_mt128_")) return kWide;
    if (std::strstr(name, "_wave32")) return kAnyShape;
    if (std::strstr(name, "_skinny_nn")) return kSkinnyNN;
    if (std::strstr(name, "_skinny_nt")) return kSkinnyNT;
    if (std::strstr(name, "_packed") || std::strstr(name, "_trb")) return kCopies;
    if (std::strstr(name, "_t128_")) return kT128;
    if (std::strstr(name, "_splitk")) return std::strstr(name, "_h128") ? kH128Split : kMT256Split;
    return std::strstr(name, "_h128r3") ? kH128R3 : std::strstr(name, "_h128") ? kH128 : kMT256;
}
const Family* families() {
    struct Table {
        Family of[kMaxKernels];
        Table() { for (uint32_t i = 0; i < kernel_count(); ++i) of[i] = family_of(kernel_at(i).name); }
    };
    static const Table t;
    return t.of;
}
// t0, per K tile and round, per further round, per Mi elements of C (and round), per K range, per K range and Mi elements, 8-bit.
struct TiledCost { uint32_t bm, bn; double t0, step, round, c, range, crange, e8; };
double tiled_cost(const TiledCost& c, const Problem& p, uint32_t ks) {
    const double elems = (double)p.s.m * p.s.n * p.batch * 1e-6;
    const double rounds = (double)cdiv64((uint64_t)cdiv(p.s.m, c.bm) * cdiv(p.s.n, c.bn) * p.batch * ks, p.cus);
    const double core = rounds * cdiv(p.steps, ks) * c.step * (p.esz == 1u ? 1.0 + c.e8 : 1.0) + (rounds - 1.0) * c.round;
    return c.t0 + longer(core, p.bytes / 4.6e6) + c.c * elems / rounds + (c.range + c.crange * elems) * ks;
}
double registry_cost(Family f, const Problem& p, uint32_t ks) {
    if (ks == 0u) ks = 1u;
    switch (f) {
        case kSkinnyNN: case kSkinnyNT: {
            const bool nn = f == kSkinnyNN;
            const uint32_t groups = p.s.m <= 16u ? 1u : p.s.m <= 32u ? 2u : 4u;
            const double rounds = (double)cdiv64((uint64_t)cdiv(p.s.n, 256) * p.batch * ks, p.cus);
            const double core = rounds * cdiv(p.steps, ks) * (nn ? 0.44 : 0.85);
            return (nn ? 3.5 : 1.0) + longer(core, p.bytes / (nn ? 6.35e6 : 5.33e6)) + (ks > 1u ? (nn ? 3.8 : 0.0) + (nn ? 0.19 : 0.65) * ks * groups : 0.0);
        }
        case kCopies: {
            const double rounds = (double)cdiv64((uint64_t)cdiv(p.s.m, 256) * cdiv(p.s.n, 256) * p.batch * ks, p.cus);
            return 16.5 + rounds * cdiv(p.steps, ks) * 1.175 + 0.69e-6 * p.batch * p.esz * ((double)p.s.m + p.s.n) * p.s.k + 2.07e-6 * p.s.m * p.s.n * p.batch * ks;
        }
        case kT128:       return tiled_cost({128, 128, 4.6, 0.385, 7.1, 0.2, 0.0, 0.0, 0.0}, p, 1u);
        case kH128:       return tiled_cost({128, 256, 5.3, 0.63, 12.0, 0.4, 0.0, 0.0, 0.45}, p, 1u);
        case kH128R3:     return tiled_cost({128, 256, 2.75, 0.775, 7.1, 0.52, 0.0, 0.0, 0.07}, p, 1u);
        case kMT256:      return tiled_cost({256, 256, 6.9, 1.27, 4.4, 0.06, 0.0, 0.0, 0.08}, p, 1u);
        case kH128Split:  return tiled_cost({128, 256, 6.6, 0.73, 8.8, 0.0, 0.37, 1.42, 0.07}, p, ks);
        case kMT256Split: return tiled_cost({256, 256, 6.8, 1.68, 12.0, 0.33, 0.0, 1.8, 0.0}, p, ks);
        default:          return 1e9;
    }
}

}  // namespace

uint32_t form_count() { return kTileForms; }
const char* form_name(uint32_t index) {
    const char* n = index < kTileForms ? names().name[index] : "";
    return n[0] ? n : nullptr;
}

bool choose_form(const maize_gemm_ex_desc_t& d, uint32_t registry, uint32_t compute_units, FormPlan* out) {
    const Family fam = families()[registry];
    if (compute_units == 0u) return false;
    Problem p;
    p.s = dims_of(d);
    p.batch = d.gemm.batch;
    p.cus = compute_units;
    const bool bits8 = d.in_type >= MAIZE_IN_E4M3 && d.in_type <= MAIZE_IN_E5M2_E4M3;
    p.esz = d.in_type == MAIZE_IN_F64 ? 8u : d.in_type == MAIZE_IN_F32 ? 4u : bits8 ? 1u : 2u;
    p.bke = 128u / p.esz;
    p.steps = cdiv(p.s.k, p.bke);
    p.tail = p.s.k % p.bke != 0u;
    const uint32_t lda = d.lda ? d.lda : d.gemm.a.ncols, ldb = d.ldb ? d.ldb : d.gemm.b.ncols, ldc = d.ldc ? d.ldc : d.gemm.c.ncols;
    // The tail's 16-byte loads end at the end of a row of A, of a row of B: there have to be that many elements.  32-bit offsets
    // span a tile's rows.
    const uint32_t chunk = 16u / p.esz;
    if (p.s.k < chunk || (!p.s.nt && p.s.n < chunk)) return false;
    if (p.s.k >= (1u << 21) || p.s.n >= (1u << 21) || lda >= (1u << 21) || ldb >= (1u << 21) || ldc >= (1u << 21)) return false;
    auto rows16 = [&](const void* ptr, uint32_t ld, uint64_t stride) {
        return (((uintptr_t)ptr | (uint64_t)ld * p.esz | (p.batch > 1u ? stride * p.esz : 0u)) & 15u) == 0u;
    };
    p.rows_a = rows16(d.gemm.a.ptr, lda, d.gemm.stride_a);
    p.rows_b = rows16(d.gemm.b.ptr, ldb, d.gemm.stride_b);
    const double c_bytes = fam == kWide ? p.esz : d.out_type == MAIZE_OUT_F32 ? 4.0 : 2.0;
    p.bytes = p.batch * (p.esz * ((double)p.s.m + p.s.n) * p.s.k + c_bytes * p.s.m * p.s.n * (d.beta != 0.0f ? 2.0 : 1.0));

    LaunchDims ld;
    std::memset(&ld, 0, sizeof ld);
    if (!kernel_at(registry).plan(d, compute_units, &ld)) return false;       // (what the registry's kernel refuses stays refused)
    // fp32 and fp64: the form always.  Of 1977 drawn products the registry's 128 x 128 tiles through registers were ahead of the
    // best tile on four, by 3 % at most, and 4.3 times as long on average.
    const double rival = fam == kAnyShape || fam == kWide ? 1e9 : registry_cost(fam, p, ld.ksplit);

    // The any-shape kernel multiplies 8-bit operands widened to bf16: its form does too.  Everywhere else the other tiles.
    const bool widened = bits8 && fam == kAnyShape;
    double best = 1e9;
    uint32_t tile = 0u, ranges = 1u;
    // The 16-bit few-row kernels on a row-major B give the same bits whatever the batch and the row group: their forms keep
    // their K ranges (blocks of 32 rows there), boundaries included.
    const bool pinned = fam == kSkinnyNN && !bits8;
    const uint32_t ks_lo = pinned && ld.ksplit > 1u ? ld.ksplit : 1u, ks_hi = pinned ? ks_lo : 16u;
    if (pinned && cdiv(cdiv(p.s.k, 32), ks_lo) * 32u != cdiv(p.steps, ks_lo) * 64u && ks_lo > 1u) return false;
    for (uint32_t t = 0; t < kTiles; ++t) {
        if ((t == T64x64W) != widened || !tile_exists(d.in_type, t)) continue;
        const TileCost& c = fam == kWide ? kFullCost[d.in_type - MAIZE_IN_F32][t] : kTileCost[t];
        const uint64_t tiles = (uint64_t)cdiv(p.s.m, c.bm) * cdiv(p.s.n, c.bn) * p.batch;
        // (a launch counts its work items in 32 bits: fewer than 2^24 workgroups of 256)
        if (tiles >= (1u << 24) || (t == T32x128 && p.s.m > 96u)) continue;
        for (uint32_t ks = ks_lo; ks <= ks_hi; ++ks) {
            // K ranges: of three K tiles or more, none empty, two workgroups per compute unit at most
            if (ks > 1u && (tiles * ks > (pinned ? 8u : 2u) * compute_units || p.steps / ks < 3u || t == T128x128)) break;
            if (ks > 1u && cdiv(p.steps, cdiv(p.steps, ks)) != ks) continue;
            // (16- and 8-bit 128 x 128: from ten K tiles on and 8 % ahead of the others by the model: of 220 products 20 then run on it,
            // 1.19x on average, one of them 3 % slower; without the two conditions up to 30 % slower, 413 deep)
            const bool big = t == T128x128 && fam != kWide;
            if (big && p.steps < 10u) break;
            const double cost = tile_cost(c, p, tiles, ks);
            if (cost < best * (big ? 0.92 : 1.0)) { best = cost; tile = t; ranges = ks; }
        }
    }
    // The form has to win 10 % by the model: of 590 products the choice is then 1.4 % behind the best of all candidates on
    // average, and six are slower than with the registry kernel alone, by 3 to 19 % (none allowed: 1.86x on average, all: 1.855x).
    if (best >= 0.9 * rival) return false;
    // A product that the launcher would cut was compared with its uncut kernel only: it stays cut (4453 x 3712 x 2432 71 us against
    // 79 on the form, 816 x 18448 x 11456 320 against 465, E4M3 1387 x 11200 x 15040 214 against 316).
    if (fam == kMT256 && cdiv64((uint64_t)cdiv(p.s.m, 256) * cdiv(p.s.n, 256), compute_units) > 1u) {
        const TailSplit cut = tail_split(d, compute_units);
        if (cut.rows || cut.cols) return false;
    }
    const TileCost& c = fam == kWide ? kFullCost[d.in_type - MAIZE_IN_F32][tile] : kTileCost[tile];
    const uint64_t items = (uint64_t)cdiv(p.s.m, c.bm) * cdiv(p.s.n, c.bn) * p.batch * ranges;
    out->kernel = (d.in_type * 2u + (p.s.nt ? 1u : 0u)) * kTiles + tile;
    out->grid = (uint32_t)items;
    out->ksplit = ranges;
    out->workspace_bytes = ranges > 1u ? kTicketBytes + (size_t)items * c.bm * c.bn * (p.esz == 8u ? 8u : 4u) : 0u;
    return true;
}

}  // namespace maize
