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
// bounds them is the rate at which a compute unit's requests arrive in its LDS: 75-100 GB/s) and `turn` for each workgroup after the first;
// rows of A (B) that are no 16-byte material make the requests longer by ua (ub), transposing reads by nn, 8-bit
// operands by e8; at least bytes / bw.
struct TileCost { uint32_t bm, bn; double t0, one, many, turn, r0, r1, ua, ub, nn, bw, tail, e8; };
// 128 x 128 has a compute unit to itself and half of the LDS fill per product of 64 x 128: where its tiles make up one round or
// few (129 to 256: 1024 x 3072 x 1999 into bf16 30.1 -> 24.5 us, 4499 x 520 x 3644 51.1 -> 35.8; below, K ranges of smaller tiles
// keep the chip busier).  Fitted to 110 timings of single requests, residuals 7 % where it is a candidate; products whose rows lie off
// 128-byte lines run on requests in pairs now (gemm_tile.hpp), 5 % faster on average and up to 22, for which there is no term.
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
    double bytes, ab_bytes;                  // each operand once; A and B alone
};
double tile_cost(const TileCost& c, const Problem& p, uint64_t tiles, uint32_t ks, double wait = 1.0) {
    const uint32_t per = cdiv(p.steps, ks);
    const double items = (double)(tiles * ks), each = (p.rows_a ? 1.0 : 1.0 + c.ua) * (p.rows_b ? 1.0 : 1.0 + c.ub) * (p.s.nt ? 1.0 : 1.0 + c.nn) * (p.esz == 1u ? 1.0 + c.e8 : 1.0);
    const uint64_t n = cdiv64(tiles * ks, p.cus);
    const double core = wait * (n <= 1u ? per * c.one * each : per * c.many * each * (n > 6u ? items / p.cus : (double)n)) + c.turn * (double)(n - 1u);
    return c.t0 + longer(core, p.bytes / (c.bw * 1e6)) + (p.tail ? c.tail : 0.0) + (ks > 1u ? c.r0 + c.r1 * ks : 0.0);
}
// Operands that the eight L2s (32 MB together) do not hold make a K tile wait longer: core * (their bytes / 32 MB)^0.18, ^0.085 for
// 128 x 128 tiles, which draw half as much (fitted to 3568 timings, up to 2.1 times the model's without).  It decides between a
// form and the registry's kernel (but for few rows, bound by the stream of B either way), not between forms, where it costs as much
// as it gives on some products.
double wait_factor(const TileCost& c, const Problem& p) {
    return p.ab_bytes > 32e6 ? std::pow(p.ab_bytes / 32e6, c.bm == 128u ? 0.085 : 0.18) : 1.0;
}

// The registry's kernels, by what their time depends on.
enum Family : uint32_t { kSkinnyNN, kSkinnyNT, kPacked, kPackedGen, kTransposed, kT128, kH128, kH128Gen, kH128R3, kH128R3Gen, kMT256, kMT256Gen, kH128Split, kMT256Split,
                         kAnyShape, kWide, kUnknown };
struct FamilyOf { Family family; bool whole_m, whole_n; };      // whole_*: a narrow last tile row (column) rides along or is split
FamilyOf family_of(const char* name) {
    const auto has = [&](const char* part) { return std::strstr(name, part) != nullptr; };
    if (has("_mt128_")) return {kWide, false, false};
    if (has("_wave32")) return {kAnyShape, false, false};
    if (has("_skinny_nn")) return {kSkinnyNN, false, false};
    if (has("_skinny_nt")) return {kSkinnyNT, false, false};
    if (has("_packed_gen")) return {kPackedGen, false, false};
    if (has("_packed")) return {kPacked, false, false};
    if (has("_trb")) return {kTransposed, false, false};
    if (has("_t128_")) return {kT128, false, false};
    if (!has("_mt256_")) return {kUnknown, false, false};
    if (has("_splitk")) return {has("_h128") ? kH128Split : kMT256Split, false, false};
    const bool gen = has("_gen");                                    // (the general epilogue)
    if (has("_h128")) return {has("_h128r3") ? (gen ? kH128R3Gen : kH128R3) : gen ? kH128Gen : kH128, false, false};
    return {gen ? kMT256Gen : kMT256, has("_edge") || has("_ragged_m"), has("_edge") || (has("_ragged") && !has("_ragged_m"))};
}
const FamilyOf* families() {
    struct Table {
        FamilyOf of[kMaxKernels];
        Table() { for (uint32_t i = 0; i < kernel_count(); ++i) of[i] = family_of(kernel_at(i).name); }
    };
    static const Table t;
    return t.of;
}
// The time of the call (kernel, copies and reduce pass), microseconds: t0 + rounds (step * K tiles of a range + round) +
// (c + crange * ranges) 10^6 elements of C + range * ranges + mb * MB of A and B + copy * MB copied first.  Fitted to the timings
// of 8630 products (operands cycled): medians of measured over fitted 1.00-1.05, the 5th and 95th percentiles 0.84-0.94 and
// 1.08-1.34.  Rows: 16-bit and 8-bit operands.
struct RegistryCost { uint32_t bm, bn; double t0, step, round, c, range, crange, mb, copy; };
constexpr RegistryCost kRegistryCost[kAnyShape][2] = {
    {}, {},                                                                                                                         // (few rows: below)
    {{256, 256, 10.7, 1.21, 3.45, 0.757, 0.274, 1.33, 0.0, 0.673}, {256, 256, 11.8, 1.21, 5.47, 0.987, 0.141, 0.859, 0.0, 1.34}},   // kPacked
    {{256, 256, 10.3, 1.12, 3.56, 0.427, 0.0, 0.0, 0.0, 0.652}, {256, 256, 11.8, 1.21, 5.47, 0.987, 0.141, 0.859, 0.0, 1.34}},      // kPackedGen
    {{}, {256, 256, 7.86, 1.33, 1.85, 0.536, 0.0, 0.0, 0.0, 0.983}},                                                                // kTransposed
    {{128, 128, 4.09, 0.363, 0.0, 0.56, 0.0, 0.0, 0.037, 0.0}, {128, 128, 4.2, 0.359, 0.0, 0.563, 0.0, 0.0, 0.002, 0.0}},           // kT128
    {{128, 256, 0.0, 0.554, 3.89, 0.348, 0.0, 0.0, 0.104, 0.0}, {}},                                                                // kH128
    {{128, 256, 0.0, 0.765, 4.67, 0.821, 0.0, 0.0, 0.061, 0.0}, {128, 256, 0.0, 0.705, 5.27, 0.74, 0.0, 0.0, 0.009, 0.0}},          // kH128Gen
    {{128, 256, 0.0, 0.633, 0.0, 0.867, 0.0, 0.0, 0.058, 0.0}, {}},                                                                 // kH128R3
    {{128, 256, 0.0, 0.819, 1.33, 1.02, 0.0, 0.0, 0.042, 0.0}, {128, 256, 0.0, 0.724, 1.8, 0.913, 0.0, 0.0, 0.054, 0.0}},           // kH128R3Gen
    {{256, 256, 2.4, 1.29, 3.47, 0.177, 0.0, 0.0, 0.055, 0.0}, {256, 256, 3.36, 1.17, 3.59, 0.192, 0.0, 0.0, 0.055, 0.0}},          // kMT256
    {{256, 256, 3.88, 1.4, 5.23, 0.226, 0.0, 0.0, 0.042, 0.0}, {256, 256, 3.36, 1.17, 3.59, 0.192, 0.0, 0.0, 0.055, 0.0}},          // kMT256Gen
    {{128, 256, 0.0, 0.537, 6.49, 2.16, 0.318, 1.51, 0.076, 0.0}, {128, 256, 0.0, 0.435, 6.93, 2.27, 0.314, 1.62, 0.05, 0.0}},      // kH128Split
    {{256, 256, 6.13, 1.4, 1.59, 1.23, 0.379, 1.06, 0.047, 0.0}, {256, 256, 0.0, 1.4, 5.99, 2.68, 0.0, 0.535, 0.053, 0.0}},         // kMT256Split
};
double registry_cost(const FamilyOf& f, const Problem& p, const LaunchDims& ld) {
    const uint32_t ks = ld.ksplit ? ld.ksplit : 1u;
    if (f.family == kSkinnyNN || f.family == kSkinnyNT) {
        const bool nn = f.family == kSkinnyNN;
        const uint32_t groups = p.s.m <= 16u ? 1u : p.s.m <= 32u ? 2u : 4u;
        const double rounds = (double)cdiv64((uint64_t)cdiv(p.s.n, 256) * p.batch * ks, p.cus);
        const double core = rounds * cdiv(p.steps, ks) * (nn ? 0.44 : 0.85);
        return (nn ? 3.5 : 1.0) + longer(core, p.bytes / (nn ? 6.35e6 : 5.33e6)) + (ks > 1u ? (nn ? 3.8 : 0.0) + (nn ? 0.19 : 0.65) * ks * groups : 0.0);
    }
    // fp32 and fp64 (but for what choose_form keeps), and the any-shape kernel: the form always
    if (f.family == kAnyShape || f.family == kWide) return 1e9;
    if (f.family == kUnknown) return 0.0;                            // (a kernel that this table does not know keeps its products)
    const RegistryCost& c = kRegistryCost[f.family][p.esz == 1u];
    if (c.bm == 0u) return 0.0;
    const auto tiles = [](uint32_t x, uint32_t b, bool whole) { return whole && x > b ? x / b : cdiv(x, b); };
    const double rounds = (double)cdiv64((uint64_t)tiles(p.s.m, c.bm, f.whole_m) * tiles(p.s.n, c.bn, f.whole_n) * p.batch * ks, p.cus);
    const double elems = (double)p.s.m * p.s.n * p.batch * 1e-6, mb = p.batch * 1e-6 * p.esz * p.s.k;
    return c.t0 + rounds * (cdiv(p.steps, ks) * c.step + c.round) + elems * (c.c + c.crange * ks) + c.range * ks +
           mb * (c.mb * ((double)p.s.m + p.s.n) + c.copy * ((ld.pack_a.on ? (double)p.s.m : 0.0) + (ld.pack_b.on ? (double)p.s.n : 0.0)));
}

}  // namespace

uint32_t form_count() { return kTileForms; }
const char* form_name(uint32_t index) {
    const char* n = index < kTileForms ? names().name[index] : "";
    return n[0] ? n : nullptr;
}

bool choose_form(const maize_gemm_ex_desc_t& d, uint32_t registry, uint32_t compute_units, FormPlan* out) {
    const FamilyOf& of = families()[registry];
    const Family fam = of.family;
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
    p.ab_bytes = (double)p.batch * p.esz * ((double)p.s.m + p.s.n) * p.s.k;
    p.bytes = p.ab_bytes + p.batch * c_bytes * p.s.m * p.s.n * (d.beta != 0.0f ? 2.0 : 1.0);

    LaunchDims ld;
    std::memset(&ld, 0, sizeof ld);
    if (!kernel_at(registry).plan(d, compute_units, &ld)) return false;       // (what the registry's kernel refuses stays refused)
    const double rival = registry_cost(of, p, ld);

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
            // 1.19x on average, one of them 3 % slower; without the two conditions up to 30 % slower, 413 deep.  Measured, as the row of
            // kTileCost, with single requests throughout)
            const bool big = t == T128x128 && fam != kWide;
            if (big && p.steps < 10u) break;
            const double cost = tile_cost(c, p, tiles, ks);
            if (cost < best * (big ? 0.92 : 1.0)) { best = cost; tile = t; ranges = ks; }
        }
    }
    const TileCost& c = fam == kWide ? kFullCost[d.in_type - MAIZE_IN_F32][tile] : kTileCost[tile];
    const uint64_t tiles = (uint64_t)cdiv(p.s.m, c.bm) * cdiv(p.s.n, c.bn) * p.batch, items = tiles * ranges;
    // fp32 and fp64: the registry's 128 x 128 tiles through registers take 4.3 (fp64 5.7) times as long on the average of 2000 drawn
    // products.  They keep those that have so short a K and so many tiles that the form's are the same, or nearly, and its ring is
    // mostly prologue, where all rows are 16-byte material (4096 x 15584 x 32 fp64 172.9 -> 143.8 us, 7203 x 17704 x 16 fp32 143.7 ->
    // 120.6).  Of 3945 fp32 products (six tenths with K up to 512) the form is more than 3 % behind on 374 without this rule and
    // on 57 with it; on 34 of the 449 that the rule keeps the registry's kernel is, by 10 % at most.  Of 2055 fp64 ones: 34, 20, 4 of 36.
    if (fam == kWide && ld.split_first == 7u) {
        const uint64_t tiles128 = (uint64_t)cdiv(p.s.m, 128) * cdiv(p.s.n, 128) * p.batch;
        if (d.in_type == MAIZE_IN_F32 ? tile == T128x128 && p.steps <= 4u : p.steps <= 3u && tiles128 >= 8u * compute_units) return false;
    }
    // The form has to win by the model; by 8 % against 128-row tiles and K ranges above 64 rows, by 10 % against the few-row kernels
    // (the shares that left the sum of all times least).  Of 4000 drawn products 3352 then run a form, in 0.47 of the registry
    // kernel's time on average; 42 of them are more than 3 % slower on it, 20 more than 10 %, at most 29 % (with one share of 0.9, and
    // without wait_factor: 68 of all 4000, 41 and 54 %).
    const bool few_rows = fam == kSkinnyNN || fam == kSkinnyNT;
    const bool close = fam == kH128 || fam == kH128Gen || fam == kH128R3 || fam == kH128R3Gen || fam == kH128Split || fam == kMT256Split;
    const double share = few_rows ? 0.9 : close && p.s.m > 64u ? 0.92 : 1.0;
    if (best >= 1e9 || (rival < 1e9 && tile_cost(c, p, tiles, ranges, few_rows ? 1.0 : wait_factor(c, p)) >= share * rival)) return false;
    // A product that the launcher would cut was compared with its uncut kernel only: it stays cut (4453 x 3712 x 2432 71 us against
    // 79 on the form, 816 x 18448 x 11456 320 against 465, E4M3 1387 x 11200 x 15040 214 against 316).
    if ((fam == kMT256 || fam == kMT256Gen) && cdiv64((uint64_t)cdiv(p.s.m, 256) * cdiv(p.s.n, 256), compute_units) > 1u) {
        const TailSplit cut = tail_split(d, compute_units);
        if (cut.rows || cut.cols) return false;
    }
    out->kernel = (d.in_type * 2u + (p.s.nt ? 1u : 0u)) * kTiles + tile;
    out->grid = (uint32_t)items;
    out->ksplit = ranges;
    out->workspace_bytes = ranges > 1u ? kTicketBytes + (size_t)items * c.bm * c.bn * (p.esz == 8u ? 8u : 4u) : 0u;
    return true;
}

}  // namespace maize
