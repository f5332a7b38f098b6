// maize_tile_*: small-tile forms of the pipelined product for any K, N, leading dimension and element-aligned pointer.
//
// The macro-tile kernels want K in whole 16-byte chunks and give every workgroup 128 x 128 elements of C or more.  These
// forms serve what is left: ragged K (a 16-byte chunk that straddles the end of a row in K), rows of C that are no 16-byte
// material, and products so small that 128-wide tiles leave most of the chip idle.  The reference's schedule
// (sm80_gemm_smem_multibuffer, crates/maize_tile/src/gemm/mod.rs:37-90) as in gemm_t128.hpp: a ring of NS LDS stages filled
// by 128-bit direct-to-LDS loads, fragments of one K half read while the other half's MFMAs run, one barrier per K tile.
//
//   * K = main + tail, main a whole number of K tiles (64 16-bit or 128 8-bit elements), which the ring streams without a
//     mask: requests may start on any byte.  The tail -- what is left of K, or the last whole tile where the range check's
//     dword granularity would drop the last elements of a row-major B -- goes through registers: 16-byte loads that end at
//     the row's (matrix's) end at the latest, shifted into place and zero-filled, written to its ring stage in the
//     layout of the others once that stage is free.  So nothing is ever read outside an
//     operand, and neither a copy of the operands nor a mask in the loop is needed;
//   * few tiles and a long K: `ksplit` K ranges per tile, combined inside the kernel -- every workgroup writes its fp32
//     partial tile in fragment order (whole cache lines), and the last to arrive adds them in range order (deterministic).
//     A partial tile is 16 KiB, so that is one short burst of loads, where the 128 KiB ones of the macro-tile kernels need
//     a pass of their own;
//   * C goes through LDS and out in runs of eight columns, whatever its alignment (128-bit stores may start on any element).
//
// What bounds them: the rate at which a compute unit's requests arrive in its LDS, 75-100 GB/s (16, 20 or 24 KiB per K tile: 0.17-0.28
// us with one workgroup per compute unit; 41 of the 64 bytes per cycle of the vector L1), and some 3 us of launch, first loads and
// epilogue.  Counters (1024^3, 544 x 2472 x 1112, E4M3 16 x 14336 x 4096): matrix pipe busy 0.13-0.19 and LDS reads 0.15-0.18 of the
// time, no bank conflicts, waves waiting 0.44-0.57.  Tiles of 64 x 64 move twice the bytes
// of 128 x 128 per multiply-add but give four times the workgroups, two per compute unit at a time: 1024^3 11.2 -> 7.0 us, 256^3
// 6.2 -> 4.5, 200 x 1072 x 368 9.9 -> 5.4; 64 x 128 where there are enough of them: 544 x 2472 x 1112 21.0 -> 11.3, 1632 x 1072 x
// 1392 22.9 -> 12.8; 32 x 128 for few rows.  Ragged K against copies of the operands in the workspace: 1024 x 3072 x 1999 61.4 -> 25.9,
// 3 x 4863 x 4281 48.6 -> 12.1, E4M3 19 x 10987 x 1494 50.1 -> 6.8; against the any-shape kernel: 150 x 201 x 333 26.1 -> 5.9, E4M3
// 128 x 168 x 296 63 -> 5.5.  (Tried and slower: twice the ring depth on one workgroup per compute unit, three stages on three.)
//
// 128 x 128 of 16- and 8-bit operands: what bounds the smaller tiles on a product of a round or two is the LDS fill, which this
// halves per multiply-add.  What bounds it in turn is one wave per SIMD (1024 x 3072 x 1999 into fp32: waits 0.32, waits to issue 0.31,
// matrix pipe 0.31).  One workgroup of four or five ring stages (of 160 KiB) per compute unit: two of two stages have too few
// registers, and the compiler then copies fragments that are still being read.  1024 x 3072 x 1999 accumulated into fp32
// 29.6 -> 25.3 us (424 -> 496 TFLOP/s), 3713 x 554 x 4707 in batches of 3 200 -> 140, E4M3 928 x 2568 x 5992 42.6 -> 32.9.
//
// They ask for the K tiles of an operand in pairs, from five ring stages, where rows do not start on 128-byte lines: a K tile's
// 128 bytes of a row are then on two lines, and the line that two K tiles share is read once if both are asked for together.
// Reads from the L2: 8.57 -> 6.48 million of 1700 x 2000 x 4999 N x K, E4M3 928 x 2568 x 5992 3.69 -> 2.86, 1192 x 2580 x
// 1856 (rows on lines) 1.474 both.  Single requests from four stages -> pairs: 1700 x 2000 x 4999 57.1 -> 52.0 us (595 ->
// 654 TFLOP/s), E4M3 928 x 2568 x 5992 35.4 -> 29.1, 1024 x 3072 x 1999 K x N into fp32 25.4 -> 24.6, 96 drawn products 5 % off on
// average and none longer.  Rows that do not start on dwords gain nothing (E4M3 1024 x 3072 x 1999 N x K 21.3 both): a request there is
// about four accesses of the vector cache, and pairs leave their number as it is (22.0 million; L2 reads 1.65 -> 1.31).
// Rows on lines share nothing, and B is asked for one step later: 32 drawn products 2 % longer on average, 7 % at most (1192 x
// 2580 x 1856 N x K 18.1 -> 19.1, E5M2 5176 x 2006 x 4096 51.2 -> 53.8, 1536 x 2203 x 4096 K x N 36.9 -> 38.2).  They have single requests and
// four stages (with five, a K tile more stands in front of the first multiplication: 1 to 5 % longer as well); so have N x K products with one
// operand on lines and one on half lines, which gain and lose 4 %.  One operand on lines and one anywhere: 1 to 5 % off on average, 2 %
// longer at most; both on half lines, or A against a row-major B: 3 % off, 3 % longer at most.  The kernel looks at its operands
// (maps::in_pairs), and what stands around the ring is there once: a body for each ring cost 1 % (1024 x 3072 x 1999 into fp32 24.6 -> 24.85 us).
// Not the 64 x 64 tiles, which have five stages too but less to multiply behind their loads: four K
// tiles in flight instead of five cost half 16 x 14336 x 4096 N x K 24.7 -> 30.8 us, 1024^3 6.8 -> 7.4 and E4M3 19 x 10987 x
// 1494 6.7 -> 6.9 (and gave 150 x 201 x 333 5.95 -> 5.43).
//
// fp32 and fp64 operands (v_mfma_f32_16x16x4_f32, v_mfma_f64_16x16x4_f64; no tf32 instruction exists): the same ring and tiles.
// What bounds them is the matrix pipe (busy 0.97 and 0.95 of the time at 4096^3): a K tile of 128 bytes of a 64 x 64 tile is 1024 of its cycles against 16 KiB of LDS fill.
// A lane's 16-byte chunk feeds four (two) instructions in turn, the same k on both sides, so a K-contiguous operand needs an
// eighth of the reads of one element per instruction, and the next K tile's reads run behind this one's instructions.  Against
// 128 x 128 tiles copied through registers, whose reads stand in front of the instructions they feed: 2048^3 fp32 N x K 162.6 ->
// 129.1 us (0.85 of the pipe), 4096^3 1040 -> 924 (0.95), 4096^3 fp64 2107 -> 1882 (0.93); and where 128-wide tiles leave the
// chip idle: 1024^3 fp64 149 -> 42, 8 x 7336 x 4464 fp32 and its like 3 to 10 times.
#pragma once
#include <type_traits>
#include "common.hpp"
#include "grid.hpp"
#include "maps.hpp"

namespace maize {
namespace tile {

using mt256::lds_ptr;
using mt256::make_rsrc;
using mt256::OOB;

template <int N, int I = 0, class F>
__device__ __forceinline__ void each(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        each<N, I + 1>(static_cast<F&&>(f));
    }
}

// Fragment reads (assembly statements, which keep their order: the compiler does not know when a direct-to-LDS load has landed).
template <int OFF, class T> __device__ __forceinline__ void rd128(T& dst, uint32_t base) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "n"(OFF)); }
template <bool IS8, int OFF> __device__ __forceinline__ void rd_tr(u32x2& dst, uint32_t base) {
    if constexpr (IS8) asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "n"(OFF));
    else               asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "n"(OFF));
}
// (the accumulator is tied to itself and stays where it is)
template <bool F16> __device__ __forceinline__ void mfma16(floatx4& c, u32x4 b, u32x4 a) {
    if constexpr (F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a));
    else               asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a));
}
// One element of a row-major 4- or 8-byte B.
template <int OFF> __device__ __forceinline__ void rd_elem(uint32_t& dst, uint32_t base) { asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "n"(OFF)); }
template <int OFF> __device__ __forceinline__ void rd_elem(u32x2& dst, uint32_t base) { asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(base), "n"(OFF)); }
// (B first, so cbsz carries B's format and blgp A's: 0 = E4M3, 1 = E5M2)
template <int A_E5M2, int B_E5M2> __device__ __forceinline__ void mfma8(floatx4& c, u32x4 b0, u32x4 b1, u32x4 a0, u32x4 a1) {
    typedef int i32x8 __attribute__((ext_vector_type(8)));
    const i32x8 b = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
    const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:%3 blgp:%4" : "+a"(c) : "v"(b), "v"(a), "n"(B_E5M2), "n"(A_E5M2));
}
// Tile `id` of the grid in sweeps of GM tile rows (grid.hpp, tile_of): the 32 or 64 tiles an XCD works on at a time make up a
// square of C, so that the operand panels its L2 draws are the fewest.
template <int BM, int BN>
__device__ __forceinline__ void place(uint32_t id, uint32_t tm, uint32_t tn, uint32_t* tile_m, uint32_t* tile_n) {
    constexpr uint32_t GM = 8;
    if (tm == 1u) { *tile_m = 0u; *tile_n = id; return; }
    const uint32_t group = id / (GM * tn), first = group * GM, in = id - group * (GM * tn), left = tm - first;
    if (left >= GM) { *tile_m = first + in % GM; *tile_n = in / GM; }
    else { *tile_n = in / left; *tile_m = first + in - *tile_n * left; }
}
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }
template <class T> __device__ __forceinline__ void pin(T& a, T& b) { asm volatile("" : "+v"(a), "+v"(b)); }

// f(I, s), f(I + 1, s + 1), ... while s < ns, at most N of them.
template <int I, int N, class F>
__device__ __forceinline__ void drain(uint32_t s, uint32_t ns, F&& f) {
    if constexpr (I < N) {
        if (s < ns) {
            f(std::integral_constant<int, I>{}, s);
            drain<I + 1, N>(s + 1u, ns, static_cast<F&&>(f));
        }
    }
}

// The layout of a row-major (K x N) B tile BN columns wide (maps.hpp): 128 / ES rows of elements of ES bytes.
template <uint32_t ES, int BN>
struct KN {
    static constexpr bool IS8 = ES == 1u;
    static constexpr uint32_t RB = BN * ES;                           // bytes per row
    static constexpr int HALF = BN * (IS8 ? 8 : 8);                   // register half h: 8 rows of 8-bit, 4 rows of 16-bit elements
    static constexpr int DEEP = BN * 64;                              // K half: 64 rows of 8-bit, 32 rows of 16-bit elements
    static __device__ __forceinline__ uint32_t row(uint32_t piece, uint32_t lane) {
        if constexpr (ES >= 4u) return maps::we_piece_row(RB, piece, lane);
        else if constexpr (IS8) return BN == 128 ? maps::sk8n_piece_row(piece, lane) : maps::sk8s_piece_row(piece, lane);
        else               return BN == 128 ? maps::sk128_piece_row(piece, lane) : maps::sk64_piece_row(piece, lane);
    }
    static __device__ __forceinline__ uint32_t chunk(uint32_t piece, uint32_t lane) {
        if constexpr (ES >= 4u) return maps::we_piece_chunk(ES, RB, piece, lane);
        else if constexpr (IS8) return BN == 128 ? maps::sk8n_piece_chunk(piece, lane) : maps::sk8s_piece_chunk(piece, lane);
        else               return BN == 128 ? maps::sk128_piece_chunk(piece, lane) : maps::sk64_piece_chunk(piece, lane);
    }
    static __device__ __forceinline__ uint32_t read(uint32_t cg, uint32_t lane) {
        if constexpr (ES >= 4u) return maps::we_read(ES, RB, cg, lane);
        else if constexpr (IS8) return BN == 128 ? maps::sk8n_tr_offset(cg, 0, 0, lane) : maps::sk8s_tr_offset(cg, 0, 0, lane);
        else               return BN == 128 ? maps::sk128_tr_offset(cg, 0, lane) : maps::sk64_tr_offset(cg, 0, lane);
    }
};

// A 128-bit value moved `bytes` bytes towards its low end, zeros behind (16 and more: all zeros).
__device__ __forceinline__ u32x4 drop_low(u32x4 v, uint32_t bytes) {
    uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    if (bytes & 8u) { lo = hi; hi = 0; }
    const uint32_t s = (bytes & 7u) * 8u;
    if (s) { lo = (lo >> s) | (hi << (64u - s)); hi >>= s; }
    if (bytes >= 16u) { lo = 0; hi = 0; }
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}
__device__ __forceinline__ u32x4 load16(const char* p) { u32x4 v; __builtin_memcpy(&v, p, 16); return v; }   // any alignment

// The first `count` of eight consecutive elements of a row of C, from element `at` on, whatever its alignment: the epilogue
// of common.hpp.
__device__ __forceinline__ void store_c8(const GemmArgs& p, void* c, uint64_t at, floatx4 lo, floatx4 hi, uint32_t count) {
    float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if (count < 8u) { store_c_elems<8>(p, c, at, x, count); return; }
    const bool f32_out = p.epi & EPI_F32, half_c = c_is_half(p.epi);
    if (p.epi & EPI_SCALE) {
        float old[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (p.beta != 0.0f) {
            if (f32_out) {
                __builtin_memcpy(old, (const float*)c + at, 32);
            } else {
                uint32_t w[4];
                __builtin_memcpy(w, (const uint16_t*)c + at, 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t h = (w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
                    old[e] = half_c ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = epi_scale(x[e], old[e], p.alpha, p.beta);
    }
    if (f32_out) {
        __builtin_memcpy((float*)c + at, x, 32);
    } else {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = half_c ? cvt_pk_f16(x[2 * e], x[2 * e + 1]) : cvt_pk_bf16(x[2 * e], x[2 * e + 1]);
        __builtin_memcpy((uint16_t*)c + at, w, 16);
    }
}

// fp32 and fp64 C: the 16 bytes of a row of C from element `at` on (the first `count` elements), C = alpha * A.B + beta * C in
// the operands' type.
template <class T>
__device__ __forceinline__ void store_c16(const GemmArgs& p, T* c, uint64_t at, u32x4 v, uint32_t count) {
    constexpr uint32_t CH = 16u / sizeof(T);
    const T alpha = (T)p.alpha, beta = (T)p.beta;
    const bool whole = count >= CH;
    T x[CH], old[CH];
    __builtin_memcpy(x, &v, 16);
    if (p.epi & EPI_SCALE) {
#pragma unroll
        for (uint32_t e = 0; e < CH; ++e) old[e] = (T)0;
        if (beta != (T)0) {
            if (whole) __builtin_memcpy(old, c + at, 16);
            else {
#pragma unroll
                for (uint32_t e = 0; e < CH; ++e) if (e < count) old[e] = c[at + e];
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < CH; ++e) {
            if constexpr (sizeof(T) == 4) x[e] = __builtin_fmaf(beta, old[e], alpha * x[e]);
            else                          x[e] = __builtin_fma(beta, old[e], alpha * x[e]);
        }
    }
    if (whole) __builtin_memcpy(c + at, x, 16);
    else {
#pragma unroll
        for (uint32_t e = 0; e < CH; ++e) if (e < count) c[at + e] = x[e];
    }
}

// Eight E4M3 (E5M2) values as bf16 (exact: bf16 holds every value of both formats).
template <int E5M2>
__device__ __forceinline__ bf16x8 widen8(uint32_t lo, uint32_t hi) {
    bf16x2 w[4];
    if constexpr (E5M2) {
        w[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(lo, 1.0f, false); w[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(lo, 1.0f, true);
        w[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(hi, 1.0f, false); w[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(hi, 1.0f, true);
    } else {
        w[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false); w[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
        w[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false); w[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    }
    return bf16x8{w[0][0], w[0][1], w[1][0], w[1][1], w[2][0], w[2][1], w[3][0], w[3][1]};
}

// ET: 0 bf16, 1 IEEE half, 2 + (A is E5M2) + 2 (B is E5M2): 8-bit operands, 6 fp32, 7 fp64.
// WIDE: 8-bit operands widened to bf16 as their fragments are read (exact) and multiplied by the bf16 instruction: the
// arithmetic of the any-shape kernel, which small 8-bit products get.
// 4 waves as WM x WN, each MI x NJ accumulators of 16 x 16; RING stages.
// BY_LINES: requests in pairs where rows share lines between K tiles, else single ones and a stage less (above).
template <int ET, bool WIDE, bool NT, int BM, int BN, int RING, bool BY_LINES>
__device__ __forceinline__ void body(const GemmArgs& p) {
    constexpr bool IS8 = ET >= 2 && ET < 6, F16 = ET == 1, FP = ET >= 6;
    static_assert(!WIDE || IS8, "only 8-bit operands are widened");
    constexpr uint32_t ES = IS8 ? 1u : ET == 6 ? 4u : ET == 7 ? 8u : 2u, CH = 16u / ES, BKE = 128u / ES;
    constexpr uint32_t AS = ET == 7 ? 8u : 4u;                        // bytes of an accumulator
    typedef std::conditional_t<ET == 7, double, float> acc_t;
    typedef acc_t accx4 __attribute__((ext_vector_type(4)));
    constexpr int WN = BM == 32 ? 4 : 2, WM = 4 / WN;
    constexpr int MI = BM / WM / 16, NJ = BN / WN / 16, NMF = MI * NJ;
    constexpr int PA = BM / 32, PB = BN / 32, P = PA + PB;            // 1 KiB requests per wave and K tile
    constexpr uint32_t ASTAGE = BM * 128u, BSTAGE = BN * 128u;
    typedef KN<ES, BN> KNB;
    static_assert(!BY_LINES || (RING == 5 && !FP), "two stages are free in every other step of a ring of five");
    static_assert(RING * (BM + BN) * 128u >= BM * BN * AS, "the epilogue's fp32 tile takes the ring's place");
    __shared__ __attribute__((aligned(1024))) char lds_a[RING * (ASTAGE + BSTAGE)];
    char* const lds_b = lds_a + RING * ASTAGE;
    typedef __attribute__((address_space(3))) void* lvp;

    const uint32_t M = p.crows, N = p.ccols, K = p.acols;
    const uint32_t lda = lda_of(p), ldb = ldb_of(p), ldc = ldc_of(p);
    // (here, where the arguments are waited for anyway, and not in front of the first request)
    const auto off = [&](const void* x, uint32_t ld, uint64_t stride) { return maps::off_lines((uint64_t)(uintptr_t)x, ld * ES, p.batch > 1u ? stride * ES : 0u); };
    const bool pairs = BY_LINES && maps::in_pairs(NT, off(p.a, lda, p.stride_a), off(p.b, ldb, p.stride_b));
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t wm = wave / WN, wn = wave % WN;
    const uint32_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN, tiles_per = tm * tn;
    const uint32_t ks = p.ksplit ? p.ksplit : 1u, total = tiles_per * p.batch * ks;
    if (blockIdx.x >= total) return;
    // (divisions that most launches do not need are branched around: each is some forty dependent instructions in front of
    // the first request)
    const uint32_t item = mt256::xcd_run(blockIdx.x, total);
    uint32_t t = item, z = 0u, bz = 0u;
    if (ks > 1u) { t = item / ks; z = item - t * ks; }
    if (p.batch > 1u) bz = t / tiles_per;
    uint32_t tile_m, tile_n;
    place<BM, BN>(t - bz * tiles_per, tm, tn, &tile_m, &tile_n);
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;

    // K tiles of this item: [s0, s0 + ns) of the list, the main tiles in order and the tail, if there is one, behind them (the
    // order of the other kernels' sums); `nd` of them come by direct-to-LDS loads.
    uint32_t tail = K % BKE;
    if (tail == 0u && !NT && (N * ES & 3u)) tail = BKE;               // the last dword of a row-major B straddles its end
    const uint32_t k_main = K - tail, listed = k_main / BKE + (tail ? 1u : 0u), per = (listed + ks - 1u) / ks, s0 = z * per;
    const uint32_t ns = s0 < listed ? (listed - s0 < per ? listed - s0 : per) : 0u;
    const bool tail_here = tail != 0u && ns != 0u && s0 + ns == listed;
    const uint32_t k_first = s0 * BKE, nd = ns - (tail_here ? 1u : 0u);

    auto span = [](uint64_t bytes) { return (uint32_t)(bytes < 0x7FFFFFFFull ? bytes : 0x7FFFFFFFull); };
    auto sc = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane(x); };
    // Descriptors start at the tile's first row and end with the operand's view: rows at or past M (N) read as zeros.
    const char* const Ab = (const char*)p.a + (uint64_t)bz * p.stride_a * ES;
    const char* const Bb = (const char*)p.b + (uint64_t)bz * p.stride_b * ES;
    const char* const Ag = Ab + (uint64_t)m0 * lda * ES;
    const uint32_t a_bytes = span(((uint64_t)(M - 1u - m0) * lda + K) * ES);
    const char* const Bg = NT ? Bb + (uint64_t)n0 * ldb * ES : Bb;
    const uint32_t b_bytes = NT ? span(((uint64_t)(N - 1u - n0) * ldb + K) * ES) : 0u;
    const uint64_t b_view = ((uint64_t)(K - 1u) * ldb + N) * ES;
    uint32_t a_vo[PA], b_vo[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const uint32_t pc = wave * PA + i;
        a_vo[i] = (maps::kc_piece_row(pc, lane) * lda + maps::kc_piece_chunk(pc, lane) * CH) * ES;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const uint32_t pc = wave * PB + i;
        if (NT) {
            b_vo[i] = (maps::kc_piece_row(pc, lane) * ldb + maps::kc_piece_chunk(pc, lane) * CH) * ES;
        } else {
            const uint32_t col = n0 + KNB::chunk(pc, lane) * CH;
            b_vo[i] = ((KNB::row(pc, lane) * ldb + col) * ES) | (col < N ? 0u : OOB);
        }
    }
    const uint32_t lds_a0 = sc((uint32_t)(uintptr_t)(lds_ptr)lds_a + wave_u * (PA * 1024u));
    const uint32_t lds_b0 = sc((uint32_t)(uintptr_t)(lds_ptr)lds_b + wave_u * (PB * 1024u));
    struct TileReq { __amdgpu_buffer_rsrc_t ra, rb; uint32_t a_so, b_so, la, lb; };
    auto tile_req = [&](uint32_t s, uint32_t st) {                    // list entry s0 + s (one of this item's) into ring stage st
        TileReq r;
        const uint32_t k = k_first + s * BKE;
        r.ra = make_rsrc(Ag, a_bytes);
        r.a_so = sc(k * ES);
        if (NT) {
            r.rb = make_rsrc(Bg, b_bytes);
            r.b_so = r.a_so;
        } else {
            const uint64_t skip = (uint64_t)sc(k) * sc(ldb * ES), base = (uint64_t)(uintptr_t)Bg + skip;
            r.rb = make_rsrc((const void*)(uintptr_t)(((uint64_t)sc((uint32_t)(base >> 32)) << 32) | sc((uint32_t)base)), sc(span(b_view - skip)));
            r.b_so = 0u;
        }
        r.la = sc(st * ASTAGE);
        r.lb = sc(st * BSTAGE);
        return r;
    };
    auto piece = [&](const TileReq& r, int q) {
        if (q < PA) __builtin_amdgcn_raw_ptr_buffer_load_lds(r.ra, (lvp)(uintptr_t)(lds_a0 + r.la + q * 1024u), 16, a_vo[q], r.a_so, 0, 0);
        else        __builtin_amdgcn_raw_ptr_buffer_load_lds(r.rb, (lvp)(uintptr_t)(lds_b0 + r.lb + (q - PA) * 1024u), 16, b_vo[q - PA], r.b_so, 0, 0);
    };
    auto request = [&](uint32_t s, uint32_t st) {
        const TileReq r = tile_req(s, st);
#pragma unroll
        for (int q = 0; q < P; ++q) piece(r, q);
    };
    auto request_pair = [&](uint32_t s, uint32_t st) {                // entries s and s + 1 into stages st and st + 1
        const TileReq r = tile_req(s, st), r2 = tile_req(s + 1u, st + 1u);
#pragma unroll
        for (int q = 0; q < P; ++q) { piece(r, q); piece(r2, q); }
    };

    accx4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = accx4{0, 0, 0, 0};

    // ---- the tail's loads, then the ring's first entries: NS, or four in two pairs -------------------------------------
    // (128 x 128 fp32: when they are placed, two workgroups per compute unit leave no registers to hold them through the loop)
    constexpr bool LATE_TAIL = FP && BM * BN > 64 * 128;
    u32x4 ta[PA], tb[PB];
    auto load_tail = [&] {
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            const uint32_t pc = wave * PA + i, k = k_main + maps::kc_piece_chunk(pc, lane) * CH, row = m0 + maps::kc_piece_row(pc, lane);
            ta[i] = load16(Ab + ((uint64_t)(row < M ? row : M - 1u) * lda + (k < K - CH ? k : K - CH)) * ES);
        }
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const uint32_t pc = wave * PB + i;
            if (NT) {
                const uint32_t k = k_main + maps::kc_piece_chunk(pc, lane) * CH, row = n0 + maps::kc_piece_row(pc, lane);
                tb[i] = load16(Bb + ((uint64_t)(row < N ? row : N - 1u) * ldb + (k < K - CH ? k : K - CH)) * ES);
            } else {
                const uint32_t k = k_main + KNB::row(pc, lane), col = n0 + KNB::chunk(pc, lane) * CH;
                tb[i] = load16(Bb + ((uint64_t)(k < K ? k : K - 1u) * ldb + (col < N - CH ? col : N - CH)) * ES);
            }
        }
    };
    if (tail_here && !LATE_TAIL) load_tail();
    // ... into ring stage st: a chunk that would have run past the end was loaded from further in front and moves down; K past
    // the end is zero.
    auto place_tail = [&](uint32_t st) {
        if constexpr (LATE_TAIL) load_tail();
        auto put = [&](uint32_t at, u32x4 v, uint32_t want, uint32_t last, bool live) {
            asm volatile("ds_write_b128 %0, %1" :: "v"(at), "v"(drop_low(v, live ? (want > last ? want - last : 0u) * ES : 16u)) : "memory");
        };
#pragma unroll
        for (int i = 0; i < PA; ++i)
            put(lds_a0 + st * ASTAGE + i * 1024u + lane * 16u, ta[i], k_main + maps::kc_piece_chunk(wave * PA + i, lane) * CH, K - CH, true);
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const uint32_t pc = wave * PB + i, at = lds_b0 + st * BSTAGE + i * 1024u + lane * 16u;
            if (NT) put(at, tb[i], k_main + maps::kc_piece_chunk(pc, lane) * CH, K - CH, true);
            else    put(at, tb[i], n0 + KNB::chunk(pc, lane) * CH, N - CH, k_main + KNB::row(pc, lane) < K);
        }
    };
    // ---- the ring (gemm_tile_ring.hpp): from the first entries' requests to the last matrix instruction -----------------------
    if constexpr (!BY_LINES) {
        constexpr bool PAIR = false;
        constexpr int NS = RING;
#include "gemm_tile_ring.hpp"
    } else if (pairs) {
        constexpr bool PAIR = true;
        constexpr int NS = RING;
#include "gemm_tile_ring.hpp"
    } else {
        constexpr bool PAIR = false;
        constexpr int NS = RING - 1;
#include "gemm_tile_ring.hpp"
    }
    // nothing may land any more, and the last MFMAs have left the pipe (assembly: invisible to the hazard recognizer)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 7\n\ts_nop 7" ::: "memory");

    // ---- K ranges: the last to arrive adds the partial tiles in range order -----------------------------------
    if (ks > 1u) {
        constexpr int COHERENT = 17;                                  // sc0 | sc1: these accesses cross the per-XCD L2s
        constexpr uint32_t PART = BM * BN * AS;
        constexpr int AW = AS / 4;                                    // 16-byte words of an accumulator
        constexpr int ZG = (NMF <= 4 ? 8 : 2) / AW;                   // ranges whose loads are in flight at a time
        struct Words { u32x4 w[AW]; };
        uint32_t* const counters = (uint32_t*)p.workspace;            // zero between launches
        const __amdgpu_buffer_rsrc_t rws = make_rsrc((const char*)p.workspace + 65536, total * PART);
        const uint32_t mine = item * PART + tid * 16u, first = t * ks * PART + tid * 16u;
#pragma unroll
        for (int q = 0; q < NMF; ++q) {
            const Words x = __builtin_bit_cast(Words, acc[q / NJ][q % NJ]);
#pragma unroll
            for (int h = 0; h < AW; ++h) __builtin_amdgcn_raw_buffer_store_b128(x.w[h], rws, mine + (q * AW + h) * 4096u, 0, COHERENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // this wave's part has reached memory
        volatile uint32_t* const ticket = (volatile uint32_t*)lds_a;   // (the ring is idle: a word of its own would cost the second workgroup of the compute unit)
        __syncthreads();
        if (tid == 0) *ticket = __hip_atomic_fetch_add(&counters[t], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*ticket != ks - 1u) return;
        for (uint32_t z0 = 0; z0 < ks; z0 += ZG) {
            accx4 part[ZG][NMF];
#pragma unroll
            for (int u = 0; u < ZG; ++u)
#pragma unroll
                for (int q = 0; q < NMF; ++q) {
                    Words x;
#pragma unroll
                    for (int h = 0; h < AW; ++h)
                        x.w[h] = __builtin_amdgcn_raw_buffer_load_b128(rws, z0 + u < ks ? first + (z0 + u) * PART + (q * AW + h) * 4096u : 0xFFFFFFF0u, 0, COHERENT);
                    part[u][q] = __builtin_bit_cast(accx4, x);
                }
#pragma unroll
            for (int u = 0; u < ZG; ++u)
#pragma unroll
                for (int q = 0; q < NMF; ++q) {
                    if (z0 + u == 0u) acc[q / NJ][q % NJ] = part[u][q];
                    else if (z0 + u < ks) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[q / NJ][q % NJ][e] += part[u][q][e];
                    }
                }
        }
        if (tid == 0) counters[t] = 0u;                               // ready for the next launch
    }

    // ---- C through LDS: the fp32 tile row by row (16-byte chunks XOR-ed with the row), then runs of 8 columns, whole rows of
    // the tile by neighbouring lanes.  A loop, not one copy of the epilogue per fragment: at these sizes a workgroup runs the
    // code once, and fetching it is what a long one costs.
    lds_ptr const ew = (lds_ptr)lds_a;
    __syncthreads();                                                  // (every wave's requests have landed, the ticket has been read)
    // (an fp64 accumulator is two chunks)
    constexpr uint32_t CW = AS / 4u;
    {
        const uint32_t l16 = lane & 15u, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint32_t row = (wm * MI + i) * 16u + l16, chunk = ((wn * NJ + j) * 4u + g) * CW;
                struct Words { u32x4 w[CW]; };
                const Words x = __builtin_bit_cast(Words, acc[i][j]);
#pragma unroll
                for (uint32_t h = 0; h < CW; ++h)
                    *(__attribute__((address_space(3))) u32x4*)(ew + row * (BN * AS) + (((chunk + h) ^ l16) * 16u)) = x.w[h];
            }
    }
    __syncthreads();
    if constexpr (FP) {
        acc_t* const Ct = (acc_t*)p.c + (uint64_t)bz * p.stride_c;
#pragma unroll 1
        for (uint32_t r = tid; r < BM * BN / CH; r += 256u) {
            const uint32_t row = r / (BN / CH), c = r % (BN / CH), grow = m0 + row, gcol = n0 + c * CH;
            if (grow >= M || gcol >= N) continue;
            store_c16<acc_t>(p, Ct, (uint64_t)grow * ldc + gcol, *(__attribute__((address_space(3))) u32x4*)(ew + row * (BN * AS) + (c ^ (row & 15u)) * 16u), N - gcol);
        }
        return;
    }
    void* const Cg = (char*)p.c + (uint64_t)bz * p.stride_c * ((p.epi & EPI_F32) ? 4u : 2u);
#pragma unroll 1
    for (uint32_t r = tid; r < BM * BN / 8u; r += 256u) {
        const uint32_t row = r / (BN / 8u), c = r % (BN / 8u), grow = m0 + row, gcol = n0 + c * 8u;
        if (grow >= M || gcol >= N) continue;
        const lds_ptr at = ew + row * (BN * 4u);
        const floatx4 lo = *(__attribute__((address_space(3))) floatx4*)(at + ((2u * c) ^ (row & 15u)) * 16u);
        const floatx4 hi = *(__attribute__((address_space(3))) floatx4*)(at + ((2u * c + 1u) ^ (row & 15u)) * 16u);
        store_c8(p, Cg, (uint64_t)grow * ldc + gcol, lo, hi, N - gcol);
    }
}

}  // namespace tile

#define MAIZE_TILE(name, et, wide, nt, bm, bn, ns, perc) \
    extern "C" __global__ __launch_bounds__(256, perc) void name(GemmArgs p) { tile::body<et, wide, nt, bm, bn, ns, false>(p); }
#define MAIZE_TILE_BY_LINES(name, et, nt) \
    extern "C" __global__ __launch_bounds__(256, 1) void name(GemmArgs p) { tile::body<et, false, nt, 128, 128, 5, true>(p); }
#define MAIZE_TILE_16(tag, et) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x64, et, false, false, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x64, et, false, true, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_32x128, et, false, false, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_32x128, et, false, true, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x128, et, false, false, 64, 128, 3, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x128, et, false, true, 64, 128, 3, 2) \
    MAIZE_TILE_BY_LINES(maize_tile_##tag##_nn_128x128, et, false) \
    MAIZE_TILE_BY_LINES(maize_tile_##tag##_nt_128x128, et, true)
MAIZE_TILE_16(bf16, 0)
MAIZE_TILE_16(f16, 1)
#define MAIZE_TILE_8(tag, et) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x64, et, false, false, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x64, et, false, true, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x64w, et, true, false, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x64w, et, true, true, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_32x128, et, false, false, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_32x128, et, false, true, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x128, et, false, false, 64, 128, 3, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x128, et, false, true, 64, 128, 3, 2) \
    MAIZE_TILE_BY_LINES(maize_tile_##tag##_nn_128x128, et, false) \
    MAIZE_TILE_BY_LINES(maize_tile_##tag##_nt_128x128, et, true)
MAIZE_TILE_8(e4m3, 2)
MAIZE_TILE_8(e5m2, 5)
MAIZE_TILE_8(e4m3e5m2, 4)
MAIZE_TILE_8(e5m2e4m3, 3)
#define MAIZE_TILE_FP(tag, et) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x64, et, false, false, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x64, et, false, true, 64, 64, 5, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_32x128, et, false, false, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_32x128, et, false, true, 32, 128, 4, 2) \
    MAIZE_TILE(maize_tile_##tag##_nn_64x128, et, false, false, 64, 128, 3, 2) \
    MAIZE_TILE(maize_tile_##tag##_nt_64x128, et, false, true, 64, 128, 3, 2)
MAIZE_TILE_FP(f32, 6)
MAIZE_TILE_FP(f64, 7)
MAIZE_TILE(maize_tile_f32_nn_128x128, 6, false, false, 128, 128, 2, 2)
MAIZE_TILE(maize_tile_f32_nt_128x128, 6, false, true, 128, 128, 2, 2)
#undef MAIZE_TILE_16
#undef MAIZE_TILE_8
#undef MAIZE_TILE_FP
#undef MAIZE_TILE_BY_LINES
#undef MAIZE_TILE

}  // namespace maize
