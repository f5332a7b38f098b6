// The ring of gemm_tile.hpp, as statements of its body<>: the first entries' requests, the K loop and the last entries.  PAIR: the
// requests of two K tiles of one operand go out together, a row of the one next to the same row of the other; NS: the
// ring's stages.  A file of statements, included for each ring: as a lambda it changes the code of the fifty-eight forms
// that have one ring only, and costs the E4M3 N x K ones 1 to 2 % (479 x 7047 x 2944 N x K 17.2 -> 17.4 us).
    constexpr uint32_t PRIME = PAIR ? 4u : (uint32_t)NS;
    const uint32_t primed = nd < PRIME ? nd : PRIME;
    if constexpr (PAIR) {
        uint32_t s = 0;
        for (; s + 1u < primed; s += 2u) request_pair(s, s);
        if (s < primed) request(s, s);
    } else {
        for (uint32_t s = 0; s < primed; ++s) request(s, s);
    }
    if (tail_here && nd < (uint32_t)NS) place_tail(nd);
    // Waits until all but the youngest `n` entries' requests of this wave have landed, then for the other waves.
    auto meet = [&](uint32_t n) {
        each<NS>([&](auto n_) {
            constexpr int c = decltype(n_)::value;
            if (n == (uint32_t)c) wait_loads<c * P>();
        });
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    meet(PAIR ? (primed > 2u ? primed - 2u : 0u) : primed ? primed - 1u : 0u);

    // Fragment reads (maps.hpp): one base per K half (K-contiguous tiles; fragment f sits 2048 f bytes further on) or per
    // column group (K x N tile).
    const uint32_t b_lane = FP ? (lane & 48u) | maps::we_column(ES, lane) : lane;      // fp64: the fragment's columns in the order of the results
    uint32_t a_rd[2], b_rd[NT ? 2 : NJ];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) a_rd[kh] = (uint32_t)(uintptr_t)(lds_ptr)lds_a + maps::kc_frag16_offset(wm * (MI * 16u), kh, lane);
    if constexpr (NT) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) b_rd[kh] = (uint32_t)(uintptr_t)(lds_ptr)lds_b + maps::kc_frag16_offset(wn * (NJ * 16u), kh, b_lane);
    } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j) b_rd[j] = (uint32_t)(uintptr_t)(lds_ptr)lds_b + KNB::read(wn * NJ + j, lane);
    }
    // ---- the K loop: a K tile's fragments are read whole, while the MFMAs of the one before run ----------------------------
    // At the top of step s entry s's fragments are in registers (set S = s % 2) for every wave.  Behind the barrier entry s + 1
    // has landed and entry s's stage is free: the requests and the reads of entry s + 1 (set 1 - S) go out behind the MFMAs.
    //   Single requests: step s asks for entry s + NS, into entry s's stage; the wait leaves the entries from s + 2 on in flight.
    //   Pairs: up to s + 3 is asked for at the top of an even step s, and s + 1 has landed.  It asks for A of s + 4 and s + 5, into the
    //   stages of s - 1 and s; step s + 1 asks for B of both, and its wait leaves that A (2 PA requests) in flight: s + 2 and s + 3 have landed.
    //   An entry s + 4 without a partner and the tail behind it are step s's, the first behind the loop.
    // One LDS round trip per step, with one wave per SIMD to hide it: reading K half by K half -- two round
    // trips -- 256 x 256 x 4096 on 16 workgroups took 17.6 us against 16.7 (and 14.4 with no requests past the end).
    // (The waits name every register the reads fill, so that nothing derived from them can move in front.)
    // 4- and 8-byte operands: a lane's 16-byte chunk (row-major B: its CH rows of one column) feeds CH instructions four deep,
    // the same k on both sides.
    constexpr int BR = ET == 6 ? 8 : 4;                               // reads of a fragment of a row-major B
    constexpr int NR = MI * 2 + NJ * (NT ? 2 : BR);                   // reads of a K tile
    constexpr int NM = FP ? 2 * (int)CH * NMF : IS8 ? NMF : 2 * NMF;  // its matrix instructions
    typedef std::conditional_t<ET == 6, uint32_t, u32x2> tr_t;
    constexpr int RPS = (NR + NM - 1) / NM;
    u32x4 fa[2][MI][2], fb[2][NT ? NJ : 1][2];                        // set, fragment, K half (8-bit: the lane's chunks l / 16 and 4 + l / 16)
    tr_t ft[2][NT ? 1 : NJ][BR];                                      // row-major B: set, fragment, 2 (K half) + register half, or CH (K half) + row
    auto read_one = [&](auto set, auto q_, uint32_t ao, uint32_t bo) {
        constexpr int S = decltype(set)::value, q = decltype(q_)::value;
        if constexpr (q < 2 * MI) rd128<(q % MI) * 2048>(fa[S][q % MI][q / MI], a_rd[q / MI] + ao);
        else if constexpr (NT) rd128<((q - 2 * MI) % NJ) * 2048>(fb[S][(q - 2 * MI) % NJ][(q - 2 * MI) / NJ], b_rd[(q - 2 * MI) / NJ] + bo);
        else if constexpr (FP) {
            constexpr int r = q - 2 * MI, f = r % NJ, k = r / NJ;     // K half k / CH, element k % CH
            rd_elem<(k / (int)CH * (int)(BKE / 2u) + k % (int)CH) * (int)KNB::RB>(ft[S][f][k], b_rd[f] + bo);
        } else {
            constexpr int r = q - 2 * MI, f = (r >> 1) % NJ, kh = (r >> 1) / NJ, h = r & 1;
            rd_tr<IS8, kh * KNB::DEEP + h * KNB::HALF>(ft[S][f][2 * kh + h], b_rd[f] + bo);
        }
    };
    auto landed = [&](auto set) {
        constexpr int S = decltype(set)::value;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < MI; ++i) pin(fa[S][i][0], fa[S][i][1]);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (NT) pin(fb[S][j][0], fb[S][j][1]);
            else {
#pragma unroll
                for (int e = 0; e < BR; e += 2) pin(ft[S][j][e], ft[S][j][e + 1]);
            }
        }
    };
    auto b_half = [&](auto set, int j, int kh) -> u32x4 {
        constexpr int S = decltype(set)::value;
        if constexpr (NT) return fb[S][j][kh];
        else if constexpr (FP) return u32x4{0u, 0u, 0u, 0u};
        else return u32x4{ft[S][j][2 * kh][0], ft[S][j][2 * kh][1], ft[S][j][2 * kh + 1][0], ft[S][j][2 * kh + 1][1]};
    };
    // Matrix instruction n of a K tile (B's fragment first: a lane ends up with 4 consecutive columns of one row of C).
    auto multiply = [&](auto set, auto n_) {
        constexpr int S = decltype(set)::value, n = decltype(n_)::value, i = n % NMF / NJ, j = n % NJ;
        if constexpr (FP) {
            // (the compiler's own instruction: it knows these, slower, pipelines' hazards)
            constexpr int k = n / NMF, kh = k / (int)CH, e = k % (int)CH;
            const u32x4 a = fa[S][i][kh];
            if constexpr (ET == 6) {
                const uint32_t av = a[e];                             // (a bit cast of the vector's element itself takes element 0)
                uint32_t bv;
                if constexpr (NT) bv = fb[S][j][kh][e]; else bv = ft[S][j][k];
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, bv), __builtin_bit_cast(float, av), acc[i][j], 0, 0, 0);
            } else {
                u32x2 b;
                if constexpr (NT) b = u32x2{fb[S][j][kh][2 * e], fb[S][j][kh][2 * e + 1]}; else b = ft[S][j][k];
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(__builtin_bit_cast(double, b), __builtin_bit_cast(double, u32x2{a[2 * e], a[2 * e + 1]}), acc[i][j], 0, 0, 0);
            }
        }
        else if constexpr (!IS8) mfma16<F16>(acc[i][j], b_half(set, j, n / NMF), fa[S][i][n / NMF]);
        else if constexpr (!WIDE) mfma8<(ET - 2) & 1, ((ET - 2) >> 1)>(acc[i][j], b_half(set, j, 0), b_half(set, j, 1), fa[S][i][0], fa[S][i][1]);
    };
    uint32_t st = 0u;                                                 // ring stage of the entry in hand
    uint32_t left = 0u;                                               // an entry without a partner is on its way
    auto step = [&](auto set, auto requests, uint32_t s) {            // 2: requests as above; 1: if there is an entry left (or places the tail); 0: there is none
        constexpr int S = decltype(set)::value;
        constexpr int REQ = decltype(requests)::value;
        constexpr std::integral_constant<int, 1 - S> other{};
        if constexpr (PAIR) {
            // (an even step's next entry landed with its own: a barrier only, but behind the last requests, where all are waited for)
            if constexpr (S == 0 && REQ != 0) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else if constexpr (REQ == 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(2 * PA) : "memory");
            else meet(REQ == 1 ? left : 0u);
        }
        else if constexpr (REQ == 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((NS - 2) * P) : "memory");
        else meet(nd < s + 2u ? 0u : nd - s - 2u < (uint32_t)NS - 2u ? nd - s - 2u : (uint32_t)NS - 2u);
        const uint32_t nst = st + 1u == (uint32_t)NS ? 0u : st + 1u, ao = nst * ASTAGE, bo = nst * BSTAGE;
        TileReq r, r2;
        constexpr int RP = !PAIR ? P : S == 0 ? 2 * PA : 2 * PB;      // requests of this step
        const uint32_t pst = st ? st - 1u : (uint32_t)NS - 1u;        // (the stage of entry s - 1 is free, too)
        if constexpr (REQ == 2 && PAIR) {
            if constexpr (S == 0) { r = tile_req(s + 4u, pst); r2 = tile_req(s + 5u, st); }
            else                  { r = tile_req(s + 3u, pst ? pst - 1u : (uint32_t)NS - 1u); r2 = tile_req(s + 4u, pst); }
        }
        else if constexpr (REQ == 2) r = tile_req(s + (uint32_t)NS, st);
        if constexpr (REQ == 1 && PAIR && S == 0) {
            if (s + 4u < nd) { request(s + 4u, pst); left = 1u; }
            if (tail_here && nd >= (uint32_t)NS) place_tail(s + 4u < nd ? st : pst);
        }
        else if constexpr (REQ == 1 && !PAIR) {
            if (s + (uint32_t)NS < nd) request(s + (uint32_t)NS, st);
            else if (tail_here && s + (uint32_t)NS == nd) place_tail(st);
        }
        each<NM>([&](auto n_) {
            constexpr int n = decltype(n_)::value;
            multiply(set, n_);
            each<RPS>([&](auto e_) {
                constexpr int q = n * RPS + decltype(e_)::value;
                if constexpr (q < NR) read_one(other, std::integral_constant<int, q>{}, ao, bo);
            });
            if constexpr (REQ == 2) {
#pragma unroll
                for (int q = n * RP / NM; q < (n + 1) * RP / NM; ++q) {
                    if constexpr (PAIR) piece(q & 1 ? r2 : r, S * PA + q / 2);
                    else piece(r, q);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (WIDE) {
            // eight bytes of a lane (k = 16 g + 64 kh + 8 h + 0..7 on both sides) -> one 32-deep bf16 step
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bf16x8 wa[MI], wb[NJ];
#pragma unroll
                for (int i = 0; i < MI; ++i) wa[i] = widen8<(ET - 2) & 1>(fa[S][i][q >> 1][2 * (q & 1)], fa[S][i][q >> 1][2 * (q & 1) + 1]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const u32x4 b = b_half(set, j, q >> 1);
                    wb[j] = widen8<((ET - 2) >> 1)>(b[2 * (q & 1)], b[2 * (q & 1) + 1]);
                }
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[j], wa[i], acc[i][j], 0, 0, 0);
            }
        }
        landed(other);
        st = nst;
    };
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    constexpr std::integral_constant<int, 2> TWO{};
    each<NR>([&](auto q_) { read_one(S0, q_, 0u, 0u); });
    landed(S0);
    uint32_t s = 0;
    for (; s + (PAIR ? 5u : (uint32_t)NS + 1u) < nd; s += 2u) {
        step(S0, TWO, s);
        step(S1, TWO, s + 1u);
    }
    // The last entries, the tail among them.  Single requests: at most NS + 1 and the tail; one of the first two steps may still have an entry
    // to request or the tail to place.  Pairs: at most five (up to s + 3 are requested) and the tail; the first step requests
    // the fifth and places the tail.
    drain<0, PAIR ? 6 : NS + 2>(s, ns, [&](auto i_, uint32_t e) { step(std::integral_constant<int, decltype(i_)::value & 1>{}, std::integral_constant<int, (decltype(i_)::value < 2)>{}, e); });
