// int4 dense tiles on fp16 MFMA (included by moe_tiles.hip after TileArgs): calls with many tokens per expert.
#pragma once

// A 4-wave block owns 128 rows of one expert (per projection) and one pass of up to BM of its tokens, NT tiles of M;
// wave w takes 32 of the rows for all the pass's tokens, so each weight is decoded once per pass. Per 128-input slice
// the tokens' activations (x16 / h16, fp16) come into LDS by DMA and the wave's weight records into registers, both one
// slice ahead in two buffers; one wait and one barrier per slice.
// Token-major product D[token, row]: A = activations, B = weights. M = 32: v_mfma_f32_32x32x16_f16, 8 steps of 16 inputs
// per slice; M = 16: v_mfma_f32_16x16x32_f16, 4 steps of 32 inputs, two B tiles per 32 rows. Lane (n, g), n = lane mod M
// its row, g = lane / M, decodes the step's word of its row from the 16-byte pieces of the tile records that it loaded
// (M = 32: lane groups 2 g and 2 g + 1 of its row's 16-row record; M = 16: lane group g), and reads the same 8 inputs of
// token n from LDS: piece p of token m lies at position p ^ (m & 15) of its 256-byte row, so the reads hit distinct banks.
// The decode (11 VALU per word) and LDS reads of step j + 1 are placed between the MFMAs of step j
// (sched_group_barrier); loads use buffer addressing (scalar base and slice offset, one 32-bit offset per lane: the 64-bit
// address pairs of flat loads spilled). They take 167 (M = 32: three blocks per CU) and 209 registers.
// Bound: decode and MFMA issue, then the chip's power: MFMAs alone on random data run at ~1.65 PFLOP/s here (1.6 GHz),
// with 24 VALU per 128 MFMA cycles at ~1.5. Gate/up kernel, against the kernel before (16 x 16 tiles at 2 blocks per CU,
// libm GLU, decode between whole steps): Mixtral T = 512 354 -> 294 us (820 TFLOP/s), Qwen3 T = 4096 320 -> 260.
//
// EX (gate/up): products on exact weights, for loads where the wave tiles' exact codes were used before. The decode
// takes s (q - 8) instead of s q + b: 8 + 3 significant bits, which fp16 holds exactly (below the subnormal line of the
// row scaling: to 2^-22 of the row's largest), and what is left, sum over groups of (b + 8 s) XS with XS = the group's sum of
// activations, is a product over groups of its own: one MFMA (M = 32) per two slices and tile pair, lane group g holding
// slice 2 i + g, both factors as fp16 hi + lo (hi hi + lo hi + hi lo, 22 bits). k_x16 writes XS in A-operand form.
// Used where the down takes the dense tiles anyway (make_plan): against 64 bits the layer is then as far off as with the wave
// tiles' gate/up before the same down (2.08e-4 of the norm either way, fp32 outputs: the fp16 rounding of h and W_down).
template <int NPROJ, int M, int BM, int MINB, bool EX = false>
__global__ void __launch_bounds__(256, MINB) k_dense_i4(TileArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // buffer resources exist in device code only
    static_assert(!EX || (NPROJ == 2 && M == 32), "exact weights: gate/up in tiles of 32 tokens");
    constexpr int NT = BM / M, BN = 128;
    constexpr int H = 32 / M;             // B tiles per projection: the wave's 32 rows
    constexpr int CB = NPROJ * H;
    constexpr int NJ = M / 4;             // steps per slice
    constexpr int NQ = M == 32 ? 4 : 1;   // groups of 4 tokens per accumulator
    constexpr int SB = TILE_SLICE_INT4;
    constexpr int DEC_EXP = 16;           // the decode's 2^-16 (below)
    typedef std::conditional_t<M == 32, f32x16, f32x4> acc_t;
    __shared__ __attribute__((aligned(1024))) uint8_t sX0[BM * 256];
    __shared__ __attribute__((aligned(1024))) uint8_t sX1[BM * 256];
    __shared__ __attribute__((aligned(16))) int sSlot[BM];
    __shared__ __attribute__((aligned(16))) int sExp[BM];

    // Work items (pass list x row blocks x K parts), ordered expert by expert, within an expert row block by row
    // block with the expert's passes adjacent, K part fastest. The launch hands workgroups to the 8 XCDs round
    // robin (workgroup b to XCD (b + c) mod 8, c fixed per launch), so XCD slot b & 7 takes the contiguous
    // eighth of the live items, in order: each XCD's L2 then holds the activations of few experts, and the
    // passes that share a weight tile run side by side on one XCD (their second reads hit its L2). The grid is
    // a multiple of 8 covering the largest possible item count.
    const int nrb = (a.N + BN - 1) / BN;
    const int nitems = a.meta[a.nidx] * nrb * a.ksplit;
    const int chunk = (nitems + 7) >> 3;
    const int rank = (int)(blockIdx.x >> 3);
    const int item = (int)(blockIdx.x & 7u) * chunk + rank;
    if (rank >= chunk || item >= nitems) return;
    const int ks = item % a.ksplit;                // K part (down only), the fastest index
    const int bid = item / a.ksplit;
    const int wq = bid / nrb;                      // some pass of the current expert
    const int e = a.items[3 * wq], np = a.items[3 * wq + 2];
    const int w0 = wq - a.items[3 * wq + 1];       // the expert's first pass
    const int local = bid - w0 * nrb;
    const int rb = local / np;
    const int tid = threadIdx.x, lane = tid & 63, ln = lane & (M - 1), lg = lane / M;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.K, N = a.N;
    const int nsl = (K + 127) >> 7;
    const int per = (nsl + a.ksplit - 1) / a.ksplit;
    const int sb0 = ks * per;                                // this block's slices: sb0 .. sb0 + scnt - 1
    const int scnt = nsl - sb0 < per ? nsl - sb0 : per;   // >= 1 (the host splits only when it is)
    const int r0 = rb * BN + wave * 32;
    const bool wvalid = r0 < N;           // N % 32 == 0: a wave's rows are all in range or all out
    const uint32_t trec = (uint32_t)nsl * SB;   // one 16-row tile's records
    __amdgpu_buffer_rsrc_t wb[NPROJ];     // the wave's two row tiles of each projection, consecutive
#pragma unroll
    for (int p = 0; p < NPROJ; ++p)
        wb[p] = buffer_of((p ? a.W1 : a.W0) + ((size_t)e * (N >> 4) + (wvalid ? (r0 >> 4) : 0)) * (size_t)trec, 2u * trec);
    const uint32_t wofs = M == 32 ? (uint32_t)(ln >> 4) * trec + 16u * (ln & 15) + 512u * lg : 16u * lane;
    const uint32_t mofs = (M == 32 ? (uint32_t)(ln >> 4) * trec : 0u) + 1024u + 8u * (ln & 15);
    struct WS { u32x4 q[NPROJ][2]; u32x2 m[CB]; };
    auto fetch_w = [&](int s, WS& w) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NPROJ; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                w.q[p][h] = __builtin_amdgcn_raw_buffer_load_b128(wb[p], wofs + (M == 32 ? 256 * h : 0),
                                                                  s * SB + (M == 32 ? 0 : h * (int)trec), 0);
                if (h < H) w.m[p * H + h] = __builtin_amdgcn_raw_buffer_load_b64(wb[p], mofs, s * SB + h * (int)trec, 0);
            }
    };
    WS wa, wn;
    fetch_w(sb0, wa);                     // in flight while the pass's tokens are looked up
    const int n = a.counts[e], beg = a.offsets[e];
    int tok0, nlive;
    pass_tokens<M>(n, np, local - rb * np, tok0, nlive);
    const int ntiles = (nlive + M - 1) / M;
    if (tid < BM) {
        const int slot = a.sorted[beg + (tok0 + tid < n ? tok0 + tid : n - 1)];
        sSlot[tid] = slot;
        // the activation row's power-of-two exponent (k_x16: per token, k_h16_fix: per slot)
        sExp[tid] = NPROJ == 2 ? a.xexp[slot / a.act_div]
                               : reinterpret_cast<const int32_t*>(reinterpret_cast<const uint8_t*>(a.actv2) + a.eslot_off)[slot];
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t xb = buffer_of(a.actv, 0xFFFFFFFFu);
    const int psw = (lane & 15) ^ ((4 * wave + (lane >> 4)) & 15);   // piece loaded by this DMA lane
    // K % 128 == 64: the last slice's pieces past K (they meet zero codes and zero metadata) are the row's last one
    const uint32_t pofs = 16u * psw, pofs_tail = 16u * ((K & 64) && psw > 7 ? 7 : psw);
    uint32_t xrow[BM / 16];               // DMA i of this wave: token rows 4 (wave + 4 i) + (lane >> 4), position lane & 15
#pragma unroll
    for (int i = 0; i < BM / 16; ++i)
        xrow[i] = (uint32_t)(sSlot[4 * (wave + 4 * i) + (lane >> 4)] / a.act_div) * (uint32_t)K * 2u;
    // EX: the lane's tokens' group sums (token ln of each tile), 16 bytes per slice
    const __amdgpu_buffer_rsrc_t gb = buffer_of(a.xsum, 0xFFFFFFFFu);
    uint32_t grow[EX ? NT : 1];
#pragma unroll
    for (int t = 0; t < (EX ? NT : 0); ++t) grow[t] = (uint32_t)(sSlot[M * t + ln] / a.act_div) * (uint32_t)nsl * 16u;
    // LDS offset of the lane's A operand of step 0; the later steps' words differ in the bits of 16 * word only
    uint32_t aofs = (uint32_t)ln * 256u + 16u * (((NJ / 2) * lg) ^ (ln & 15));

    acc_t acc[CB][NT];
#pragma unroll
    for (int b = 0; b < CB; ++b)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4 * NQ; ++v) acc[b][t][v] = 0.f;

    auto run = [&](auto ntl) __attribute__((always_inline)) {
        constexpr int L = decltype(ntl)::value;   // live token tiles
        auto fetch_x = [&](int s, uint8_t* buf) __attribute__((always_inline)) {
            const uint32_t po = s == nsl - 1 ? pofs_tail : pofs;
#pragma unroll
            for (int i = 0; i < L * M / 16; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, MOE_LDSP(buf + 4 * (wave + 4 * i) * 256), 16, xrow[i] + po,
                                                         256 * s, 0, 0);
        };
        auto compute = [&](const uint8_t* xs, const WS& w) __attribute__((always_inline)) {
            h2x s2[2][CB], b2[2][CB];
            asm volatile("" : "+v"(aofs));   // the steps' addresses are one xor each, not a register each
            auto scale = [&](int G) __attribute__((always_inline)) {
#pragma unroll
                for (int b = 0; b < CB; ++b) {
                    const uint32_t mw = G ? w.m[b].y : w.m[b].x;
                    const _Float16 s16 = (_Float16)(bf16lo(mw) * 16.0f), b16 = (_Float16)(EX ? bf16lo(mw) * -0x1p-13f : bf16hi(mw) * 0x1p-16f);
                    s2[G][b] = h2x{s16, s16};
                    b2[G][b] = h2x{b16, b16};
                }
            };
            // B operand b of step j, w' = (s q + b) 2^-16 in one rounding: each code pair (q_k, q_{k+4}) is masked into
            // bits 4-7 of two fp16 halves with exponent 0, which makes them the exact subnormals q 2^-20, and one
            // v_pk_fma_f16 takes q 2^-20 (16 s) + b 2^-16. The records' row scaling keeps |s|, |b| below 2^11, so
            // 16 s < 2^15 fits fp16 and |w'| < 2^-1: a weight stays a normal fp16 number down to 2^-13 of that bound,
            // and below it rounds to fp16's subnormal step 2^-24 (2^-19 of the row's largest |s|, |b| in w' units). The
            // epilogue adds 16 to the row exponent. (Codes left in bits 0-3 as q 2^-24 save two shifts, but bound
            // |w'| by 2^-5 and so put weights 2^9 below the row's largest into the subnormal range: one group per row
            // at 64x the others' scale and small x on it then reached 8e-3 of the output RMS in a numpy emulation.)
            auto decode = [&](int j, int b) __attribute__((always_inline)) {
                const uint32_t x = M == 32 ? w.q[b][(j >> 1) & 1][(j & 1) + 2 * (j >> 2)] : w.q[b / H][b % H][j];
                const int G = 2 * j / NJ;
                const uint32_t c4[4] = {(x << 4) & 0x00F000F0u, x & 0x00F000F0u, (x >> 4) & 0x00F000F0u, (x >> 8) & 0x00F000F0u};
                h2x v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = __builtin_elementwise_fma(__builtin_bit_cast(h2x, c4[i]), s2[G][b], b2[G][b]);
                return f16x8{v[0][0], v[0][1], v[1][0], v[1][1], v[2][0], v[2][1], v[3][0], v[3][1]};
            };
            auto load_a = [&](int j, int t) __attribute__((always_inline)) {
                const uint32_t o = aofs ^ (16u * (j % (NJ / 2) + 8 * (2 * j / NJ)));
                return *reinterpret_cast<const f16x8*>(xs + o + 256 * M * t);
            };
            f16x8 A[2][L], B[2][CB];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < L; ++t) A[0][t] = load_a(0, t);
            scale(0);
#pragma unroll
            for (int b = 0; b < CB; ++b) B[0][b] = decode(0, b);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if (j == NJ / 2 - 2 + (M == 16)) scale(1);
                if (j < NJ - 1) {
#pragma unroll
                    for (int t = 0; t < L; ++t) A[(j + 1) & 1][t] = load_a(j + 1, t);
#pragma unroll
                    for (int b = 0; b < CB; ++b) B[(j + 1) & 1][b] = decode(j + 1, b);
                }
#pragma unroll
                for (int t = 0; t < L; ++t)
#pragma unroll
                    for (int b = 0; b < CB; ++b) {
                        if constexpr (M == 32)
                            acc[b][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[j & 1][t], B[j & 1][b], acc[b][t], 0, 0, 0);
                        else
                            acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[j & 1][t], B[j & 1][b], acc[b][t], 0, 0, 0);
                    }
                // the next step's LDS reads and decode between this step's MFMAs
#pragma unroll
                for (int i = 0; i < CB * L; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i < L) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (12 + L - 1) / L, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // EX: the group-sum term of slices s2 and s2 + 1 (s2 even), loaded at slice s2, multiplied two slices later
        f16x8 gx[EX ? L : 1];
        u32x2 gm[EX ? CB : 1];
        auto fetch_g = [&](int s2) __attribute__((always_inline)) {
            if constexpr (EX) {
                const int sl = s2 + lg < nsl ? s2 + lg : nsl - 1;
#pragma unroll
                for (int t = 0; t < L; ++t)
                    gx[t] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(gb, grow[t] + 16u * sl, 0, 0));
#pragma unroll
                for (int b = 0; b < CB; ++b) gm[b] = __builtin_amdgcn_raw_buffer_load_b64(wb[b], mofs + (uint32_t)(sl * SB), 0, 0);
                if (s2 + lg >= nsl)
#pragma unroll
                    for (int b = 0; b < CB; ++b) gm[b] = u32x2{0u, 0u};
            }
        };
        auto apply_g = [&]() __attribute__((always_inline)) {
            if constexpr (EX) {
#pragma unroll
                for (int b = 0; b < CB; ++b) {
                    _Float16 hi[2], lo[2];
#pragma unroll
                    for (int G = 0; G < 2; ++G) {   // (b + 8 s) 2^-16, times the 2^6 that XS is scaled down by
                        const float v = __builtin_fmaf(8.f, bf16lo(gm[b][G]), bf16hi(gm[b][G])) * 0x1p-10f;
                        hi[G] = (_Float16)v;
                        lo[G] = (_Float16)(v - (float)hi[G]);
                    }
                    const f16x8 Bg = {hi[0], hi[1], lo[0], lo[1], hi[0], hi[1], (_Float16)0, (_Float16)0};
#pragma unroll
                    for (int t = 0; t < L; ++t) acc[b][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(gx[t], Bg, acc[b][t], 0, 0, 0);
                }
            }
        };
        fetch_x(sb0, sX0);
        MOE_VMWAIT0();
        MOE_BARRIER();
        int j = 0;
        for (; j + 2 <= scnt; j += 2) {
            fetch_w(sb0 + j + 1, wn);
            fetch_x(sb0 + j + 1, sX1);
            if constexpr (EX) {
                if (j) apply_g();
                fetch_g(j);
            }
            compute(sX0, wa);
            MOE_VMWAIT0();
            MOE_BARRIER();
            const int jn = sb0 + (j + 2 < scnt ? j + 2 : j + 1);   // the last slice again: no branch around the loads
            fetch_w(jn, wa);
            fetch_x(jn, sX0);
            compute(sX1, wn);
            MOE_VMWAIT0();
            MOE_BARRIER();
        }
        if constexpr (EX) {   // the last group sums: fetched in the loop but not multiplied, or not fetched yet
            if (j) apply_g();
            if (j < scnt) {
                fetch_g(j);
                apply_g();
            }
        }
        if (j < scnt) compute(sX0, wa);   // odd count: the last slice is in buffer 0
    };
    if (NT == 1 || ntiles == 1) run(std::integral_constant<int, 1>{});
    else if constexpr (NT >= 2) {
        if (NT == 2 || ntiles == 2) run(std::integral_constant<int, 2>{});
        else if constexpr (NT == 4) {
            if (ntiles == 3) run(std::integral_constant<int, 3>{});
            else run(std::integral_constant<int, 4>{});
        }
    }

    // ---- epilogue: lane holds row r0 + M b + ln of tokens M t + (8 q) + 4 lg + v of the pass (v = 0..3, acc entry 4 q + v)
    if (!wvalid) return;
    int rex[CB];   // row exponents (the records hold s 2^-E, b 2^-E), plus the decode's
#pragma unroll
    for (int b = 0; b < CB; ++b)
        rex[b] = tile_row_exps(b / H ? a.W1 : a.W0, a.E, N, K)[(size_t)e * N + r0 + M * (b % H) + ln] + DEC_EXP;
    auto each_quad = [&](auto fn) __attribute__((always_inline)) {   // fn(t, q, first token, exponents, slots) of 4 tokens
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (t >= ntiles) break;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int j0 = M * t + 8 * q + 4 * lg;
                const int4 x4 = *reinterpret_cast<const int4*>(&sExp[j0]), s4 = *reinterpret_cast<const int4*>(&sSlot[j0]);
                const int xe[4] = {x4.x, x4.y, x4.z, x4.w}, sl[4] = {s4.x, s4.y, s4.z, s4.w};
                fn(t, q, j0, xe, sl);
            }
        }
    };
    if constexpr (NPROJ == 2) {
        // h of the wave's 32 rows as fp16 h16 = h 2^-e, e per (slot, 32-row chunk): h16_exponent of the chunk's largest.
        // Two tokens' values of a lane pair are exchanged so that each lane stores two adjacent rows of one token.
        int8_t* hexp_out = reinterpret_cast<int8_t*>(a.hout2);
        const int nch = N >> 5;
        float bg[H], bu[H];
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const size_t r = (size_t)e * N + r0 + M * h + ln;
            bg[h] = a.b0 ? a.b0[r] : 0.f;
            bu[h] = a.b1 ? a.b1[r] : 0.f;
        }
        const __amdgpu_buffer_rsrc_t hb = buffer_of(a.hout, (uint32_t)ACT_BYTES_MAX);   // a dead token's offset lies past it
        const bool odd = ln & 1;
        const uint32_t lofs = 2u * (uint32_t)(ln & ~1), psel = odd ? 0x05040100u : 0x01000504u;   // (own, received)
        each_quad([&](int t, int q, int j0, const int (&xe)[4], const int (&sl)[4]) __attribute__((always_inline)) {
            float hv[H][4], am[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                am[v] = 0.f;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float g = __builtin_ldexpf(acc[h][t][4 * q + v], xe[v] + rex[h]) + bg[h];
                    const float up = __builtin_ldexpf(acc[H + h][t][4 * q + v], xe[v] + rex[H + h]) + bu[h];
                    hv[h][v] = glu_fast(a.act, g, up);
                    am[v] = fmaxf(am[v], fabsf(hv[h][v]));
                }
                am[v] = max_lanes<M>(am[v]);
            }
            int ex[4] = {0, 0, 0, 0};
            const float lo = fminf(fminf(am[0], am[1]), fminf(am[2], am[3])), hi = fmaxf(fmaxf(am[0], am[1]), fmaxf(am[2], am[3]));
            if (!__all(lo >= 0.00390625f && hi < 32768.f)) {   // else every exponent is 0
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    ex[v] = h16_exponent(am[v]);
#pragma unroll
                    for (int h = 0; h < H; ++h) hv[h][v] = __builtin_ldexpf(hv[h][v], -ex[v]);
                }
            }
            if (ln < 4 && j0 + ln < nlive)
                hexp_out[(size_t)sSlot[j0 + ln] * nch + (r0 >> 5)] =
                    (int8_t)(ln == 0 ? ex[0] : (ln == 1 ? ex[1] : (ln == 2 ? ex[2] : ex[3])));
#pragma unroll
            for (int v = 0; v < 4; v += 2) {
                const int j = j0 + v + (odd ? 1 : 0);
                const uint32_t o = j < nlive ? (uint32_t)(odd ? sl[v + 1] : sl[v]) * (2u * (uint32_t)N) + lofs : 0xFFFFF800u;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const uint32_t h0 = __builtin_bit_cast(uint16_t, (_Float16)hv[h][v]),
                                   h1 = __builtin_bit_cast(uint16_t, (_Float16)hv[h][v + 1]);
                    const uint32_t own = odd ? h1 : h0;
                    const uint32_t got = (uint32_t)__builtin_amdgcn_mov_dpp((int)(odd ? h0 : h1), 0xB1, 0xF, 0xF, true);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_amdgcn_perm(own, got, psel), hb, o, 2 * r0 + 32 * h, 0);
                }
            }
        });
    } else {
        each_quad([&](int t, int q, int j0, const int (&xe)[4], const int (&sl)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (j0 + v >= nlive) continue;
#pragma unroll
                for (int b = 0; b < CB; ++b)
                    a.yp[ks * a.plane + (size_t)sl[v] * N + r0 + M * b + ln] =
                        __builtin_ldexpf(acc[b][t][4 * q + v], xe[v] + rex[b]);
            }
        });
    }
#endif
}
