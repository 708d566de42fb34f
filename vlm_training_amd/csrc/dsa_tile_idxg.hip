// Indexer backward, query side (see dsa_tile_idx.hip for the sums): dq_idx and dw of one query per wave, over the keys it selected and no
// others.  A wave's rows are the query's indexer heads, RG groups of 32; its selected keys, 32 at a time, are gathered from k_idx
// straight into its own LDS ring by their indices (ascending, so that the walk's order is the list's), their gradients lie one behind
// the other.  No bitmap, no slot arithmetic, no barrier: a workgroup is one wave.
//   S^T = K Q^T (A = gathered tile row-wise, B = Q^T in registers), G = dscore where S > 0, dw += dscore relu(S),
//   dQ^T += K^T G^T (A = the tile transposed, B = G from the C layout; sums in accumulation registers)
// Step t runs S(t+1), behind it the gating of tile t, then dQ(t), behind it the addresses of tile t+4.  Tile t+3 is requested at the
// start of step t, waited for in the middle of step t+1.
//
// What bounds it: 32 MFMAs (1024 clocks) per tile at 64 heads of 128 beside about 155 vector and as many other instructions, the latency
// of what a step waits for (LDS reads right in front of their use took another 250 us), and about 4 us around a query's walk.  32 768
// tokens, 2048 of up to 7168 keys, 64 heads of 128: 2192 us over every causal tile, 1652 so; dsa_tile_idx.hip has the line between them.
#include "dsa_tile.h"

template <int D> constexpr size_t idxg_lds_bytes() { return 4 * (size_t)DirectTile<D>::BYTES + 8 * 256 + 4 * 256; }
template <int D, int RG>
__global__ __launch_bounds__(64, 1) void dsa_tile_idxg_kernel(
    const bf16_t *__restrict__ q_idx, const bf16_t *__restrict__ k_idx, const bf16_t *__restrict__ w_idx, const int32_t *__restrict__ idx,
    const int32_t *__restrict__ nsel, const float *__restrict__ dscore, const float *__restrict__ grad, int ldw, const int32_t *__restrict__ cu, int N,
    int T, int Hi, int K, float cscale, bf16_t *__restrict__ dq_idx, void *__restrict__ dw, int dw_bf16) {
    typedef DirectTile<D> TL;
    constexpr int KS = D / 16, DT = D / 32, NP = 2 * DT, LOADS = TL::LOADS, LPS = LOADS + 2, AHEAD = 4, E = 16 * RG;
    static_assert(TL::SOURCES == 1 && (LOADS == 8 || LOADS == 4) && KS % AHEAD == 0 && NP == KS && AHEAD <= NP && LOADS == NP, "");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // 4 K slots | indices [tile % 8] | gradients [tile % 4]
    constexpr int IDS = 4 * TL::BYTES, GRADS = IDS + 8 * 256;

    const int lane = threadIdx.x, h = lane >> 5, j = lane & 31;
    const int t = T - 1 - (int)blockIdx.x;
    const int seg = find_segment_wave(cu, N, t);
    const int s0 = __builtin_amdgcn_readfirstlane(cu[seg]);
    const int L = min(__builtin_amdgcn_readfirstlane(cu[seg + 1]) - s0, ldw * 32);    // (no key past the longest segment the caller names)
    if (t - s0 >= L || !idx_segment_gathers(Hi, K, L)) return;
    const int n = __builtin_amdgcn_readfirstlane(max(min(nsel[t], K), 0)), ntiles = max((n + 31) / 32, 1);

    // ---- requests ----
    const uint32_t lds0 = lds_address(dyn_lds);
    const buffer_rsrc keys = make_buffer_rsrc(k_idx + (int64_t)s0 * D, (int64_t)L * 2 * D);
    const buffer_rsrc ids = make_buffer_rsrc(idx + (int64_t)t * K, (int64_t)n * 4), grads = make_buffer_rsrc(dscore + (int64_t)t * K, (int64_t)n * 4);
    const int row = lane / TL::CPR;
    const uint32_t key0 = ((lane % TL::CPR) ^ TL::xor_of(row)) * 16 - (uint32_t)s0 * (2 * D);    // (indices outside the segment leave the buffer)
    auto load_ids = [&](int tile) __attribute__((always_inline)) { buffer_load_lds4(ids, tile * 128 + lane * 4, lds0 + IDS + (tile & 7) * 256); };
    auto load_grads = [&](int tile) __attribute__((always_inline)) { buffer_load_lds4(grads, tile * 128 + lane * 4, lds0 + GRADS + (tile & 3) * 256); };
    int voff[LOADS];                                     // the lane's 16 bytes of each piece of the tile requested next
    int id[LOADS];
    auto read_ids = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) id[p] = *reinterpret_cast<const int *>(dyn_lds + IDS + (tile & 7) * 256 + (p * TL::LOAD_ROWS + row) * 4);
    };
    auto find_keys = [&](int tile, int p) __attribute__((always_inline)) {
        asm volatile("" : "+v"(id[p]));                  // (read in any case: no branch)
        voff[p] = tile * 32 + p * TL::LOAD_ROWS + row < n ? (int)((uint32_t)id[p] * (2 * D) + key0) : (int)0x80000000;        // (past the list: zeros)
    };
    auto load_keys = [&](int tile) __attribute__((always_inline)) {
        constexpr int P1 = TL::load_lds(1), P2 = TL::load_lds(2) - P1, P3 = TL::load_lds(3) - TL::load_lds(2);
#pragma unroll
        for (int i = 0; i < LOADS; i += 4) {
            const int v[4] = {voff[i], voff[i + 1], voff[i + 2], voff[i + 3]};
            buffer_load_lds16_n<4, P1, P2, P3>(keys, v, lds0 + (tile & 3) * TL::BYTES + TL::load_lds(i));
        }
    };
#pragma unroll
    for (int u = 0; u < 5; ++u) load_ids(u);
    load_grads(0);
    load_grads(1);
    bf16x8 qB[RG][KS];
    float w[RG], dwacc[RG];
    f32x16 acc[RG][DT];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        const int head = 32 * g + j;
        const int64_t at = (int64_t)t * Hi + min(head, Hi - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qB[g][ks] = head < Hi ? load_bf16x8(q_idx + at * D + 16 * ks + 8 * h) : zero_bf16x8();
        w[g] = head < Hi ? (float)w_idx[at] : 0.f;
        dwacc[g] = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            acc[g][dt] = zero16();
            settle(acc[g][dt]);
        }
    }
    if (grad) cscale *= *grad;
    wait_vmcnt<0>();
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        read_ids(u);
#pragma unroll
        for (int p = 0; p < LOADS; ++p) find_keys(u, p);
        load_keys(u);
    }
    read_ids(3);
#pragma unroll
    for (int p = 0; p < LOADS; ++p) find_keys(3, p);
    lds_u8 *aR[4], *aT[4];                               // operand addresses: row-wise of the tile of S, transposed of the tile of dQ
    {
        TL tl;
        tl.init(lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aR[i] = (lds_u8 *)dyn_lds + tl.rowq[i];
            aT[i] = (lds_u8 *)dyn_lds + tl.trq[i];
        }
    }
    wait_vmcnt<0>();
    auto fence = [&]() __attribute__((always_inline)) {
        asm volatile("" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto advance = [&](lds_u8 *(&a)[4], int tile) __attribute__((always_inline)) {         // from tile - 1 to tile
        const int by = tile & 3 ? TL::BYTES : -3 * TL::BYTES;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] += by;
            asm volatile("" : "+v"(a[i]));
        }
    };
    auto row_op = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(aR[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto tr_op = [&](int i) __attribute__((always_inline)) {              // MFMA i of dQ: keys of half i / DT, d-tile i % DT
        const int pair = i / DT, dt = i % DT;
        return tr_pair(aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair), aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair + 1));
    };
    f32x16 sE[RG], sO[RG];                               // S of even and of odd tiles
    bf16x8 op[AHEAD];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const bf16x8 a = row_op(ks);
#pragma unroll
        for (int g = 0; g < RG; ++g) sE[g] = mfma32(a, qB[g][ks], ks == 0 ? zero16() : sE[g]);
    }
    advance(aR, 1);
#pragma unroll
    for (int m = 0; m < AHEAD; ++m) op[m] = row_op(m);

    f32x4 d4[4];                                         // gradients of tile t: element vi is key 8*(vi/4) + 4h + vi%4
    auto read_grads = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) d4[g4] = *reinterpret_cast<const f32x4 *>(dyn_lds + GRADS + (tile & 3) * 256 + 32 * g4 + 16 * h);
    };
    read_grads(0);

    // Step t: S(t+1) into `sn` (NEXT), behind it the gating of tile t from `s`; dQ(t), behind it the addresses of tile t+4.
    auto step = [&](auto next_, int t_, const f32x16 (&s)[RG], f32x16 (&sn)[RG]) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(next_)::value;
        constexpr int M = 2 * KS, SL = RG * KS;
        auto refill = [&](int m) __attribute__((always_inline)) {         // operand m is used up (in pairs where two groups share them)
            if (RG == 2 && m % 2 == 0) return;
#pragma unroll
            for (int x = RG == 2 ? m - 1 : m; x <= m; ++x) {
                const int y = x + AHEAD;
                if (y >= M && !NEXT) continue;
                if (y == M) advance(aR, t_ + 2);
                op[x % AHEAD] = y < KS ? row_op(y) : y < M ? tr_op(y - KS) : row_op(y - M);
                if (y == M - 1) advance(aT, t_ + 1);
            }
        };
        auto pair = [&](int m) __attribute__((always_inline)) {
            if (RG == 2 && m % 2 == 0) asm volatile("" : "+v"(op[m % AHEAD]), "+v"(op[(m + 1) % AHEAD]));
        };
        if (NEXT) {
            load_keys(t_ + 3);
            load_grads(t_ + 2);
            load_ids(t_ + 5);
        }
        fence();
        uint32_t gp[RG][8];                              // G in bf16
        float x[E];
        auto gate = [&](int e) __attribute__((always_inline)) {
            const int g = e / 16, vi = e % 16;
            x[e] = s[g][vi] > 0.f ? d4[vi >> 2][vi & 3] : 0.f;           // (the row's weight multiplies the finished sum instead)
            dwacc[g] = fmaf(x[e], s[g][vi], dwacc[g]);                   // dscore * relu(s)
            asm volatile("" : "+v"(x[e]), "+v"(dwacc[g]));
            if (vi & 1) {
                gp[g][vi >> 1] = pack2bf(x[e - 1], x[e]);
                asm volatile("" : "+v"(gp[g][vi >> 1]));
            }
        };
        if (NEXT) {
#pragma unroll
            for (int m = 0; m < KS; ++m) {
                pair(m);
#pragma unroll
                for (int g = 0; g < RG; ++g) {
                    const int u = m * RG + g;
                    sn[g] = mfma32(op[m % AHEAD], qB[g][m], m == 0 ? zero16() : sn[g]);
                    if (g == RG - 1) refill(m);
#pragma unroll
                    for (int e = E * u / SL; e < E * (u + 1) / SL; ++e) gate(e);
                    fence();
                }
            }
            wait_vmcnt<LPS>();                           // all but what this step requested
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) gate(e);
#pragma unroll
            for (int m = 0; m < AHEAD; ++m) op[m] = tr_op(m);
            fence();
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int m = NEXT ? KS + i : i;
            pair(m);
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                const int c = i < DT ? 0 : 4;
                const u32x4 b = {gp[g][c], gp[g][c + 1], gp[g][c + 2], gp[g][c + 3]};
                mfma32_agpr(acc[g][i % DT], op[m % AHEAD], __builtin_bit_cast(bf16x8, b), !NEXT);
                if (NEXT && g == RG - 1) refill(m);
                if (!NEXT && g == RG - 1 && i + AHEAD < NP) op[i % AHEAD] = tr_op(i + AHEAD);
                if (NEXT && g == 0) {                    // (read half a phase before they are needed)
                    if (i == 0) read_ids(t_ + 4);
                    if (i == NP / 2 - 1) read_grads(t_ + 1);
                    if (i >= NP / 2)
#pragma unroll
                        for (int p = 0; p < 2; ++p) find_keys(t_ + 4, 2 * (i - NP / 2) + p);
                }
                fence();
            }
        }
    };
    const std::true_type yes;
    const std::false_type no;
    int tt = 0;
    for (; tt + 2 < ntiles; tt += 2) {
        step(yes, tt, sE, sO);
        step(yes, tt + 1, sO, sE);
    }
    if (tt + 1 < ntiles) {
        step(yes, tt, sE, sO);
        ++tt;
#pragma unroll
        for (int g = 0; g < RG; ++g) sE[g] = sO[g];
    }
#pragma unroll
    for (int i = 0; i < RG * DT; ++i) settle(acc[i / DT][i % DT]);
    asm volatile("s_nop 1");
    step(no, tt, sE, sO);
    wait_vmcnt<0>();                                     // no load is left on its way into LDS

#pragma unroll
    for (int g = 0; g < RG; ++g) {
        const int head = 32 * g + j;
        const float dwt = half_sum_f(dwacc[g]) * cscale;
        const int64_t at = (int64_t)t * Hi + head;
        if (head < Hi) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                settle(acc[g][dt]);
                store_c_tile(dq_idx + at * D + dt * 32, acc[g][dt], cscale * w[g], h);
            }
            if (h == 0) {
                if (dw_bf16) reinterpret_cast<bf16_t *>(dw)[at] = (bf16_t)dwt;
                else reinterpret_cast<float *>(dw)[at] = dwt;
            }
        }
    }
}

template <int D, int RG>
static hipError_t launch_idxg(hipStream_t stream, const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                              const float *dscore, const float *grad, int ldw, const int32_t *cu, int N, int T, int Hi, int K, float cscale, void *dq_idx,
                              void *dw, int dw_bf16) {
    constexpr size_t lds = idxg_lds_bytes<D>();
    hipLaunchKernelGGL((dsa_tile_idxg_kernel<D, RG>), dim3((unsigned)T), dim3(64), lds, stream, (const bf16_t *)q_idx, (const bf16_t *)k_idx,
                       (const bf16_t *)w_idx, idx, n, dscore, grad, ldw, cu, N, T, Hi, K, cscale, (bf16_t *)dq_idx, dw, dw_bf16);
    return hipGetLastError();
}
// D = indexer head_dim (64 or 128), at most 64 indexer heads; grad: one fp32 factor of every gradient on the device, or null
extern "C" hipError_t dsa_launch_indexer_bwd_gather(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                                               const float *dscore, const float *grad, int ldw, const int32_t *cu, int N, int T, int Hi, int Di, int K,
                                               float cscale, void *dq_idx, void *dw, int dw_bf16, hipStream_t stream) {
    if (Hi < 1 || Hi > 64 || !(Di == 64 || Di == 128)) return hipErrorInvalidValue;
#define IDXG(D_, RG_) launch_idxg<D_, RG_>(stream, q_idx, k_idx, w_idx, idx, n, dscore, grad, ldw, cu, N, T, Hi, K, cscale, dq_idx, dw, dw_bf16)
    if (Di == 128) return Hi > 32 ? IDXG(128, 2) : IDXG(128, 1);
    return Hi > 32 ? IDXG(64, 2) : IDXG(64, 1);
#undef IDXG
}
