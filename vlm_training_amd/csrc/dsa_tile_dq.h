// dQ over 32x32 MFMA tiles, query-stationary, the same walk as the forward (dsa_tile_fwd.hip):
//   S^T = K Q^T, dP^T = V dO^T  (A = K / V tiles row-wise from LDS, B = Q^T / dO^T in registers; the sums of dP start from -delta)
//   dS^T = P^T * dP^T           on the C layout, P = exp2(S * scale*log2e - lse*log2e)
//   dQ^T[d,row] += K^T[d,key] dS^T[key,row]   (A = K tile transposed, B = dS^T from the C layout)
//
// One wave per SIMD with 512 registers and 64 rows (RG = 2 groups of 32), so that each operand read from LDS feeds two MFMAs; 32 rows at
// head_dim 256, where a row alone fills the registers, and in launches of little work (dq_one_row_group).  Step t runs dQ(t) mixed
// with dP(t+1), the logits and exponentials P(t+1) behind them, then S(t+2), the products and packing of dS(t+1) behind it; operand reads
// run four ahead through all of it, in pairs where two groups share them.  K and V tiles go from memory straight into LDS, rings of five
// and three: step t requests K(t+4), V(t+3) and the selection words of tile t+3, at its end waits for what step t-1 requested and meets
// the one barrier.  Tiles that every row attends whole run without mask arithmetic (with a selection: in blocks inside the first K positions).
//
// What bounds it: the issue of one instruction stream per SIMD - at head_dim 128 48 MFMAs (1536 clocks) beside about 125 vector
// instructions (195 with a mask), 33 LDS reads and 70 scalar ones - and the chip's power.  Same box, us, against the kernels before
// (head_dim 128: two waves of 32 rows per SIMD, tiles through registers; elsewhere 32 rows per wave, the three chains one after the
// other): 32 768 tokens dense 1727 -> 1613, with a selection 1775 -> 1709; head_dim 256, 16 384 tokens in short segments 277 -> 243;
// towers at head_dim 64 / 72, whole backward 775 -> 749 / 960 -> 934.  Two waves a workgroup, two workgroups a CU: level dense, 25 us more
// with a selection (each tile is staged twice as often).  Operands of one row group in pairs: 254 instead of 243 at head_dim 256.
#pragma once
#include "dsa_tile.h"

#define DQ_RK 5                                          // K tiles in LDS: K(t) to K(t+4)
#define DQ_RV 3                                          // V tiles: V(t+1) to V(t+3)
template <int D, int NW> constexpr size_t dq_lds_bytes(bool has_idx) { return (DQ_RK + DQ_RV) * (size_t)DirectTile<D>::BYTES + (has_idx ? NW * 4 * 256 : 0); }

// Workgroup `block` of `blocks`
template <int D, bool HAS_IDX, int NW, int RG, bool CARRIED>
__device__ __forceinline__ void dq_block(int block, int blocks,
    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k,
    const bf16_t *__restrict__ v, const float *__restrict__ lse, const float *delta,
    const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv, int gshift,
    float scale, int pos_split, int split_len, int pos_short, int window, int causal, int d_real, bf16_t *__restrict__ dq, const bf16_t *__restrict__ out_for_delta,
    float *delta_out) {
    typedef DirectTile<D> TL;
    constexpr int KS = CARRIED ? DSA_CARRIED_KS : D / 16, DT = CARRIED ? 4 : (D + 31) / 32, NP = 2 * DT;
    auto tile_of = [](int dt) __attribute__((always_inline)) { return CARRIED ? carried_tile(dt) : dt; };
    constexpr int LPW = TL::LOADS / NW;                  // wave loads per wave, step and operand
    constexpr int LPS = 2 * LPW + (HAS_IDX ? 1 : 0);     // everything a wave requests in a step
    constexpr int AHEAD = 4;                             // operands read ahead
    constexpr int K_END = DQ_RK * TL::BYTES, V_END = (DQ_RK + DQ_RV) * TL::BYTES;
    static_assert(TL::LOADS % NW == 0 && AHEAD <= NP, "every wave loads the same number of pieces");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // K slots | V slots | selection words

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv, kvh = block % Hkv, QBW = (NW * RG * 32) >> gshift;
    const int dr = HAS_IDX || CARRIED ? D : d_real, chunks = CARRIED ? 2 * KS : dr / 8;   // elements and 16-byte chunks of a row in memory
    int s0, L, blk;
    if (!LOCATE_QUERY_BLOCK(causal, blocks, cu, N, block / Hkv, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = __builtin_amdgcn_readfirstlane(L);
    if (HAS_IDX) L = min(L, ldw * 32);                   // a bitmap row has ldw words whatever the caller's max_seqlen
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (qc0 >= min(L, tile_rows_end(L, pos_split, split_len, pos_short))) return;       // rows past the split are not the tile kernels'
    const int ntiles = (causal ? min(qc0 + QBW - 1, L - 1) : L - 1) / 32 + 1;

    // ---- requests ----
    const int tok_b = Hkv * dr * 2;                      // bytes from one key row to the next
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k + ((int64_t)s0 * Hkv + kvh) * dr);
    const unsigned char *vptr = reinterpret_cast<const unsigned char *>(v + ((int64_t)s0 * Hkv + kvh) * dr);
    int voff[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) voff[i] = TL::source(wv * LPW + i, lane, tok_b, chunks);
    const uint32_t lds0 = lds_address(dyn_lds);
    const uint32_t full_b = 31 * tok_b + dr * 2, last_b = full_b - max(ntiles * 32 - L, 0) * tok_b;
    // the wave's pieces of K (or V) tile `tile` to byte `slot`; called in tile order.  Rows past the segment and columns past the true
    // head_dim read as zero.
    auto load_tile = [&](const unsigned char *&p, int tile, int slot) __attribute__((always_inline)) {
        const uint32_t bytes = tile < ntiles - 1 ? full_b : tile == ntiles - 1 ? last_b : 0u;
        constexpr int P1 = LPW > 1 ? 1 : 0, P2 = LPW > 2 ? 2 : P1, P3 = LPW > 2 ? 3 : P2;
        buffer_load_lds16_n<LPW, TL::load_lds(P1), TL::load_lds(P2) - TL::load_lds(P1), TL::load_lds(P3) - TL::load_lds(P2)>(
            scalar_buffer_rsrc(p, bytes), voff, lds0 + slot + TL::load_lds(wv * LPW));
        p += (int64_t)32 * tok_b;
        asm volatile("" : "+s"(p));
    };
    // selection words: lane l loads that of the wave's row l (32 rows: of row l % 32)
    const int r0 = wv * 32 * RG, wq0 = min(qc0 + (r0 >> gshift), L - 1);   // the wave's first row and query
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + wq0) * ldw);
    const int wvoff = (min(qc0 + ((r0 + lane % (32 * RG)) >> gshift), L - 1) - wq0) * ldw * 4;
    auto load_w = [&](int tile) __attribute__((always_inline)) {
        if (HAS_IDX) {
            buffer_load_lds4(make_buffer_rsrc(wptr, 64 * (int64_t)ldw * 4), wvoff, lds0 + V_END + wv * 1024 + (tile & 3) * 256);
            wptr += tile + 1 < ntiles ? 4 : 0;           // (past the block's tiles: the last word again, never used)
            asm volatile("" : "+s"(wptr));
        }
    };
    auto request_first = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            load_tile(kptr, u, u * TL::BYTES);
            if (u < 2) {
                load_tile(vptr, u, K_END + u * TL::BYTES);
                load_w(u);
            }
        }
    };
    // One row group: the wave's rows of q and dO come in whole rows through the rings' eight slots, in front of the tiles (read where they lie, each
    // load would touch 32 rows: 8000 clocks of a block at head_dim 256); not where they are off 16-byte addresses
    TL tl;
    tl.init(lane);
    static_assert(DQ_RK + DQ_RV == 2 * NW, "");
    const bool staged = RG == 1 && !(((uintptr_t)q | (uintptr_t)dout) & 15) && (int64_t)Hq * dr < (1 << 24);
    if (staged) {
        const WaveRows<TL> wr(gshift, lane);
        const int row_b = dr * 2, q_b = Hq * row_b, there = L - (qc0 + (r0 >> gshift)), place = wr.place(q_b, row_b);
        const int64_t base = ((int64_t)(s0 + wq0) * Hq + kvh * G) * dr;
        const buffer_rsrc q_rows = make_buffer_rsrc(q + base, 0x7fffffff), do_rows = make_buffer_rsrc(dout + base, 0x7fffffff);
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i) {
            const int c = (lane % TL::CPR) ^ TL::xor_of(i * TL::LOAD_ROWS + lane / TL::CPR);
            const int off[1] = {wr.query(i) < there && wr.head(i) < G && c < chunks ? place + wr.piece(i, q_b, row_b) + c * 16 : (int)0x80000000};
            buffer_load_lds16_n<1, 0, 0, 0>(q_rows, off, lds0 + wv * TL::BYTES + TL::load_lds(i));
            buffer_load_lds16_n<1, 0, 0, 0>(do_rows, off, lds0 + (NW + wv) * TL::BYTES + TL::load_lds(i));
        }
    } else {
        request_first();
    }
    // rows of the wave: (query, head of the group), RG groups of 32; a lane holds row j of each group, half h of every 16 elements
    bf16x8 qB[RG][KS], doB[RG][KS];
    float neg_lse2[RG];
    f32x16 dneg[RG];                                     // the sums of dP start from -delta
    int klim[RG];                                        // last key column the row may attend (dense mode); -1: no such row
    uint32_t row_mask[RG];
    const float scale_log2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(scale * LOG2E_F)));
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        const int r = r0 + 32 * g + j, qcol = qc0 + (r >> gshift), head = r & ((1 << gshift) - 1);
        const bool row_ok = qcol < L && head < G;
        const int t = s0 + min(qcol, L - 1), hq = kvh * G + min(head, G - 1);
        klim[g] = row_ok ? (causal ? qcol : L - 1) : -1;
        row_mask[g] = row_ok ? 0xffffffffu : 0u;
        if (staged) {
            wait_vmcnt<0>();                             // (the wave's own pieces)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                lds_u8 *const at = (lds_u8 *)dyn_lds + wv * TL::BYTES + tl.rowq[TL::row_q(ks)] + TL::row_imm(ks);
                qB[g][ks] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(at);
                doB[g][ks] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(at + NW * TL::BYTES);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
            barrier_only();                              // every wave has its rows: the slots may be filled
            request_first();
        } else {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int64_t off = ((int64_t)t * Hq + hq) * dr + 16 * ks + 8 * h;
                const bool there = row_ok && (HAS_IDX || 2 * ks + h < chunks);
                qB[g][ks] = there ? load_bf16x8(q + off) : zero_bf16x8();
                doB[g][ks] = there ? load_bf16x8(dout + off) : zero_bf16x8();
            }
        }
        neg_lse2[g] = -lse[(int64_t)hq * T + t] * LOG2E_F;
        // delta = rowsum(dO * O) of the lane's row: read, or - when every query row of the launch belongs to this kernel -
        // formed here from the dO row the lane already holds and written out for the key-side pass (one launch and one
        // pass over dO and O less)
        float dlt;
        if (out_for_delta) {                             // (kernel argument: the same for every wave)
            // the order of delta_row, so that both give the same bits: chain j of this lane covers the 8-element chunks 2*ks+h with
            // ks = j, j+8, ... (its lane 2*j+h), then its butterfly over 16 lanes - the three steps between lanes of one parity
            // here, the last one across the lane pair
            float p[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                p[c] = 0.f;
#pragma unroll
                for (int ks = c; ks < KS; ks += 8) {
                    const int64_t off = ((int64_t)t * Hq + hq) * dr + 16 * ks + 8 * h;
                    const bf16x8 o8 = row_ok && (HAS_IDX || 2 * ks + h < chunks) ? load_bf16x8(out_for_delta + off) : zero_bf16x8();
                    p[c] = dot8_chain(doB[g][ks], o8, p[c]);
                }
            }
            dlt = half_sum_f(((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7])));
            if (row_ok && h == 0) delta_out[(int64_t)hq * T + t] = dlt;
        } else {
            dlt = delta[(int64_t)hq * T + t];
        }
#pragma unroll
        for (int vi = 0; vi < 16; ++vi) dneg[g][vi] = -dlt;
    }
    f32x16 acc[RG][DT];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            acc[g][dt] = zero16();
            settle(acc[g][dt]);
        }
        asm volatile("" : "+v"(dneg[g]));                // (one tuple: the compiler would form it again in front of every chain)
    }
    lds_u8 *aR[4], *aT[4];                               // operand addresses: row-wise of K(0), transposed of K(t)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aR[i] = (lds_u8 *)dyn_lds + tl.rowq[i];
            aT[i] = (lds_u8 *)dyn_lds + tl.trq[i] + K_END - TL::BYTES;
        }
    }
    const unsigned char *const words = dyn_lds + V_END + wv * 1024 + j * 4;
    wait_vmcnt<0>();
    barrier_only();

    auto fence = [&]() __attribute__((always_inline)) {
        asm volatile("" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto row_op = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(aR[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto tr_op = [&](int i) __attribute__((always_inline)) {              // MFMA i of dQ: keys of half i / DT, d-tile i % DT
        const int pair = i / DT, dt = tile_of(i % DT);
        return tr_pair(aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair), aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair + 1));
    };
    auto advance = [&](lds_u8 *(&a)[4], int by) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] += by;
            asm volatile("" : "+v"(a[i]));
        }
    };
    // byte offsets of the slots: K(t), K(t+2), K(t+4); V(t+1), V(t+3)
    int kT = K_END - TL::BYTES, kR = TL::BYTES, kQ = 3 * TL::BYTES, vR = K_END, vQ = K_END + 2 * TL::BYTES;      // (t = -1)
    auto next_slot = [](int x, int end, int begin) __attribute__((always_inline)) { return x + TL::BYTES == end ? begin : x + TL::BYTES; };

    f32x16 snew[RG];                                     // S(t+1)
    uint32_t ds[RG][8];                                  // dS(t) in bf16
    bf16x8 op[AHEAD];
    // S(0)
#pragma unroll
    for (int g = 0; g < RG; ++g) snew[g] = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const bf16x8 a = row_op(ks);
#pragma unroll
        for (int g = 0; g < RG; ++g) snew[g] = mfma32(a, qB[g][ks], snew[g]);
    }
    advance(aR, vR);
    // Step t: phase B = dQ(t) and dP(t+1), behind them P(t+1); phase A = S(t+2), behind it dS(t+1).  MASK: tile t+1 needs its mask.
    auto step = [&](auto mask_, auto cur_, auto next_, int t) __attribute__((always_inline)) {
        constexpr bool MASK = decltype(mask_)::value, CUR = decltype(cur_)::value, NEXT = decltype(next_)::value;
        constexpr int PRE = !CUR ? 0 : NP < 4 ? NP : 4;
        typedef PhaseOrder<NEXT ? KS : 0, CUR ? NP : 0, PRE> PO;
        constexpr int NB = PO::M, M = NB + (NEXT ? KS : 0), SB = RG * NB, SA = RG * KS, E = 16 * RG;
        const int kT1 = next_slot(kT, K_END, 0), kR1 = next_slot(kR, K_END, 0), vR1 = next_slot(vR, V_END, K_END);
        auto fetch = [&](int m) __attribute__((always_inline)) {          // operand m of the step; from M on: of the next step
            if (m == M) advance(aT, kT1 - kT);
            if (m >= M) return tr_op(m - M);
            if (m == NB) advance(aR, kR - vR);
            if (m >= NB) return row_op(m - NB);
            return PO::is_row(m) ? row_op(PO::index(m)) : tr_op(PO::index(m));
        };
        if (!CUR) {
#pragma unroll
            for (int m = 0; m < AHEAD; ++m) op[m] = fetch(m);
        }
        // Operands in pairs: one wait in front of two of them, both refilled behind the second (a wait takes an issue slot)
        static_assert(M % 2 == 0, "");
        auto pair = [&](int m) __attribute__((always_inline)) {
            if (RG == 2 && m % 2 == 0) asm volatile("" : "+v"(op[m % AHEAD]), "+v"(op[(m + 1) % AHEAD]));
        };
        auto refill = [&](int m) __attribute__((always_inline)) {
            if (RG == 2 && m % 2 == 0) return;
#pragma unroll
            for (int x = RG == 2 ? m - 1 : m; x <= m; ++x)
                if (x + AHEAD < M || NEXT) op[x % AHEAD] = fetch(x + AHEAD);
        };
        uint32_t word[RG];
        if (NEXT && MASK) {
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                const uint32_t w = HAS_IDX ? *reinterpret_cast<const uint32_t *>(words + ((t + 1) & 3) * 256 + g * 128) & row_mask[g]
                                           : causal_bits(klim[g] - (t + 1) * 32);
                word[g] = w >> (4 * h);                  // element vi then sits at bit 8*(vi/4) + vi%4
            }
        }
        // ---- B ----
        float y[E];
        f32x16 dp[RG], s2[RG];
        constexpr int SP = SB - 2;                       // logits behind MFMA 1 + u, P behind the next
#pragma unroll
        for (int m = 0; m < NB; ++m) {
            pair(m);
#pragma unroll
            for (int g = 0; g < RG; ++g) {
                const int i = PO::index(m), n = m * RG + g, u = n - 1;
                if (PO::is_row(m)) {
                    dp[g] = mfma32(op[m % AHEAD], doB[g][i], i == 0 ? dneg[g] : dp[g]);
                } else {
                    const u32x4 w = {ds[g][4 * (i / DT)], ds[g][4 * (i / DT) + 1], ds[g][4 * (i / DT) + 2], ds[g][4 * (i / DT) + 3]};
                    mfma32_agpr(acc[g][i % DT], op[m % AHEAD], __builtin_bit_cast(bf16x8, w), !NEXT);
                }
                if (g == RG - 1) refill(m);
                if (NEXT) {
                    if (n == 1) load_tile(kptr, t + 4, kQ);
                    if (n == SB / 3) load_tile(vptr, t + 3, vQ);
                    if (n == 2 * SB / 3) load_w(t + 3);
                }
                if (NEXT && u >= 0) {
#pragma unroll
                    for (int e = E * u / SP; e < E * (u + 1) / SP; ++e) {
                        if (e >= E) continue;
                        const int ge = e / 16, vi = e % 16;
                        const float x = fmaf(snew[ge][vi], scale_log2, neg_lse2[ge]);
                        y[e] = MASK ? keep_or_neginf(x, bit_mask(word[ge], 8 * (vi >> 2) + (vi & 3))) : x;
                        asm volatile("" : "+v"(y[e]));
                    }
#pragma unroll
                    for (int e = E * (u - 1) / SP; u >= 1 && e < E * u / SP; ++e) {
                        y[e] = fast_exp2(y[e]);
                        asm volatile("" : "+v"(y[e]));
                    }
                }
                fence();
            }
        }
        // ---- A ----
        if (NEXT) {
            constexpr int SS = SA - 2;                   // products behind MFMA 1 + u, packed behind the next
#pragma unroll
            for (int m = 0; m < KS; ++m) {
                pair(NB + m);
#pragma unroll
                for (int g = 0; g < RG; ++g) {
                    const int n = m * RG + g, u = n - 1, mm = NB + m;
                    s2[g] = mfma32(op[mm % AHEAD], qB[g][m], m == 0 ? zero16() : s2[g]);
                    if (g == RG - 1) refill(mm);
                    if (u >= 0) {
#pragma unroll
                        for (int e = E * u / SS; e < E * (u + 1) / SS; ++e) {
                            if (e >= E) continue;
                            y[e] *= dp[e / 16][e % 16];
                            asm volatile("" : "+v"(y[e]));
                        }
#pragma unroll
                        for (int e = E * (u - 1) / SS; u >= 1 && e < E * u / SS; ++e)
                            if (e % 2) {
                                ds[e / 16][e % 16 / 2] = pack2bf(y[e - 1], y[e]);
                                asm volatile("" : "+v"(ds[e / 16][e % 16 / 2]));
                            }
                    }
                    fence();
                }
            }
#pragma unroll
            for (int g = 0; g < RG; ++g) snew[g] = s2[g];
            if (M % AHEAD) {
                bf16x8 o[AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) o[i] = op[(M + i) % AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) op[i] = o[i];
            }
            advance(aR, vR1 - kR);
            kT = kT1;
            kR = kR1;
            kQ = next_slot(kQ, K_END, 0);
            vR = vR1;
            vQ = next_slot(vQ, V_END, K_END);
            wait_vmcnt<LPS>();                           // all but what this step requested
            barrier_only();
        }
    };
    const std::true_type yes;
    const std::false_type no;
    step(yes, no, yes, -1);
    int t = 0;
    {                                                    // tiles that every row of the block attends whole: no mask arithmetic
        const int whole = (HAS_IDX && min(qc0 + QBW, L) > window ? 0 : causal ? qc0 + 1 : L) / 32;
        for (; t + 1 < whole; ++t) step(no, yes, yes, t);     // (rows that do not exist may turn to NaN: a row is one lane's)
    }
    for (; t + 1 < ntiles; ++t) step(yes, yes, yes, t);
    step(yes, yes, no, t);
    wait_vmcnt<0>();                                     // no load is left on its way into LDS

    // whole rows per store, through LDS (as in the key-side kernel)
    barrier_only();                                      // the ring is read out
    unsigned char *const rows_out = dyn_lds + wv * (RG * 32 * TL::ROW_B);
    auto chunk_at = [&](int row, int c) __attribute__((always_inline)) {
        return row * TL::ROW_B + ((c ^ (D == 64 ? (row >> 1) & 7 : row & 15)) << 4);
    };
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            f32x16 &a = acc[g][dt];
            settle(a);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t a0 = pack2bf(a[8 * i] * scale, a[8 * i + 1] * scale), a1 = pack2bf(a[8 * i + 2] * scale, a[8 * i + 3] * scale);
                const uint32_t b0 = pack2bf(a[8 * i + 4] * scale, a[8 * i + 5] * scale), b1 = pack2bf(a[8 * i + 6] * scale, a[8 * i + 7] * scale);
                const auto x0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
                const auto x1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
                *reinterpret_cast<u32x4 *>(rows_out + chunk_at(32 * g + j, 4 * tile_of(dt) + 2 * i + h)) = u32x4{x0[0], x1[0], x0[1], x1[1]};
            }
        }
    // (a group's rows read in front of its first store: a read and its store in turn would wait for the LDS each time)
    const WaveRows<TL> wr(gshift, lane);
    const int q0 = qc0 + (r0 >> gshift), to_tok = Hq * dr * 2, c = lane % TL::CPR, place = wr.place(to_tok, dr * 2) + c * 16;
    unsigned char *const to = reinterpret_cast<unsigned char *>(dq + ((int64_t)(s0 + q0) * Hq + kvh * G) * dr);
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        u32x4 x[TL::LOADS];
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i) x[i] = *reinterpret_cast<const u32x4 *>(rows_out + chunk_at(32 * g + i * TL::LOAD_ROWS + lane / TL::CPR, c));
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i)
            if (q0 + wr.query(i, 32 * g) < L && wr.head(i, 32 * g) < G && (CARRIED ? carried_chunk(c, true) : c < chunks))
                *reinterpret_cast<u32x4 *>(to + (place + wr.piece(i, to_tok, dr * 2, 32 * g))) = x[i];
    }
}
