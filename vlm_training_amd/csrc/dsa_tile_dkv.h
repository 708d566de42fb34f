// dK, dV over 32x32 MFMA tiles, key-stationary ("scatter by key": every key row is reduced by one wave, in a fixed query order - or,
// when the launch cuts the walk into pieces, by one wave per piece and a sum over the pieces in piece order - so the result needs no
// atomics and is bit-reproducible).  A workgroup owns a 128-key tile of one segment and kv head and walks the later queries in blocks
// of 32 (query, head) rows, from the end of the segment down to the key tile: workgroups that run side by side then read the same
// q / dO rows at about the same time and share them in L2.
//   S = Q K^T, dP = dO V^T          (A = q / dO block row-wise from LDS, B = the wave's K / V rows in registers; the sums start from
//                                    -lse/scale and -delta, so that P = exp2(S * scale*log2e) and dS = P dP need no subtraction)
//   dV^T += dO^T P, dK^T += Q^T dS  (A = the blocks transposed, B = P / dS from the C layout)
// One wave per SIMD, each with all four chains of its keys and 512 registers: 64 keys up to head_dim 128 (two waves a workgroup, two
// workgroups a CU), 32 keys at head_dim 256 and in launches of little work (four waves, one workgroup: dkv_key_groups).  The sums of
// dK and dV fill up to 256 accumulation registers, K and V rows 128 of the others.  An operand read from LDS feeds the MFMAs of both key groups, P and dS never leave
// the wave, nothing is formed twice.  Step s runs dV(s) mixed with S(s+1), the products of dS(s) behind them, then dK(s) mixed with
// dP(s+1), P(s+1) behind them in three stages (logit, exponential, packing) that do not wait for each other.  P stays in fp32 until dS is
// formed (from its bf16 form dK is 3.0e-3 off 64 bits instead of 2.5e-3, and unpacking that is another 32 instructions).  q and dO blocks, row
// data and selection words go from memory straight into LDS, two to three steps ahead, one barrier per step.
//
// What bounds it: the issue of one instruction stream per SIMD - at head_dim 128 64 MFMAs (2048 clocks) beside about 160 vector
// instructions (210 with a selection), 60 LDS reads and as many scalar ones take 3000 - and the chip's power (MFMA busy 0.69 of a CU's
// time, 1.85 GHz under this load).  Same box, us, against the kernels before (eight waves; at head_dim 128 one wave per chain, P handed
// over in LDS; at 256 each half of head_dim formed S and dP; q and dO through registers): 32 768 tokens dense 2630 -> 2200, with a
// selection 2680 -> 2240; head_dim 256, 16 384 tokens in short segments 548 -> 327 (in finer pieces 309); towers at head_dim 64 / 72, whole backward
// 553 -> 440 / 1131 -> 976; one segment of 4096 / 12 288 tokens 451 -> 300 / 2430 -> 2000.  32 keys per wave at head_dim 128: 2440
// dense, each operand read feeding one MFMA, but a walk's step 1600 instead of 3000 clocks: 1000 tokens, forward and backward, 118 -> 99
// (64 keys: 124).
#pragma once
#include "dsa_tile.h"

// KG: groups of 32 keys per wave
template <int D, int KG> constexpr int dkv_ring() { return D == 128 && KG == 1 ? 8 : 4; }                // q/dO blocks in LDS
template <int D, int KG> constexpr int dkv_aux_bytes() { return dkv_ring<D, KG>() * 512 + 512 + (D == 128 && KG == 2 ? 5120 : 0); }
template <int D, int KG> constexpr size_t dkv_lds_bytes() {
    return dkv_ring<D, KG>() * 2 * (size_t)DirectTile<D>::BYTES + 4 / KG * (size_t)dkv_aux_bytes<D, KG>();
}
// One workgroup of a launch, number `block`: as a function for the launch that holds both passes (DKV_AS_FUNCTION), else as the kernel it
// is (called from one, the instance of two heads per kv head without a selection reads a spilled operand in its loop).
template <int D, int KG, bool HAS_IDX, int GSHIFT, bool UNALIGNED, bool CARRIED>
#ifdef DKV_AS_FUNCTION
__device__ __forceinline__ void dkv_block(int block,
#else
__global__ __launch_bounds__(256 / KG, 1) void dsa_tile_dkv_kernel(
#endif
    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k,
    const bf16_t *__restrict__ v, const float *__restrict__ lse, const float *__restrict__ delta,
    const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv,
    float scale, float logit_scale, int causal, int d_real, int skip_len, const int32_t *__restrict__ order, float *__restrict__ partial, bf16_t *__restrict__ dk,
    bf16_t *__restrict__ dv) {
#ifndef DKV_AS_FUNCTION
    const int block = blockIdx.x;
#endif
    typedef DirectTile<D> TL;
    constexpr int RING = dkv_ring<D, KG>(), NW = 4 / KG;
    constexpr int KS = CARRIED ? DSA_CARRIED_KS : D / 16, DT = CARRIED ? 4 : (D + 31) / 32, NP = 2 * DT;
    auto tile_of = [](int dt, bool of_v) __attribute__((always_inline)) { return CARRIED && of_v ? carried_tile(dt) : dt; };
    constexpr int LPW = TL::LOADS / NW, LPS = 2 * LPW + (HAS_IDX ? 2 : 1);
    constexpr int Gp = 1 << GSHIFT, QB = 32 >> GSHIFT;
    constexpr int RPW = Gp < 4 ? Gp : 4;                 // neighbouring rows of a lane that are one query's
    constexpr int SLOT = 2 * TL::BYTES;                  // q block | dO block
    // LDS of a wave: RING x (lse, delta | selection words), 2 x row data as the chains start from it, and at head_dim 128, where the
    // loop has no registers left for them, the lane's source offsets and the last K and V operand of each key group
    constexpr int AUX = dkv_aux_bytes<D, KG>();
    constexpr bool TIGHT = D == 128 && KG == 2;
    constexpr int AHEAD = TIGHT ? 2 : 4;                 // operands read ahead: four MFMAs or more
    constexpr bool PAIRS = KG == 2 && !TIGHT;            // operands waited for and refilled in pairs
    static_assert(TL::LOADS % NW == 0 && (RING & (RING - 1)) == 0 && AHEAD <= NP, "");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv;
    const int dr = HAS_IDX || CARRIED ? D : d_real, chunks = CARRIED ? 2 * KS : dr / 8;   // elements and 16-byte chunks of a row in memory
    const int kvh = block % Hkv;
    int s0, L, blk, piece, mslot, pb;
    if (!locate_key_tile(order, cu, N, block / Hkv, s0, L, blk, piece, mslot, pb)) return;
    if (HAS_IDX) L = min(L, ldw * 32);                   // a bitmap row has ldw words whatever the caller's max_seqlen
    if (blk * 128 >= L || (HAS_IDX && L >= skip_len)) return;     // (whole workgroup, before its first barrier; long segments may be the compacted walk's)
    const int c0 = blk * 128, kc = c0 + wv * 32 * KG;    // the wave's first key
    const float scale_log2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(logit_scale * LOG2E_F))), inv_scale = 1.f / logit_scale;
    // the walk: queries q0 .. Lq-1 in nblocks steps (step s handles block nblocks-1-s) - all queries that can see this key tile, or
    // one piece of them
    int q0_ = causal ? c0 : 0, Lq_ = L, nblocks_ = (L - q0_ + QB - 1) / QB;
    const int npieces = walk_piece((causal && partial && mslot >= 0) ? pb / QB : 0, piece, QB, q0_, Lq_, nblocks_);
    if (npieces == 0) return;
    const int q0 = q0_, Lq = Lq_, nblocks = nblocks_, last = nblocks - 1;
    const int over_rows = q0 + nblocks * QB - Lq;        // queries of step 0's block that do not exist

    // ---- requests ----
    const int tok_b = Hq * dr * 2;                       // bytes from one query to the next
    const int64_t q_first = (int64_t)(s0 + q0 + last * QB);
    const unsigned char *qptr = reinterpret_cast<const unsigned char *>(q + (q_first * Hq + kvh * G) * dr);
    const unsigned char *dptr = reinterpret_cast<const unsigned char *>(dout + (q_first * Hq + kvh * G) * dr);
    int voff[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const int row = (wv * LPW + i) * TL::LOAD_ROWS + lane / TL::CPR, c = (lane % TL::CPR) ^ TL::xor_of(row);
        const int hd = row & (Gp - 1);
        voff[i] = hd < G && c < chunks ? (row >> GSHIFT) * tok_b + hd * dr * 2 + c * 16 : (int)0x80000000;
    }
    const uint32_t lds0 = lds_address(dyn_lds);
    unsigned char *const aux = dyn_lds + RING * SLOT + wv * AUX;
    const uint32_t aux0 = lds0 + RING * SLOT + wv * AUX;
    if constexpr (TIGHT) *reinterpret_cast<u32x4 *>(aux + RING * 512 + 512 + lane * 16) = u32x4{(uint32_t)voff[0], (uint32_t)voff[1], (uint32_t)voff[2], (uint32_t)voff[3]};
    const int full_b = (QB - 1) * tok_b + G * dr * 2, first_b = full_b - over_rows * tok_b;
    const int64_t blk_b = (int64_t)QB * tok_b;
    auto block_bytes = [&](int b) __attribute__((always_inline)) { return b > last ? 0 : b == 0 ? first_b : full_b; };
    // the wave's pieces of q (or dO) of block b; called in turn.  Rows past the walk and columns past the true head_dim read as zero.
    auto load_tile = [&](const int (&voff)[LPW], const unsigned char *&p, int b, int tile, uint32_t bytes) __attribute__((always_inline)) {
        if (UNALIGNED) bytes = 0u;
        constexpr int P1 = LPW > 1 ? 1 : 0, P2 = LPW > 2 ? 2 : P1, P3 = LPW > 2 ? 3 : P2;
        buffer_load_lds16_n<LPW, TL::load_lds(P1), TL::load_lds(P2) - TL::load_lds(P1), TL::load_lds(P3) - TL::load_lds(P2)>(
            scalar_buffer_rsrc(p, bytes), voff, lds0 + (b & (RING - 1)) * SLOT + tile * TL::BYTES + TL::load_lds(wv * LPW));
        p -= blk_b;
        asm volatile("" : "+s"(p));
    };
    // UNALIGNED: q or dO on no 16-byte boundary.  The requests read nothing, and the pieces of a block come through registers, here.
    auto copy_block = [&](int b) __attribute__((always_inline)) {
        wait_vmcnt<0>();                                 // what the requests of this block wrote is there
#pragma unroll 1
        for (int x = 0; x < 2 * LPW; ++x) {
            const int i = x % LPW, row = (wv * LPW + i) * TL::LOAD_ROWS + lane / TL::CPR, c = (lane % TL::CPR) ^ TL::xor_of(row), hd = row & (Gp - 1);
            const unsigned char *base = reinterpret_cast<const unsigned char *>((x < LPW ? q : dout) + (q_first * Hq + kvh * G) * dr) - b * blk_b;
            const int off = (row >> GSHIFT) * tok_b + hd * dr * 2 + c * 16;
            u32x4 w = {0u, 0u, 0u, 0u};
            if (hd < G && c < chunks && off < block_bytes(b)) w = *reinterpret_cast<const u32x4 *>(base + off);
            *reinterpret_cast<u32x4 *>(dyn_lds + (b & (RING - 1)) * SLOT + x / LPW * TL::BYTES + TL::load_lds(wv * LPW + i) + lane * 16) = w;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    };
    const unsigned char *rp, *wp = nullptr;              // this lane's row data and selection word of the block requested next
    const int rhead = lane & (Gp - 1);
    const int rq = (lane & 31) >> GSHIFT, wq = lane % QB;
    {
        const float *base = (lane < 32 ? lse : delta) + (int64_t)(kvh * G + min(rhead, G - 1)) * T + s0;
        rp = reinterpret_cast<const unsigned char *>(base + min(q0 + last * QB + rq, Lq - 1));
        if (HAS_IDX) {
            const int col = min((kc >> 5) + (lane / QB) % KG, ldw - 1);
            wp = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + min(q0 + last * QB + wq, Lq - 1)) * ldw + col);
        }
    }
    const int64_t w_step = (int64_t)QB * ldw * 4;
    auto load_rows = [&](int b) __attribute__((always_inline)) {
        global_load_lds4(rp, aux0 + (b & (RING - 1)) * 512);
        rp -= b < last ? 4 * QB : 0;
        asm volatile("" : "+v"(rp));
    };
    auto load_words = [&](int b) __attribute__((always_inline)) {
        if (HAS_IDX) {
            global_load_lds4(wp, aux0 + (b & (RING - 1)) * 512 + 256);
            wp -= b < last ? w_step : 0;
            asm volatile("" : "+v"(wp));
        }
    };
    bf16x8 kB[KG][KS], vB[KG][KS];
    TL tl;
    tl.init(lane);
    // The wave's rows of k and v (past the segment its last one) come in whole rows through eight slots of the ring, in front of the blocks (as q
    // and dO in dQ)
    if constexpr (!UNALIGNED) {
        const int first = min(kc, L - 1), kv_b = Hkv * dr * 2;
        const int64_t base = ((int64_t)(s0 + first) * Hkv + kvh) * dr;
        const buffer_rsrc k_rows = make_buffer_rsrc(k + base, 0x7fffffff), v_rows = make_buffer_rsrc(v + base, 0x7fffffff);
#pragma unroll
        for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int i = 0; i < TL::LOADS; ++i) {
                const int row = i * TL::LOAD_ROWS + lane / TL::CPR, c = (lane % TL::CPR) ^ TL::xor_of(row);
                const int off[1] = {c < chunks ? (min(kc + 32 * g + row, L - 1) - first) * kv_b + c * 16 : (int)0x80000000};
                buffer_load_lds16_n<1, 0, 0, 0>(k_rows, off, lds0 + (wv * KG + g) * TL::BYTES + TL::load_lds(i));
                buffer_load_lds16_n<1, 0, 0, 0>(v_rows, off, lds0 + (4 + wv * KG + g) * TL::BYTES + TL::load_lds(i));
            }
        wait_vmcnt<0>();                                 // (the wave's own pieces)
#pragma unroll
        for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                lds_u8 *const at = (lds_u8 *)dyn_lds + (wv * KG + g) * TL::BYTES + tl.rowq[TL::row_q(ks)] + TL::row_imm(ks);
                kB[g][ks] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(at);
                vB[g][ks] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(at + 4 * TL::BYTES);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        barrier_only();                                  // every wave has its rows: the slots may be filled
    } else {
#pragma unroll
        for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int64_t at = ((int64_t)(s0 + min(kc + 32 * g + j, L - 1)) * Hkv + kvh) * dr + 16 * ks + 8 * h;
                const bool there = HAS_IDX || 2 * ks + h < chunks;
                kB[g][ks] = there ? load_bf16x8(k + at) : zero_bf16x8();
                vB[g][ks] = there ? load_bf16x8(v + at) : zero_bf16x8();
            }
    }
    load_rows(0);
    load_words(0);
    if (last > 0) {                                      // leaving block 0: undo its clamps
        rp += 4 * max(q0 + last * QB + rq - (Lq - 1), 0);
        if (HAS_IDX) wp += (int64_t)max(q0 + last * QB + wq - (Lq - 1), 0) * ldw * 4;
    }
#pragma unroll
    for (int b = 0; b < RING - 2; ++b) {
        load_tile(voff, qptr, b, 0, block_bytes(b));
        load_tile(voff, dptr, b, 1, block_bytes(b));
        load_rows(b + 1);
        load_words(b + 1);
    }
    unsigned char *const klast = aux + RING * 512 + 1536 + lane * 16, *const vlast = klast + 2048;
#pragma unroll
    for (int g = 0; g < KG; ++g)
        if (TIGHT) {
            *reinterpret_cast<bf16x8 *>(klast + g * 1024) = kB[g][KS - 1];
            *reinterpret_cast<bf16x8 *>(vlast + g * 1024) = vB[g][KS - 1];
        }
    f32x16 dkacc[KG][DT], dvacc[KG][DT];
#pragma unroll
    for (int g = 0; g < KG; ++g)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            dkacc[g][dt] = zero16();
            dvacc[g][dt] = zero16();
            settle(dkacc[g][dt]);                        // (cleared here, not in front of the first MFMA)
            settle(dvacc[g][dt]);
        }
    wait_vmcnt<0>();
    if (UNALIGNED)
        for (int b = 0; b < RING - 2; ++b) copy_block(b);
    barrier_only();

    // Row data of block b as the chains start from it: -lse/scale and -delta; rows that do not exist get values that make P and dS vanish
    const float row_mul = lane < 32 ? -inv_scale : -1.f;
    const bool dead_pad = rhead >= G;
    unsigned char *const rows_raw = aux + lane * 4, *const rows_st = aux + RING * 512 + lane * 4;
    const unsigned char *const rows_in = aux + RING * 512 + 16 * h, *const words_in = aux + 256;
    auto raw_row = [&](int b) __attribute__((always_inline)) { return *reinterpret_cast<const float *>(rows_raw + (b & (RING - 1)) * 512); };
    auto put_row = [&](int b, float x, bool dead) __attribute__((always_inline)) {
        float low = __int_as_float(__float_as_int(-1e30f) ^ (__float_as_int(logit_scale) & (int)0x80000000));
        asm volatile("" : "+s"(low));                    // (the choice is made here, not kept in a register over the loop)
        *reinterpret_cast<float *>(rows_st + (b & 1) * 256) = dead ? (lane < 32 ? low : 0.f) : x * row_mul;
    };
    auto rows_init = [&](int b, int part) __attribute__((always_inline)) {
        f32x16 c;
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const f32x4 r = *reinterpret_cast<const f32x4 *>(rows_in + (b & 1) * 256 + part * 128 + 32 * g4);
#pragma unroll
            for (int e = 0; e < 4; ++e) c[4 * g4 + e] = r[e];
        }
        return c;
    };
    put_row(0, raw_row(0), dead_pad || q0 + last * QB + rq >= Lq);
    put_row(1, raw_row(1), dead_pad);

    constexpr float DKV_SPLIT_MIN = 0.015625f;
    f32x16 pacc[KG];                                     // dP of the block ahead
    uint32_t pw[KG][8];                                  // its P in bf16
    float pf[KG][16];                                    // and in fp32, for dS
    bf16x8 op[AHEAD];
    lds_u8 *aR[4], *aT[4];                               // operand addresses: row-wise of block s+1, transposed of block s
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aR[i] = (lds_u8 *)dyn_lds + tl.rowq[i];
            aT[i] = (lds_u8 *)dyn_lds + tl.trq[i] + (RING - 1) * SLOT;
        }
    }
    auto fence = [&]() __attribute__((always_inline)) {
        asm volatile("" : : : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto row_op = [&](int ks, int off) __attribute__((always_inline)) {
        return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(aR[TL::row_q(ks)] + TL::row_imm(ks) + off);
    };
    auto tr_op = [&](int i, int off) __attribute__((always_inline)) {
        const int pair = i / DT, dt = tile_of(i % DT, off != 0);   // (off: the operand is of dO)
        return tr_pair(aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair) + off, aT[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair + 1) + off);
    };
    const int jb = 31 - j, key_bias = (causal ? 0 : 0x40000000) - kc - 31;      // key_bias + jb = bias - the lane's first key
    // Step s: phase X = dV(s) and S(s+1), behind them dS(s); phase Y = dK(s) and dP(s+1), behind them P(s+1).
    auto step = [&](auto diag_, auto cur_, auto next_, int s) __attribute__((always_inline)) {
        constexpr bool DIAG = decltype(diag_)::value, CUR = decltype(cur_)::value, NEXT = decltype(next_)::value;
        constexpr int PRE = !CUR ? 0 : NP < 4 ? NP : 4;
        typedef PhaseOrder<NEXT ? KS : 0, CUR ? NP : 0, PRE> PO;
        constexpr int NX = PO::M, M = 2 * NX, SL = KG * NX;
        const int adv = ((s + 1) & (RING - 1)) ? SLOT : -(RING - 1) * SLOT;      // from the slot of block s to that of s+1
        auto fetch = [&](int m) __attribute__((always_inline)) {          // operand m of the step; from M on: of the next step
            if (m == M) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    aT[i] += adv;
                    asm volatile("" : "+v"(aT[i]));
                }
            }
            if (m >= M) return tr_op(m - M, TL::BYTES);
            const bool x = m < NX;
            const int i = x ? m : m - NX;
            if (PO::is_row(i)) return row_op(PO::index(i), x ? 0 : TL::BYTES);
            return tr_op(PO::index(i), x ? TL::BYTES : 0);
        };
        if (!CUR) {
#pragma unroll
            for (int m = 0; m < AHEAD; ++m) op[m] = fetch(m);
        }
        // Operands in pairs where registers allow: one wait in front of two of them, both refilled behind the second (a wait takes an
        // issue slot)
        auto pair = [&](int m) __attribute__((always_inline)) {
            if (PAIRS && m % 2 == 0) asm volatile("" : "+v"(op[m % AHEAD]), "+v"(op[(m + 1) % AHEAD]));
        };
        auto refill = [&](int m) __attribute__((always_inline)) {
            if (PAIRS && m % 2 == 0) return;
#pragma unroll
            for (int x = PAIRS ? m - 1 : m; x <= m; ++x)
                if (x + AHEAD < M || NEXT) op[x % AHEAD] = fetch(x + AHEAD);
        };
        f32x16 snew[KG], pnew[KG];
        int vo[LPW];
        if (NEXT) {
            if (TIGHT) {                              // (kept in LDS: the loop has no registers left for them)
                const u32x4 x = *reinterpret_cast<const u32x4 *>(aux + RING * 512 + 512 + lane * 16);
#pragma unroll
                for (int i = 0; i < LPW; ++i) vo[i] = x[i];
            } else {
#pragma unroll
                for (int i = 0; i < LPW; ++i) vo[i] = voff[i];
            }
#pragma unroll
            for (int g = 0; g < KG; ++g) snew[g] = rows_init(s + 1, 0);
        }
        // ---- X ----
        bf16x8 kl[KG], vl[KG];
        uint32_t dw[KG][8];
        float dsv[2 * KG * 16];
        constexpr int E = 16 * KG, SX = SL - 2;          // dS: product behind MFMA 1 + u, packed behind the next
#pragma unroll
        for (int m = 0; m < NX; ++m) {
            pair(m);
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                const int i = PO::index(m), n = m * KG + g, u = n - 1;
                if (PO::is_row(m)) {
                    snew[g] = mfma32(op[m % AHEAD], TIGHT && i == KS - 1 ? kl[g] : kB[g][i], snew[g]);
                } else {
                    const u32x4 w = {pw[g][4 * (i / DT)], pw[g][4 * (i / DT) + 1], pw[g][4 * (i / DT) + 2], pw[g][4 * (i / DT) + 3]};
                    mfma32_agpr(dvacc[g][i % DT], op[m % AHEAD], __builtin_bit_cast(bf16x8, w), !NEXT);
                }
                if (g == KG - 1) refill(m);
                if (NEXT) {
                    if (n == 1) load_tile(vo, qptr, s + RING - 1, 0, s + RING - 1 <= last ? full_b : 0);
                    if (n == SL / 4) load_tile(vo, dptr, s + RING - 1, 1, s + RING - 1 <= last ? full_b : 0);
                    if (n == SL / 2) load_rows(s + RING);
                    if (n == 3 * SL / 4) load_words(s + RING);
                }
                if (TIGHT && m == NX - 3) kl[g] = *reinterpret_cast<const bf16x8 *>(klast + g * 1024);
                if (CUR && u >= 0) {
#pragma unroll
                    for (int e = E * u / SX; e < E * (u + 1) / SX; ++e) {
                        if (e >= E) continue;
                        const int ge = e / 16, vi = e % 16;
                        dsv[e] = pf[ge][vi] * pacc[ge][vi];
                        asm volatile("" : "+v"(dsv[e]));
                    }
#pragma unroll
                    for (int e = E * (u - 1) / SX; u >= 1 && e < E * u / SX; ++e)
                        if (e % 2) {
                            dw[e / 16][e % 16 / 2] = pack2bf(dsv[e - 1], dsv[e]);
                            asm volatile("" : "+v"(dw[e / 16][e % 16 / 2]));
                        }
                }
                fence();
            }
        }
        // ---- Y ----
        float raw;
        uint32_t mw[KG][16];
        auto words = [&](int e) __attribute__((always_inline)) {          // selection words of elements e .. e+3
            const int ge = e / 16, g4 = e % 16 / 4;
            const unsigned char *p = words_in + ((s + 1) & (RING - 1)) * 512 + ge * QB * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i % RPW == 0) mw[ge][4 * g4 + i] = *reinterpret_cast<const uint32_t *>(p + 4 * ((8 * g4 + 4 * h + i) >> GSHIFT));
        };
        if (NEXT) {
#pragma unroll
            for (int g = 0; g < KG; ++g) pnew[g] = rows_init(s + 1, 1);
            if (HAS_IDX) words(0);
            raw = raw_row(s + 2);
        }
        const int qk = q0 + (last - (s + 1)) * QB + key_bias;      // + jb: first query of block s+1 minus the lane's first key
        uint32_t keep = 0u, pn[KG][8];
        float pm = 0.f, y[KG * 16];
        auto logit = [&](int e) __attribute__((always_inline)) {
            const int ge = e / 16, vi = e % 16;
            if ((HAS_IDX || DIAG) && vi % RPW == 0) {     // rows of one query share the mask bit
                keep = HAS_IDX ? (uint32_t)((int32_t)(mw[ge][vi] << jb) >> 31) : 0xffffffffu;
                if (DIAG) keep &= ~(uint32_t)((jb + (qk - 32 * ge) + ((8 * (vi / 4) + 4 * h + vi % 4) >> GSHIFT)) >> 31);
            }
            const float x = snew[ge][vi] * scale_log2;
            return HAS_IDX || DIAG ? keep_or_neginf(x, keep) : x;
        };
        constexpr int SY = SL - 3;                       // logits behind MFMA 1 + u, P behind the next, packed behind the one after
#pragma unroll
        for (int m = 0; m < NX; ++m) {
            pair(NX + m);
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                const int i = PO::index(m), n = m * KG + g, u = n - 1, mm = NX + m;
                if (PO::is_row(m)) {
                    pnew[g] = mfma32(op[mm % AHEAD], TIGHT && i == KS - 1 ? vl[g] : vB[g][i], pnew[g]);
                } else {
                    const u32x4 w = {dw[g][4 * (i / DT)], dw[g][4 * (i / DT) + 1], dw[g][4 * (i / DT) + 2], dw[g][4 * (i / DT) + 3]};
                    mfma32_agpr(dkacc[g][i % DT], op[mm % AHEAD], __builtin_bit_cast(bf16x8, w), !NEXT || (UNALIGNED && i >= DT));
                }
                if (g == KG - 1) refill(mm);
                if (TIGHT && m == NX - 3) vl[g] = *reinterpret_cast<const bf16x8 *>(vlast + g * 1024);
                if (NEXT && u >= 0) {
#pragma unroll
                    for (int e = E * u / SY; e < E * (u + 1) / SY; ++e) {
                        if (e >= E) continue;
                        if (HAS_IDX && e % 4 == 0 && e + 4 < E) words(e + 4);
                        y[e] = logit(e);
                        asm volatile("" : "+v"(y[e]));
                    }
#pragma unroll
                    for (int e = E * (u - 1) / SY; u >= 1 && e < E * u / SY; ++e) {
                        if (e >= E) continue;
                        y[e] = fast_exp2(y[e]);
                        asm volatile("" : "+v"(y[e]));
                    }
#pragma unroll
                    for (int e = E * (u - 2) / SY; u >= 2 && e < E * (u - 1) / SY; ++e)
                        if (e % 2) {
                            pm = fmaxf(fmaxf(pm, y[e - 1]), y[e]);
                            pn[e / 16][e % 16 / 2] = pack2bf(y[e - 1], y[e]);
                            asm volatile("" : "+v"(pn[e / 16][e % 16 / 2]), "+v"(pm));
                        }
                    if (n == SL / 2) put_row(s + 2, raw, dead_pad);
                }
                fence();
            }
        }
        if (NEXT) {
#pragma unroll
            for (int e = 0; e < E; ++e) pf[e / 16][e % 16] = y[e];
            // dV also takes what bf16 rounds off the larger probabilities: few keys per query and many rows in one key pile that
            // rounding up.  Wave-uniform and rare.
            if (__builtin_amdgcn_ballot_w64(pm >= DKV_SPLIT_MIN) != 0ull) {
#pragma unroll
                for (int g = 0; g < KG; ++g) {
                    float lo[16];
#pragma unroll
                    for (int vi = 0; vi < 16; ++vi) {
                        const uint32_t w = pn[g][vi >> 1];
                        lo[vi] = y[16 * g + vi] - __uint_as_float(vi & 1 ? w & 0xffff0000u : w << 16);
                    }
                    bf16x8 l0 = pack8(lo), l1 = pack8(lo + 8);
                    asm volatile("s_nop 1" : "+v"(l0), "+v"(l1));
#pragma unroll
                    for (int i = 0; i < NP; ++i) mfma32_agpr(dvacc[g][i % DT], tr_op(i, TL::BYTES), i < DT ? l0 : l1, i >= DT);
                }
            }
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                pacc[g] = pnew[g];
#pragma unroll
                for (int e = 0; e < 8; ++e) pw[g][e] = pn[g][e];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int adv2 = ((s + 2) & (RING - 1)) ? SLOT : -(RING - 1) * SLOT;
                aR[i] += adv2;
                asm volatile("" : "+v"(aR[i]));
            }
            if (M % AHEAD) {
                bf16x8 t[AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) t[i] = op[(M + i) % AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) op[i] = t[i];
            }
            if (UNALIGNED) copy_block(s + RING - 1);
            wait_vmcnt<(RING - 3) * LPS>();              // all but what the last RING - 3 steps requested
            barrier_only();
        }
    };
    const std::true_type yes;
    const std::false_type no;
    const int nb_diag = causal ? max(kc + 32 * KG - q0 + QB - 1, 0) / QB : 0;
    const int steady = max(nblocks - nb_diag, 1);        // blocks [1, steady) lie past the diagonal
    step(yes, no, yes, -1);
    int s = 0;
    if constexpr (!UNALIGNED)                            // (no loop of its own for the rare form)
        for (; s + 1 < steady; ++s) step(no, yes, yes, s);
    for (; s + 1 < nblocks; ++s) step(yes, yes, yes, s);
    step(yes, yes, no, s);
    wait_vmcnt<0>();                                     // no load is left on its way into LDS
    if (npieces > 1) {                                   // a piece of the walk: fp32 partial sums, added by the reduction
        constexpr int TD = (D + 31) / 32;
        float *const p = piece_partial(partial, mslot, piece, Hkv, kvh, TD);
#pragma unroll
        for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                settle(dkacc[g][dt]);
                settle(dvacc[g][dt]);
                store_c_tile_f32(p + ((wv * KG + g) * TD + dt) * 1024, dkacc[g][dt], lane);
                store_c_tile_f32(p + ((4 + wv * KG + g) * TD + tile_of(dt, true)) * 1024, dvacc[g][dt], lane);
            }
        return;
    }
    // Rows go out through LDS, whole rows per store (as the accumulators lie, a store would touch 32 rows, 32 bytes of each: 2 to 5 us
    // a workgroup).  16-byte chunk c of row r sits at c ^ x(r): sixteen rows at one chunk and the chunks of a row each cover the banks once.
    barrier_only();                                      // the ring is read out
    unsigned char *const rows_out = dyn_lds + wv * (2 * KG * 32 * TL::ROW_B);
    int lane_ = lane;                                    // (places are formed here: the loop needs its registers)
    asm volatile("" : "+v"(lane_));
    const int h_ = lane_ >> 5, j_ = lane_ & 31;
    auto chunk_at = [&](int row, int c) __attribute__((always_inline)) {
        return row * TL::ROW_B + ((c ^ (D == 64 ? (row >> 1) & 7 : row & 15)) << 4);
    };
#pragma unroll
    for (int g = 0; g < KG; ++g)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                f32x16 &acc = m ? dvacc[g][dt] : dkacc[g][dt];
                settle(acc);
                const float mul = m ? 1.f : scale;
#pragma unroll
                for (int i = 0; i < 2; ++i) {            // (chunks 4 dt + 2 i + h, as in store_c_tile)
                    const uint32_t a0 = pack2bf(acc[8 * i] * mul, acc[8 * i + 1] * mul), a1 = pack2bf(acc[8 * i + 2] * mul, acc[8 * i + 3] * mul);
                    const uint32_t b0 = pack2bf(acc[8 * i + 4] * mul, acc[8 * i + 5] * mul), b1 = pack2bf(acc[8 * i + 6] * mul, acc[8 * i + 7] * mul);
                    const auto r0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
                    const auto r1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
                    *reinterpret_cast<u32x4 *>(rows_out + (2 * g + m) * 32 * TL::ROW_B + chunk_at(j_, 4 * tile_of(dt, m) + 2 * i + h_)) = u32x4{r0[0], r1[0], r0[1], r1[1]};
                }
            }
#pragma unroll
    for (int g = 0; g < KG; ++g)
#pragma unroll
        for (int m = 0; m < 2; ++m)
            for (int part = 0; part < (TL::LOADS > 8 ? 2 : 1); ++part) {  // (up to eight rows read in front of their stores)
                constexpr int NL = TL::LOADS > 8 ? 8 : TL::LOADS;
                const int row0 = part * NL * TL::LOAD_ROWS + lane_ / TL::CPR, c = lane_ % TL::CPR, key0 = kc + 32 * g + row0;
                u32x4 x[NL];
#pragma unroll
                for (int i = 0; i < NL; ++i)
                    x[i] = *reinterpret_cast<const u32x4 *>(rows_out + (2 * g + m) * 32 * TL::ROW_B + chunk_at(row0 + i * TL::LOAD_ROWS, c));
                unsigned char *const to = reinterpret_cast<unsigned char *>((m ? dv : dk) + ((int64_t)(s0 + key0) * Hkv + kvh) * dr + c * 8);
#pragma unroll
                for (int i = 0; i < NL; ++i)
                    if (key0 + i * TL::LOAD_ROWS < L && (CARRIED ? carried_chunk(c, m) : c < chunks))
                        *reinterpret_cast<u32x4 *>(to + i * TL::LOAD_ROWS * Hkv * dr * 2) = x[i];
            }
}
