// dQ over 32x32 MFMA tiles, query-stationary, the same walk as the forward (dsa_tile_fwd.hip):
//   S^T = K Q^T, dP^T = V dO^T  (A = K / V tiles row-wise from LDS, B = Q^T / dO^T in registers)
//   dS^T = P^T * (dP^T - delta)  on the C layout, P = exp2(S * scale*log2e - lse*log2e)
//   dQ^T[d,row] += K^T[d,key] dS^T[key,row]   (A = K tile transposed, B = dS^T from the C layout)
//
// A step runs the three chains of MFMAs dP(t), S(t+1), dQ(t) one after the other with the vector work of the neighbouring chains
// behind them: the second half of P(t) behind dP(t), dS(t) behind S(t+1), the first half of P(t+1) behind dQ(t).  Operand reads
// run four MFMAs ahead through all three chains.  K and V tiles go from memory straight into LDS, rings of four: step t requests
// K(t+3), V(t+2) and the selection words of tile t+3, at its end waits for what step t-1 requested and meets the one barrier.
//
// What bounds it: 24 MFMAs (768 clocks at head_dim 128) per tile and wave beside about 110 vector instructions, 16 of them
// exponentials.  Same box, us, against the kernel before (tiles staged through registers, two to four barriers per pair of tiles, no
// vector work behind the chains): head_dim 256 on the fp32 carrier, 2048 tokens 65 -> 48; head_dim 256, 16 384 tokens in short
// segments, backward 840 -> 770; 72-wide vision heads, 16 384 patches 495 -> 455, the whole step 1580 -> 1550 when the chip runs hot.
// Head_dim 97 to 128 keeps that kernel (dsa_tile_dq128_kernel): there two waves per SIMD overlap by themselves, long launches
// are held by the chip's power, and this form was level to 3 % slower (it has no path without mask arithmetic - a second loop
// body spills - and four-wave workgroups, 6 % faster alone, stage twice as much and slow the kernels behind them by as much).
#include "dsa_tile.h"

template <int D, int NW> constexpr size_t dq_lds_bytes(bool has_idx) { return 8 * (size_t)DirectTile<D>::BYTES + (has_idx ? NW * 4 * 256 : 0); }

template <int D, bool HAS_IDX, int NW>
__global__ __launch_bounds__(NW * 64, (D <= 128 && NW == 4) ? 2 : 1) void dsa_tile_dq_kernel(
    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k,
    const bf16_t *__restrict__ v, const float *__restrict__ lse, const float *delta,
    const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv, int gshift,
    float scale, int pos_split, int causal, int d_real, bf16_t *__restrict__ dq, const bf16_t *__restrict__ out_for_delta,
    float *delta_out) {
    typedef DirectTile<D> TL;
    constexpr int KS = D / 16, DT = (D + 31) / 32, NP = 2 * DT;
    constexpr int LPW = TL::LOADS / NW;                  // wave loads per wave, step and operand
    constexpr int LPS = 2 * LPW + (HAS_IDX ? 1 : 0);     // everything a wave requests in a step
    static_assert(TL::LOADS % NW == 0, "every wave loads the same number of pieces");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // 4 K slots | 4 V slots | selection words

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv, kvh = blockIdx.x % Hkv, QBW = (NW * 32) >> gshift;
    const int dr = HAS_IDX ? D : d_real, chunks = dr / 8;   // elements and 16-byte chunks of a row in memory
    int s0, L, blk;
    if (!LOCATE_QUERY_BLOCK(causal, cu, N, blockIdx.x / Hkv, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = __builtin_amdgcn_readfirstlane(L);
    if (HAS_IDX) L = min(L, ldw * 32);                   // a bitmap row has ldw words whatever the caller's max_seqlen
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (qc0 >= pos_split || qc0 >= L) return;            // rows past the split belong to the gather kernel
    const int ntiles = (causal ? min(qc0 + QBW - 1, L - 1) : L - 1) / 32 + 1;

    const int r = wv * 32 + j;
    const int qcol = qc0 + (r >> gshift), head = r & ((1 << gshift) - 1);
    const bool row_ok = qcol < L && head < G;
    const int t = s0 + min(qcol, L - 1), hq = kvh * G + min(head, G - 1);
    const int klim = causal ? qcol : L - 1;              // last key column this row may attend (dense mode)

    // ---- requests (as in the forward) ----
    const int tok_b = Hkv * dr * 2;                      // bytes from one key row to the next
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k + ((int64_t)s0 * Hkv + kvh) * dr);
    const unsigned char *vptr = reinterpret_cast<const unsigned char *>(v + ((int64_t)s0 * Hkv + kvh) * dr);
    constexpr int NV = LPW < TL::SOURCES ? LPW : TL::SOURCES;   // the lane's source offsets repeat after that many pieces
    int voff[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) voff[i] = TL::source(wv * LPW + i, lane, tok_b, chunks);
    const uint32_t lds0 = lds_address(dyn_lds);
    const int Lend = min(L, ntiles * 32);
    auto left = [&](int tile) __attribute__((always_inline)) {
        const int rows = __builtin_amdgcn_readfirstlane(max(min(Lend - tile * 32, 32), 0));
        return rows ? (rows - 1) * tok_b + dr * 2 : 0;
    };
    // piece i of K (or V) tile `tile`; called in tile order.  Rows past the segment and columns past the true head_dim read as zero.
    auto load_piece = [&](const unsigned char *&p, int base, int tile, int i) __attribute__((always_inline)) {
        buffer_load_lds16(make_buffer_rsrc(p, left(tile)),
                          voff[i % NV] + i / NV * NV * TL::LOAD_ROWS * tok_b, lds0 + (base + (tile & 3)) * TL::BYTES + TL::load_lds(wv * LPW + i));
        if (i == LPW - 1) {
            p += (int64_t)32 * tok_b;
            asm volatile("" : "+s"(p));
        }
    };
    unsigned char *const words = dyn_lds + 8 * TL::BYTES + wv * 1024;     // [tile % 4][lane]
    const int wq0 = min(qc0 + ((wv * 32) >> gshift), L - 1);               // the wave's first query
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + wq0) * ldw);
    const int wvoff = (t - s0 - wq0) * ldw * 4;          // (at most 31 rows of bitmap)
    auto load_w = [&](int tile) __attribute__((always_inline)) {
        if (HAS_IDX) {
            buffer_load_lds4(make_buffer_rsrc(wptr, 32 * (int64_t)ldw * 4), wvoff, lds0 + 8 * TL::BYTES + wv * 1024 + (tile & 3) * 256);
            if (tile + 1 < ntiles) {                      // (past the block's tiles: the last word again, never used)
                wptr += 4;
                asm volatile("" : "+s"(wptr));
            }
        }
    };
#pragma unroll
    for (int u = 0; u < 3; ++u) {
#pragma unroll
        for (int i = 0; i < LPW; ++i) load_piece(kptr, 0, u, i);
        load_w(u);
        if (u < 2) {
#pragma unroll
            for (int i = 0; i < LPW; ++i) load_piece(vptr, 4, u, i);
        }
    }
    bf16x8 qB[KS], doB[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int64_t off = ((int64_t)t * Hq + hq) * dr + 16 * ks + 8 * h;
        const bool there = row_ok && (HAS_IDX || 2 * ks + h < chunks);
        qB[ks] = there ? load_bf16x8(q + off) : zero_bf16x8();
        doB[ks] = there ? load_bf16x8(dout + off) : zero_bf16x8();
    }
    const float scale_log2 = scale * LOG2E_F, neg_lse2 = -lse[(int64_t)hq * T + t] * LOG2E_F;
    // delta = rowsum(dO * O) of the lane's row: read, or - when every query row of the launch belongs to this kernel -
    // formed here from the dO row the lane already holds and written out for the key-side pass (one launch and one
    // pass over dO and O less)
    float dlt;
    if (out_for_delta) {                                 // (kernel argument: the same for every wave)
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
                p[c] = dot8_chain(doB[ks], o8, p[c]);
            }
        }
        dlt = half_sum_f(((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7])));
        if (row_ok && h == 0) delta_out[(int64_t)hq * T + t] = dlt;
    } else {
        dlt = delta[(int64_t)hq * T + t];
    }

    TL tl;
    tl.init(lane);
    constexpr int AHEAD = 4;                             // MFMAs an operand is read ahead
    f32x16 acc[DT], sE, sO;                              // S of even and of odd tiles
    float eE[8], eO[8];                                  // P of their first eight elements
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();
    wait_vmcnt<0>();
    barrier_only();

    const uint32_t row_mask = row_ok ? 0xffffffffu : 0u;
    // the keys of a tile this lane keeps: element vi then sits at bit 8*(vi/4) + vi%4
    auto word_of = [&](int tile) __attribute__((always_inline)) {
        const uint32_t w = HAS_IDX ? *reinterpret_cast<const uint32_t *>(words + (tile & 3) * 256 + lane * 4) : causal_bits(klim - tile * 32);
        return (w >> (4 * h)) & row_mask;
    };
    auto prob = [&](bool masked, float s, uint32_t word, int vi) __attribute__((always_inline)) {
        const float y = fmaf(s, scale_log2, neg_lse2);
        return fast_exp2(masked ? keep_or_neginf(y, bit_mask(word, 8 * (vi >> 2) + (vi & 3))) : y);
    };
    int a4[4];                                           // operand addresses: V(t) row-wise, K(t+1) row-wise, K(t) transposed in turn
    auto row_op = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8 *>(dyn_lds + a4[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto tr_op = [&](int i) __attribute__((always_inline)) {             // MFMA i of dQ: keys of half i / DT, d-tile i % DT
        const int pair = i / DT, dt = i % DT;
        lds_u8 *p = (lds_u8 *)dyn_lds + a4[TL::tr_q(dt)];
        return LaneOffsets<D>::tr_pair(p + TL::tr_imm(dt, 2 * pair), p + TL::tr_imm(dt, 2 * pair + 1));
    };
    // S of tile 0, first half of its P
    uint32_t word_cur = word_of(0);
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) a4[i] = tl.rowq[i];
        bf16x8 a[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a[ks] = row_op(ks);
        sE = zero16();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sE = mfma32(a[ks], qB[ks], sE);
#pragma unroll
        for (int vi = 0; vi < 8; ++vi) eE[vi] = prob(true, sE[vi], word_cur, vi);
    }
    auto request = [&](int t_, int r_) __attribute__((always_inline)) {
        if (r_ < LPW) load_piece(kptr, 0, t_ + 3, r_);
        else if (r_ < 2 * LPW) load_piece(vptr, 4, t_ + 2, r_ - LPW);
        else load_w(t_ + 3);
    };
    // Step t: `e` holds P of elements 0-7 of tile t, `s` its S (8-15 are still to come), `en` and `sn` get the same of tile t+1
    // (NEXT).  MA, MC: tile t, t+1 needs its mask.
    auto step = [&](auto ma_, auto mc_, auto next_, int t_, const float (&e)[8], const f32x16 &s, float (&en)[8], f32x16 &sn) __attribute__((always_inline)) {
        constexpr bool MA = decltype(ma_)::value, MC = decltype(mc_)::value, NEXT = decltype(next_)::value;
        constexpr int M1 = KS, M2 = NEXT ? 2 * KS : KS, M = M2 + NP, LAG = 2;
        auto fetch = [&](int m) __attribute__((always_inline)) {          // operand of MFMA m; called for m = 0, 1, 2, ...
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (m == 0) a4[i] = tl.rowq[i] + (4 + (t_ & 3)) * TL::BYTES;
                else if (m == M2) a4[i] = tl.trq[i] + (t_ & 3) * TL::BYTES;
                else if (m == M1) a4[i] = tl.rowq[i] + ((t_ + 1) & 3) * TL::BYTES;
            }
            return m < M2 ? row_op(m < M1 ? m : m - M1) : tr_op(m - M2);
        };
        bf16x8 op[AHEAD];
#pragma unroll
        for (int m = 0; m < AHEAD; ++m) op[m] = fetch(m);
        const uint32_t word = word_cur;
        if (NEXT) word_cur = word_of(t_ + 1);
        float p2[8], first;
        f32x16 dp, snew;
        uint32_t ds[8];
        auto form_ds = [&](int vi) __attribute__((always_inline)) {
            const float x = (vi < 8 ? e[vi & 7] : p2[vi & 7]) * (dp[vi] - dlt);
            if (vi & 1) {
                ds[vi >> 1] = pack2bf(first, x);
                asm volatile("" : "+v"(ds[vi >> 1]));
            } else {
                first = x;
            }
        };
        auto fence = [&]() __attribute__((always_inline)) {
            asm volatile("" : : : "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < KS; ++i) {                   // dP(t), behind it the second half of P(t) and the step's requests
            dp = mfma32(op[i % AHEAD], doB[i], i == 0 ? zero16() : dp);
            if (i + AHEAD < M) op[i % AHEAD] = fetch(i + AHEAD);
#pragma unroll
            for (int r_ = 0; r_ < LPS; ++r_)
                if (NEXT && r_ * KS / LPS == i) request(t_, r_);
#pragma unroll
            for (int vi = 8 * i / KS; vi < 8 * (i + 1) / KS; ++vi) {
                p2[vi] = prob(MA, s[8 + vi], word, 8 + vi);
                asm volatile("" : "+v"(p2[vi]));
            }
            fence();
        }
        if constexpr (NEXT) {
#pragma unroll
            for (int i = 0; i < KS; ++i) {               // S(t+1), behind it dS(t)
                const int m = M1 + i;
                snew = mfma32(op[m % AHEAD], qB[i], i == 0 ? zero16() : snew);
                if (m + AHEAD < M) op[m % AHEAD] = fetch(m + AHEAD);
                constexpr int S = KS - LAG + 1;
                const int u = i - LAG + 1;
#pragma unroll
                for (int vi = 16 * u / S; vi < 16 * (u + 1) / S; ++vi)
                    if (u >= 0) form_ds(vi);
                fence();
            }
        } else {
#pragma unroll
            for (int vi = 0; vi < 16; ++vi) form_ds(vi);
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {                   // dQ(t), behind it the first half of P(t+1)
            const int m = M2 + i;
            const u32x4 w = i < DT ? u32x4{ds[0], ds[1], ds[2], ds[3]} : u32x4{ds[4], ds[5], ds[6], ds[7]};
            acc[i % DT] = mfma32(op[m % AHEAD], __builtin_bit_cast(bf16x8, w), acc[i % DT]);
            if (m + AHEAD < M) op[m % AHEAD] = fetch(m + AHEAD);
            if (NEXT) {
                constexpr int S = NP - LAG + 1;
                const int u = i - LAG + 1;
#pragma unroll
                for (int vi = 8 * u / S; vi < 8 * (u + 1) / S; ++vi)
                    if (u >= 0) {
                        en[vi] = prob(MC, snew[vi], word_cur, vi);
                        asm volatile("" : "+v"(en[vi]));
                    }
            }
            fence();
        }
        if (NEXT) {
            sn = snew;
            wait_vmcnt<LPS>();                           // all but what this step requested
            barrier_only();
        }
    };
    const std::true_type yes;
    const std::false_type no;
    int tt = 0;
    if (!HAS_IDX && D < 256) {
        // tiles every row of the block attends whole: no mask arithmetic (tile tt+1 of the step's second half included; at
        // head_dim 256 a second loop body spills)
        const int whole = (causal ? qc0 : L) / 32;
        for (; tt + 2 < ntiles && tt + 2 < whole; tt += 2) {
            step(no, no, yes, tt, eE, sE, eO, sO);
            step(no, no, yes, tt + 1, eO, sO, eE, sE);
        }
    }
    for (; tt + 2 < ntiles; tt += 2) {
        step(yes, yes, yes, tt, eE, sE, eO, sO);
        step(yes, yes, yes, tt + 1, eO, sO, eE, sE);
    }
    if (tt + 1 < ntiles) {
        step(yes, yes, yes, tt, eE, sE, eO, sO);
        step(yes, no, no, tt + 1, eO, sO, eE, sE);
    } else {
        step(yes, no, no, tt, eE, sE, eO, sO);
    }
    wait_vmcnt<0>();                                     // no load is left on its way into LDS when the workgroup ends

    if (row_ok) {
        bf16_t *op = dq + ((int64_t)t * Hq + hq) * dr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store_c_tile(op + dt * 32, acc[dt], scale, h, chunks - 4 * dt);
    }
}

extern "C" hipError_t dsa_launch_tile_dq_128(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                                             const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real,
                                             float scale, int pos_split, int causal, void *dq, const void *out_for_delta,
                                             float *delta_out, hipStream_t stream);
template <int D, bool HAS_IDX>
static hipError_t launch_dq_i(hipStream_t stream, const void *dout, const void *q, const void *k, const void *v, const float *lse,
                              const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, int gs,
                              int d_real, float scale, int pos_split, int causal, void *dq, const void *out_for_delta, float *delta_out) {
    constexpr int NW = D > 64 && D < 256 ? 8 : 4;        // waves that share the staged tiles
    constexpr size_t lds = dq_lds_bytes<D, NW>(HAS_IDX);
    const auto kernel = &dsa_tile_dq_kernel<D, HAS_IDX, NW>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(((int64_t)T / ((32 * NW) >> gs) + N + 1) * Hkv));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), lds, stream, (const bf16_t *)dout, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, lse, delta,
                       bitmap, ldw, cu, N, T, Hq, Hkv, gs, scale, pos_split, causal, d_real, (bf16_t *)dq, (const bf16_t *)out_for_delta, delta_out);
    return hipGetLastError();
}
// d_real: elements of a row, without a selection any multiple of 8 (dense_kernel_dim).  out_for_delta != null: the kernel forms
// delta = rowsum(dO * O) of its rows itself and writes it to delta_out
extern "C" hipError_t dsa_launch_tile_dq(const void *dout, const void *q, const void *k, const void *v,
                                         const float *lse, const float *delta, const uint32_t *bitmap, int ldw,
                                         const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real, float scale,
                                         int pos_split, int causal, void *dq, const void *out_for_delta, float *delta_out,
                                         hipStream_t stream) {
    const int gs = group_shift(Hq, Hkv);
#define DQ_CASE(D_, HI) return launch_dq_i<D_, HI>(stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, gs, d_real, scale, pos_split, \
                                                   causal, dq, out_for_delta, delta_out)
    if (d_real > 96 && d_real <= 128)
        return dsa_launch_tile_dq_128(dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, pos_split, causal, dq, out_for_delta, delta_out, stream);
    if (bitmap) switch (d_real) {
        case 64: DQ_CASE(64, true);
        case 256: DQ_CASE(256, true);
    } else switch (dense_kernel_dim(d_real)) {
        case 64: DQ_CASE(64, false);
        case 80: DQ_CASE(80, false);
        case 96: DQ_CASE(96, false);
        case 256: DQ_CASE(256, false);
    }
#undef DQ_CASE
    return hipErrorInvalidValue;
}
