// Indexer backward over 32x32 MFMA tiles.  The indexer score of a selected pair is  I[t,s] = c * sum_h w[t,h] relu(r[t,h,s]),
// r = q_idx[t,h,:] . k_idx[s,:]  (multi-query attention with ReLU in place of the softmax: Hi heads, one key head).  Given
// dscore[t,j] = dLoss/dI at the selected keys (slot j of key s = its rank in the ascending selection list = selected keys of
// earlier tiles + those below it in the tile's word):
//     G[t,h,s]   = dscore[t,s] * w[t,h] * (r > 0)
//     dq_idx[t,h,:] = c * sum_s G[t,h,s] k_idx[s,:]      dw[t,h] = c * sum_s dscore[t,s] relu(r[t,h,s])
//     dk_idx[s,:]   = c * sum_t sum_h G[t,h,s] q_idx[t,h,:]
// (the query side of a selection that is short against the segments: dsa_tile_idxg.hip)
// Query side: rows = (query, indexer head), padded to 32 or 64 rows per query so that the 32 rows of a wave belong to one query;
// the wave walks the key tiles: S^T = K Q^T, G^T on the C layout, dQ^T += K^T G^T.  Key side: a wave owns 32 keys (rows in
// registers) and walks the later queries in tiles of 32 heads of one query: S = Q K^T, G on the C layout, dK^T += Q^T G.  Every
// output row is reduced in a fixed order: deterministic, no atomics.
//
// Both sides are the same walk over tiles of one moving operand, read row-wise by the first product and transposed by the second
// (`gated_walk`).  Each wave runs three tiles at once: step t issues the MFMAs of acc += A(t)^T G(t) and of S(t+2) in pairs, and
// the gating of tile t+1 stands between them.  Tiles, gradients and head weights go from memory straight into LDS, requested
// three to six tiles ahead; the gather of a tile's 32 gradients takes its offsets from the selection word (held 64 words at a
// time in a wave's lanes) and lets the buffer bound answer zero for keys that are not selected.  One barrier per two tiles.
//
// What bounds it: 16 MFMAs (512 clocks) per tile and wave against about 80 vector instructions and 16 LDS operand reads, one barrier per
// two tiles; at about 1.1 PFLOP/s of executed MFMA work the chip's power limit holds the clock near 1.9 GHz (one barrier per tile
// instead of two: 1 % slower; operand addresses moved on in place instead of formed per tile: key side 2412 -> 2365, query side 2192 ->
// 2178).  Same box, us, against the kernels before (operands staged through registers, the two products and
// the gating of a tile one after the other): 32 768 tokens, 64 heads of 128: query side 2750 -> 2340, key side 2870 -> 2460; 8192
// tokens, 32 heads of 64, both side by side: 150 -> 127.
#include "dsa_tile.h"

// acc += sum over the tiles of A(t)^T G(t), G(t) = gate of A(t) B.  ring: eight tile slots (tile u in slot u % 8).
//   request(t, i):      issues piece i of P of what the even step t requests: tiles t+5 and t+6 and whatever gates tiles t+3 and
//                       t+4; the caller has requested tiles 0..4 and the gates of tiles 0..2
//   gate_load(t):       reads what gates tile t;  gate(vi, s): element vi of G from element vi of S
template <int D, int P, class Request, class GateLoad, class Gate>
__device__ __forceinline__ void gated_walk(unsigned char *ring, int lane, int ntiles, const bf16x8 (&b)[D / 16], f32x16 (&acc)[D / 32],
                                           Request request, GateLoad gate_load, Gate gate) {
    typedef DirectTile<D> TL;
    constexpr int KS = D / 16, DT = D / 32, AHEAD = D == 64 ? 2 : 4;
    static_assert(KS == 2 * DT && KS % AHEAD == 0);
    TL tl;
    tl.init(lane);
    f32x16 sE, sO;                                      // S of even and of odd tiles
    uint32_t pE[8], pO[8];                              // G of even and of odd tiles, packed
    wait_vmcnt<0>();
    barrier_only();
    lds_u8 *ra[4], *ta[4];                              // operand addresses in the tile of S(t+2) and in tile t
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ra[i] = (lds_u8 *)ring + tl.rowq[i];
        ta[i] = (lds_u8 *)ring + tl.trq[i];
    }
    auto advance = [&](lds_u8 *(&a)[4], int tile) __attribute__((always_inline)) {         // from tile - 1 to tile
        const int by = tile & 7 ? TL::BYTES : -7 * TL::BYTES;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] += by;
            asm volatile("" : "+v"(a[i]));
        }
    };
    auto read_row = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(ra[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto read_tr = [&](int i) __attribute__((always_inline)) {           // MFMA i of the second product: rows of half i / DT, d-tile i % DT
        const int pair = i / DT, dt = i % DT;
        lds_u8 *p = ta[TL::tr_q(dt)];
        return tr_pair(p + TL::tr_imm(dt, 2 * pair), p + TL::tr_imm(dt, 2 * pair + 1));
    };
    auto gemm_s = [&](f32x16 &s) __attribute__((always_inline)) {
        s = zero16();
        bf16x8 a[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a[ks] = read_row(ks);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s = mfma32(a[ks], b[ks], s);
    };
    gemm_s(sE);
    advance(ra, 1);
    if (ntiles > 1) gemm_s(sO);
    gate_load(0);
#pragma unroll
    for (int vi = 0; vi < 16; vi += 2) {
        const float x = gate(vi, sE[vi]), y = gate(vi + 1, sE[vi + 1]);
        pE[vi >> 1] = pack2bf(x, y);
    }
    bf16x8 rr[AHEAD], tr[AHEAD];                        // operands of the next MFMA pairs
    advance(ra, 2);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) { rr[i] = read_row(i); tr[i] = read_tr(i); }

    // Step t: acc += A(t)^T G(t) with `p`; gating of tile t+1 from `s` into `pn` (SM); S(t+2) into `sn` (NEXT).
    auto step = [&](auto sm_, auto next_, auto req_, int t_, const uint32_t (&p)[8], const f32x16 &s, uint32_t (&pn)[8],
                    f32x16 &sn) __attribute__((always_inline)) {
        constexpr bool SM = decltype(sm_)::value, NEXT = decltype(next_)::value, REQ = decltype(req_)::value;
        const u32x4 w0 = {p[0], p[1], p[2], p[3]}, w1 = {p[4], p[5], p[6], p[7]};
        const bf16x8 g0 = __builtin_bit_cast(bf16x8, w0), g1 = __builtin_bit_cast(bf16x8, w1);
        f32x16 snew;
        if (SM) gate_load(t_ + 1);
        constexpr int LAG = 3, H = 2 * KS - LAG;        // the gate's operands have LAG MFMAs to arrive
        float first;
        auto behind = [&](int hs) __attribute__((always_inline)) {
            if (SM && hs >= LAG) {
#pragma unroll
                for (int vi = 16 * (hs - LAG) / H; vi < 16 * (hs - LAG + 1) / H; ++vi) {
                    const float x = gate(vi, s[vi]);
                    if (vi & 1) {
                        pn[vi >> 1] = pack2bf(first, x);
                        asm volatile("" : "+v"(pn[vi >> 1]));
                    } else {
                        first = x;
                        asm volatile("" : "+v"(first));
                    }
                }
            }
            asm volatile("" : : : "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            acc[i % DT] = mfma32(tr[i % AHEAD], i < DT ? g0 : g1, acc[i % DT]);
#pragma unroll
            for (int r = 0; r < P; ++r)
                if (REQ && r * KS / P == i) request(t_, r);
            if (i == KS - AHEAD && SM) advance(ta, t_ + 1);
            if (i + AHEAD < KS || SM) tr[i % AHEAD] = read_tr((i + AHEAD) % KS);
            behind(2 * i);
            if (NEXT) {
                snew = mfma32(rr[i % AHEAD], b[i], i == 0 ? zero16() : snew);
                if (i == KS - AHEAD) advance(ra, t_ + 3);
                rr[i % AHEAD] = read_row((i + AHEAD) % KS);
            }
            behind(2 * i + 1);
        }
        if (NEXT) sn = snew;
    };
    const std::true_type yes;
    const std::false_type no;
    int tt = 0;
    for (; tt + 3 < ntiles; tt += 2) {
        step(yes, yes, yes, tt, pE, sO, pO, sE);
        step(yes, yes, no, tt + 1, pO, sE, pE, sO);
        wait_vmcnt<0>();
        barrier_only();
    }
    // at most three tiles are left, all of them in LDS
    if (tt + 2 < ntiles) {
        step(yes, yes, no, tt, pE, sO, pO, sE);
        step(yes, no, no, tt + 1, pO, sE, pE, sO);
        step(no, no, no, tt + 2, pE, sO, pO, sE);
    } else if (tt + 1 < ntiles) {
        step(yes, no, no, tt, pE, sO, pO, sE);
        step(no, no, no, tt + 1, pO, sE, pE, sO);
    } else {
        step(no, no, no, tt, pE, sO, pO, sE);
    }
    wait_vmcnt<0>();                                    // no load is left on its way into LDS when the workgroup ends
}
// what a load leaves out of its buffer: such a lane gets zero
#define IDX_NOT_THERE ((int)0x80000000)

// ---- query side ---------------------------------------------------------------------------------------------------------
template <int D, int NW> constexpr size_t idxq_lds_bytes() { return 8 * (size_t)DirectTile<D>::BYTES + NW * 4 * 256; }
template <int D, int GSHIFT, int NW>
__global__ __launch_bounds__(NW * 64, D == 64 ? 3 : 2) void dsa_tile_idxq_kernel(
    const bf16_t *__restrict__ q_idx, const bf16_t *__restrict__ k_idx, const bf16_t *__restrict__ w_idx,
    const float *__restrict__ dscore, const float *__restrict__ grad, const uint32_t *__restrict__ bitmap, int ldw,
    const int32_t *__restrict__ cu, int N, int T, int Hi, int K, float cscale, bf16_t *__restrict__ dq_idx, void *__restrict__ dw, int dw_bf16) {
    typedef DirectTile<D> TL;
    constexpr int KS = D / 16, DT = D / 32, Gp = 1 << GSHIFT, QBW = (NW * 32) >> GSHIFT, LPW = TL::LOADS / NW;
    static_assert(TL::LOADS % NW == 0 && GSHIFT >= 5, "a wave's 32 rows are heads of one query");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // 8 K slots | gradients [wave][tile % 4][key]

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int s0, L, blk;
    if (!LOCATE_QUERY_BLOCK(true, gridDim.x, cu, N, blockIdx.x, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = min(__builtin_amdgcn_readfirstlane(L), ldw * 32);
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (qc0 >= L || idx_segment_gathers(Hi, K, L)) return;
    const int ntiles = min(qc0 + QBW - 1, L - 1) / 32 + 1;
    const int qw = qc0 + ((wv * 32) >> GSHIFT), t = s0 + min(qw, L - 1);         // the wave's query
    const int head = ((wv * 32) & (Gp - 1)) + j;
    const bool row_ok = qw < L && head < Hi;

    // ---- requests ----
    const uint32_t lds0 = lds_address(dyn_lds);
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k_idx + (int64_t)s0 * D);
    const int Lend = min(L, ntiles * 32), koff = TL::source(wv * LPW, lane, 2 * D, D / 8);
    auto load_k = [&](int tile, int i) __attribute__((always_inline)) {
        buffer_load_lds16(make_buffer_rsrc(kptr, max(min(Lend - tile * 32, 32), 0) * 2 * D), koff + i * TL::LOAD_ROWS * 2 * D,
                          lds0 + (tile & 7) * TL::BYTES + TL::load_lds(wv * LPW + i));
        if (i == LPW - 1) {
            kptr += 32 * 2 * D;
            asm volatile("" : "+s"(kptr));
        }
    };
    const uint32_t *const wrow = bitmap + (int64_t)t * ldw;
    const bool q_ok = qw < L;
    uint32_t words = q_ok ? wrow[min(lane, ntiles - 1)] : 0u, words_next = q_ok ? wrow[min(64 + lane, ntiles - 1)] : 0u;
    int seen = 0;                                       // selected keys in the tiles requested so far
    const buffer_rsrc grads = make_buffer_rsrc(dscore + (int64_t)t * K, (int64_t)K * 4);
    const uint32_t grad_lds = lds0 + 8 * TL::BYTES + wv * 1024;
    // the gradients of a tile's keys, key j by lane j; called for tile 0, 1, 2, ... in turn
    auto load_grads = [&](int tile) __attribute__((always_inline)) {
        if ((tile & 63) == 0 && tile > 0) {
            words = words_next;
            words_next = q_ok ? wrow[min(tile + 64 + lane, ntiles - 1)] : 0u;
        }
        const uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)words, tile & 63) & (tile < ntiles ? 0xffffffffu : 0u);
        const int slot = seen + (int)__builtin_amdgcn_mbcnt_lo(word, 0u);
        const bool sel = lane < 32 && ((word >> j) & 1u);
        buffer_load_lds4(grads, sel ? slot * 4 : IDX_NOT_THERE, grad_lds + (tile & 3) * 256);
        seen += __popc(word);
    };
#pragma unroll
    for (int u = 0; u < 5; ++u) {
#pragma unroll
        for (int i = 0; i < LPW; ++i) load_k(u, i);
        if (u < 3) load_grads(u);
    }
    bf16x8 qB[KS];
    const int hrow = min(head, Hi - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qB[ks] = row_ok ? load_bf16x8(q_idx + ((int64_t)t * Hi + hrow) * D + 16 * ks + 8 * h) : zero_bf16x8();
    const float wrow_v = row_ok ? (float)w_idx[(int64_t)t * Hi + hrow] : 0.f;
    if (grad) cscale *= *grad;
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();
    float dwacc = 0.f;
    f32x4 d4[4];                                        // element vi is key column 8*(vi/4) + 4h + vi%4
    gated_walk<D, 2 * LPW + 2>(
        dyn_lds, lane, ntiles, qB, acc,
        [&](int t_, int i) __attribute__((always_inline)) {
            if (i < LPW) load_k(t_ + 5, i);
            else if (i < 2 * LPW) load_k(t_ + 6, i - LPW);
            else load_grads(t_ + 3 + i - 2 * LPW);
        },
        [&](int tile) __attribute__((always_inline)) {
            const unsigned char *g = dyn_lds + 8 * TL::BYTES + wv * 1024 + (tile & 3) * 256 + 16 * h;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) d4[g4] = *reinterpret_cast<const f32x4 *>(g + 32 * g4);
        },
        [&](int vi, float s) __attribute__((always_inline)) {
            const float x = s > 0.f ? d4[vi >> 2][vi & 3] : 0.f;     // (the row's weight multiplies the finished sum instead)
            dwacc = fmaf(x, s, dwacc);                               // dscore * relu(s)
            asm volatile("" : "+v"(dwacc));                            // (formed here: its operands are not kept)
            return x;
        });
    const float dwt = half_sum_f(dwacc);
    if (row_ok) {
        bf16_t *op = dq_idx + ((int64_t)t * Hi + hrow) * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store_c_tile(op + dt * 32, acc[dt], cscale * wrow_v, h);
        if (h == 0) {
            if (dw_bf16) reinterpret_cast<bf16_t *>(dw)[(int64_t)t * Hi + hrow] = (bf16_t)(dwt * cscale);
            else reinterpret_cast<float *>(dw)[(int64_t)t * Hi + hrow] = dwt * cscale;
        }
    }
}

// ---- key side -----------------------------------------------------------------------------------------------------------
// Workgroup = 4 waves x 32 keys = one 128-key tile of a segment; the walk takes the queries from the end of the segment down to
// the tile (HB tiles of 32 heads each), so that the workgroups of a segment that run side by side read the same index-query rows
// at about the same time and share them in L2.
template <int D> constexpr size_t idxk_lds_bytes() { return 8 * (size_t)DirectTile<D>::BYTES + 4 * 4 * 512; }
template <int D, int GSHIFT>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void dsa_tile_idxk_kernel(
    const bf16_t *__restrict__ q_idx, const bf16_t *__restrict__ k_idx, const float *__restrict__ w_f32,
    const float *__restrict__ dscore, const float *__restrict__ grad, const uint32_t *__restrict__ bitmap,
    const int32_t *__restrict__ prefix, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hi, int K, float cscale,
    int chunk_steps, float *__restrict__ partial) {
    typedef DirectTile<D> TL;
    constexpr int KS = D / 16, DT = D / 32, HB = (1 << GSHIFT) / 32, LPW = TL::LOADS / 4;
    static_assert(TL::LOADS % 4 == 0 && (HB == 1 || HB == 2), "tiles of 32 heads of one query");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // 8 q slots | [wave][step % 4] gradients, head weights

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int s0, L, blk;
    if (!locate_block(cu, N, blockIdx.x, 128, false, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = min(__builtin_amdgcn_readfirstlane(L), ldw * 32);
    const int c0 = __builtin_amdgcn_readfirstlane(blk) * 128, kc = c0 + wv * 32;
    if (c0 >= L) return;
    // queries L-1 down to c0 can have selected keys of this tile; the walk is cut into pieces of chunk_steps queries (blockIdx.y),
    // each piece leaving a partial sum: a tile at the start of a long segment would otherwise be one long serial walk
    const int st0 = blockIdx.y * chunk_steps, nsteps = min(L - c0 - st0, chunk_steps);
    if (nsteps <= 0) return;
    const int ntiles = nsteps * HB, q_first = s0 + L - 1 - st0;          // token of step 0
    const bool key_ok = kc + j < L;
    const int64_t krow = (int64_t)s0 + min(kc + j, L - 1);

    // ---- requests ----
    const uint32_t lds0 = lds_address(dyn_lds);
    const int qoff = TL::source(wv * LPW, lane, 2 * D, D / 8);
    const unsigned char *qptr = reinterpret_cast<const unsigned char *>(q_idx + (int64_t)q_first * Hi * D);
    // tile u: heads 32 (u % HB) .. of step u / HB (padded heads read as zero); called for u = 0, 1, 2, ... in turn
    auto load_q = [&](auto odd_, int u, int i) __attribute__((always_inline)) {
        constexpr int hb = HB == 2 && decltype(odd_)::value ? 1 : 0;
        const int heads = u < ntiles ? (HB == 2 && hb == 0 ? 32 : Hi - 32 * hb) : 0;
        buffer_load_lds16(make_buffer_rsrc(qptr, heads * 2 * D), qoff + i * TL::LOAD_ROWS * 2 * D,
                          lds0 + (u & 7) * TL::BYTES + TL::load_lds(wv * LPW + i));
        if (i == LPW - 1) {
            qptr += HB == 2 && hb == 0 ? 32 * 2 * D : -(int64_t)(Hi + 32 * hb) * 2 * D;
            asm volatile("" : "+s"(qptr));
        }
    };
    // selection word and slot base of (query of a step, this wave's 32 keys), 64 steps at a time, one per lane
    const int kw = kc < L ? kc >> 5 : 0;                // the word column of this wave's keys, where it exists
    auto word_row = [&](int step) __attribute__((always_inline)) { return (int64_t)(q_first - min(step, nsteps - 1)) * ldw + kw; };
    uint32_t words = bitmap[word_row(lane)], words_next = bitmap[word_row(64 + lane)];
    int32_t bases = prefix[word_row(lane)], bases_next = prefix[word_row(64 + lane)];
    const unsigned char *dptr = reinterpret_cast<const unsigned char *>(dscore + (int64_t)q_first * K);
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(w_f32 + (int64_t)q_first * 64);
    const uint32_t aux_lds = lds0 + 8 * TL::BYTES + wv * 2048;
    // the gradients of (step, key j) by lane j and the head weights of the step; called for step 0, 1, 2, ... in turn
    auto load_grads = [&](int step) __attribute__((always_inline)) {
        if ((step & 63) == 0 && step > 0) {
            words = words_next;
            bases = bases_next;
            words_next = bitmap[word_row(step + 64 + lane)];
            bases_next = prefix[word_row(step + 64 + lane)];
        }
        const bool live = step < nsteps;
        const uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)words, step & 63) & (live && kc < L ? 0xffffffffu : 0u);
        const int slot = __builtin_amdgcn_readlane(bases, step & 63) + (int)__builtin_amdgcn_mbcnt_lo(word, 0u);
        const bool sel = lane < 32 && ((word >> j) & 1u);
        buffer_load_lds4(make_buffer_rsrc(dptr, live ? (int64_t)K * 4 : 0), sel ? slot * 4 : IDX_NOT_THERE, aux_lds + (step & 3) * 256);
    };
    auto load_weights = [&](int step) __attribute__((always_inline)) {
        buffer_load_lds4(make_buffer_rsrc(wptr, step < nsteps ? 256 : 0), lane * 4, aux_lds + 1024 + (step & 3) * 256);
        dptr -= (int64_t)K * 4;
        wptr -= 256;
        asm volatile("" : "+s"(dptr), "+s"(wptr));
    };
    const std::true_type odd;
    const std::false_type even;
#pragma unroll
    for (int u = 0; u < 5; ++u) {
#pragma unroll
        for (int i = 0; i < LPW; ++i)
            if (u & 1) load_q(odd, u, i); else load_q(even, u, i);
        if (u < 3 && u % HB == 0) { load_grads(u / HB); load_weights(u / HB); }
    }
    bf16x8 kB[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kB[ks] = load_bf16x8(k_idx + krow * D + 16 * ks + 8 * h);
    if (grad) cscale *= *grad;
    f32x16 dkacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) dkacc[dt] = zero16();
    float dl = 0.f;                                     // gradient of (query of the tile, this lane's key)
    f32x4 w4[4];                                        // element vi is head 8*(vi/4) + 4h + vi%4 of the tile
    gated_walk<D, 2 * LPW + (HB == 2 ? 2 : 4)>(
        dyn_lds, lane, ntiles, kB, dkacc,
        [&](int t_, int i) __attribute__((always_inline)) {
            const int g = i - 2 * LPW, s = HB == 2 ? (t_ + 4) / 2 : t_ + 3 + g / 2;      // (two heads tiles: step s has both)
            if (i < LPW) load_q(odd, t_ + 5, i);
            else if (i < 2 * LPW) load_q(even, t_ + 6, i - LPW);
            else if (g % 2 == 0) load_grads(s);
            else load_weights(s);
        },
        [&](int tile) __attribute__((always_inline)) {
            const int step = tile / HB;
            const unsigned char *a = dyn_lds + 8 * TL::BYTES + wv * 2048 + (step & 3) * 256;
            dl = *reinterpret_cast<const float *>(a + 4 * j);
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) w4[g4] = *reinterpret_cast<const f32x4 *>(a + 1024 + (tile % HB) * 128 + 32 * g4 + 16 * h);
        },
        [&](int vi, float s) __attribute__((always_inline)) { return s > 0.f ? dl * w4[vi >> 2][vi & 3] : 0.f; });
    if (key_ok) {
        float *pk = partial + ((int64_t)blockIdx.y * T + krow) * D + 4 * h;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const f32x4 o4 = {dkacc[dt][4 * g4] * cscale, dkacc[dt][4 * g4 + 1] * cscale, dkacc[dt][4 * g4 + 2] * cscale,
                                  dkacc[dt][4 * g4 + 3] * cscale};
                *reinterpret_cast<f32x4 *>(pk + dt * 32 + 8 * g4) = o4;
            }
    }
}

// dk_idx[s,:] = sum of the partial sums of the pieces of its tile's walk, in piece order
__global__ __launch_bounds__(256) void dsa_idxk_reduce_kernel(const float *__restrict__ partial,
                                                               const int32_t *__restrict__ cu, int N, int T, int D,
                                                               int chunk_steps, int max_cols, bf16_t *__restrict__ dk_idx) {
    const int s = blockIdx.x * (256 / 32) + (threadIdx.x >> 5), c4 = (threadIdx.x & 31) * 4;   // 32 threads x 4 columns per pass
    if (s >= T) return;
    const int seg = find_segment(cu, N, s);
    const int s0 = cu[seg], L = min(cu[seg + 1] - s0, max_cols);     // as the walk: no column past the bitmap row
    const int c0 = ((s - s0) >> 7) << 7;
    if (c0 >= L) return;
    const int pieces = (L - c0 + chunk_steps - 1) / chunk_steps;
    for (int c = c4; c < D; c += 128) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int pc = 0; pc < pieces; ++pc) acc += *reinterpret_cast<const f32x4 *>(partial + ((int64_t)pc * T + s) * D + c);
        const u32x2 o = {pack2bf(acc[0], acc[1]), pack2bf(acc[2], acc[3])};
        *reinterpret_cast<u32x2 *>(dk_idx + (int64_t)s * D + c) = o;
    }
}

// prefix[t][w] = selected keys of query t in the words before w (the slot of the first selected key of word w);
// w_f32[t][0..63] = the head weights of query t in fp32, zero past the last head
__global__ __launch_bounds__(64) void dsa_bitmap_prefix_kernel(const uint32_t *__restrict__ bitmap, int ldw,
                                                                int32_t *__restrict__ prefix, const bf16_t *__restrict__ w_idx, int Hi,
                                                                float *__restrict__ w_f32) {
    const int lane = threadIdx.x;
    w_f32[(int64_t)blockIdx.x * 64 + lane] = lane < Hi ? (float)w_idx[(int64_t)blockIdx.x * Hi + lane] : 0.f;
    const uint32_t *row = bitmap + (int64_t)blockIdx.x * ldw;
    int32_t *orow = prefix + (int64_t)blockIdx.x * ldw;
    int carry = 0;
    for (int w0 = 0; w0 < ldw; w0 += 64) {
        const int w = w0 + lane;
        const int c = w < ldw ? (int)__popc(row[w]) : 0;
        int incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(incl, off, 64);
            if (lane >= off) incl += u;
        }
        if (w < ldw) orow[w] = carry + incl - c;
        carry += __shfl(incl, 63, 64);
    }
}


// indexer backward: prefix table, query side (dq_idx, dw), key side (dk_idx).  D = indexer head_dim (64 or 128),
// at most 64 indexer heads.
// Queries per piece of a key tile's walk in the indexer backward.  A piece is one workgroup and about 1.3 us per query:
// the finer the pieces, the better a launch of few thousand of them balances over 512 workgroup slots (32 768 tokens:
// 6.26 -> 5.95 ms with 256 instead of 512, 6.31 with 128; 8192 tokens: 0.44 -> 0.31 -> 0.25 ms), the more fp32 partial
// sums (one (T, Di) plane per piece index).  Depends on T, and on the bound of the longest segment only where the
// planes would pass 1.25 GiB.
static int idxk_chunk(int T, int Di, int ldw) {
    int c = T <= 16384 ? 128 : 256;
    while ((size_t)((ldw * 32 + c - 1) / c) * T * Di * 4 > ((size_t)5 << 28) && c < (1 << 20)) c *= 2;
    return c;
}
extern "C" hipError_t dsa_launch_indexer_bwd_gather(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                                                    const float *dscore, const float *grad, int ldw, const int32_t *cu, int N, int T, int Hi, int Di, int K,
                                                    float cscale, void *dq_idx, void *dw, int dw_bf16, hipStream_t stream);   // dsa_tile_idxg.hip
template <int D, int GS>
static hipError_t launch_idx_bwd_i(hipStream_t stream, const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n, const float *w_f32, const float *dscore,
                             const float *grad, const uint32_t *bitmap, const int32_t *prefix, int ldw, const int32_t *cu, int N, int T, int Hi,
                             int K, float cscale, void *dq_idx, void *dk_idx, void *dw, int dw_bf16, float *partial, hipStream_t stream_q) {
    // (waves that share the staged key tiles: two workgroups of four on a CU do not meet at each other's barriers, so the gating of
    // one runs beside the matrix work of the other - head_dim 128, 32 768 tokens: 2340 -> 2250 us against one of eight)
    constexpr int NW = 4;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&dsa_tile_idxk_kernel<D, GS>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)idxk_lds_bytes<D>());
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&dsa_tile_idxq_kernel<D, GS, NW>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)idxq_lds_bytes<D, NW>());
    if (e != hipSuccess) return e;
    // (the key side, the longer pass, is issued first: with two streams it gets the GPU first)
    const int chunk = idxk_chunk(T, D, ldw);
    const dim3 gk((unsigned)((int64_t)T / 128 + N + 1), (unsigned)((ldw * 32 + chunk - 1) / chunk));
    hipLaunchKernelGGL((dsa_tile_idxk_kernel<D, GS>), gk, dim3(256), idxk_lds_bytes<D>(), stream, (const bf16_t *)q_idx,
                       (const bf16_t *)k_idx, w_f32, dscore, grad, bitmap, prefix, ldw, cu, N, T, Hi, K, cscale, chunk, partial);
    hipLaunchKernelGGL(dsa_idxk_reduce_kernel, dim3((unsigned)((T + 7) / 8)), dim3(256), 0, stream, partial, cu, N, T, D,
                       chunk, ldw * 32, (bf16_t *)dk_idx);
    // segment by segment: the bound of the longest one only says which of the two kernels can have any
    if (idx_segment_gathers(Hi, K, ldw * 32)) {
        e = dsa_launch_indexer_bwd_gather(q_idx, k_idx, w_idx, idx, n, dscore, grad, ldw, cu, N, T, Hi, D, K, cscale, dq_idx, dw, dw_bf16, stream_q);
        if (e != hipSuccess) return e;
    }
    const dim3 gq((unsigned)((int64_t)T / ((32 * NW) >> GS) + N + 1));
    hipLaunchKernelGGL((dsa_tile_idxq_kernel<D, GS, NW>), gq, dim3(64 * NW), (idxq_lds_bytes<D, NW>()), stream_q, (const bf16_t *)q_idx,
                       (const bf16_t *)k_idx, (const bf16_t *)w_idx, dscore, grad, bitmap, ldw, cu, N, T, Hi, K, cscale,
                       (bf16_t *)dq_idx, dw, dw_bf16);
    return hipGetLastError();
}
extern "C" size_t dsa_indexer_bwd_partial_bytes(int T, int Di, int ldw) {
    const int chunk = idxk_chunk(T, Di, ldw);
    return (size_t)((ldw * 32 + chunk - 1) / chunk) * T * Di * 4;
}
// w_f32: T * 64 floats of scratch; grad: one fp32 factor of every gradient on the device, or null
extern "C" hipError_t dsa_launch_indexer_bwd(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                                             const float *dscore, const float *grad, const uint32_t *bitmap, int32_t *prefix, float *w_f32, int ldw, const int32_t *cu, int N,
                                             int T, int Hi, int Di, int K, float cscale, void *dq_idx, void *dk_idx,
                                             void *dw, int dw_bf16, float *partial, hipStream_t stream, hipStream_t stream_q) {
    if (Hi < 1 || Hi > 64 || !(Di == 64 || Di == 128)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(dsa_bitmap_prefix_kernel, dim3(T), dim3(64), 0, stream, bitmap, ldw, prefix, (const bf16_t *)w_idx, Hi, w_f32);
#define IDX_BWD(D_, GS_) launch_idx_bwd_i<D_, GS_>(stream, q_idx, k_idx, w_idx, idx, n, w_f32, dscore, grad, bitmap, prefix, ldw, cu, N, T, Hi, K, \
                                                   cscale, dq_idx, dk_idx, dw, dw_bf16, partial, stream_q)
    if (Di == 128) return Hi > 32 ? IDX_BWD(128, 6) : IDX_BWD(128, 5);
    return Hi > 32 ? IDX_BWD(64, 6) : IDX_BWD(64, 5);
#undef IDX_BWD
}
