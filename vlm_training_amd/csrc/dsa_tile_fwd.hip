// Attention forward over 32x32 MFMA tiles, query-stationary, selection (or the causal limit) as a bit mask.
//
// A workgroup holds 32*NW rows - a row is one (query, head of the kv group) - of one segment and kv head and walks the keys in
// tiles of 32:
//   S^T[key,row] = K[key,:].Q[row,:]            (A = K tile row-wise from LDS, B = Q^T in registers)
//   online softmax on the C layout (lane = row; one cross-lane step per statistic)
//   O^T[d,row]  += V^T[d,key] P^T[key,row]      (A = V tile transposed from LDS, B = P^T from the C layout)
//
// Each wave runs three tiles at once: step t issues the MFMAs of O += P(t) V(t) and of S(t+2) in pairs, and the softmax of
// tile t+1 stands between the pairs, a fixed number of elements behind each (every pair ends in an empty asm statement its
// results pass through, which fixes that order).  So the vector work of a tile - as long as its matrix work - runs in the
// MFMAs' shadow of the same wave, and the LDS operands are read four MFMA pairs ahead, across the tile's end.
//
// K and V tiles go from memory straight into LDS (buffer_load ... lds), rings of four: step t requests K(t+5) and V(t+3), at
// its end waits for what step t-1 requested and meets the barrier; rows past the segment and columns past the true head_dim
// read as zero.  The selection words take the same way, each wave its own rows' into its own slots.
//
// What bounds it: the power of the chip (MFMA busy 0.61 of a CU's time without a selection, at 1.79 GHz) and, with a selection, the
// vector instructions (about 92 and 16 exponentials beside 16 MFMAs at head_dim 128, 32 of them the mask); the softmax of tiles every row
// attends whole drops the mask: all but the last without a selection, those of blocks inside the first K positions with one (`window`; the
// same in dQ.  Step of 8192 tokens, K = 1024: 300.2 -> 295.4 us, forward of 16 384 in mixed segments, K = 2048: 673 -> 661).  Both make every instruction beside the MFMAs count: a tile's buffer size comes from two
// constants, its pieces follow one another under one buffer, operand addresses move on in place.  Same box, us, against a size formed per
// piece, addresses formed per tile and eight waves per workgroup in large launches: 32 768 tokens dense 1289 -> 1229, with a selection
// 1408 -> 1371; 8192 tokens with a selection 62.5 -> 59; 512 tokens 15.9 -> 15.1; head_dim 256, 16 384 tokens 210 -> 195; vision towers at
// head_dim 72 354 -> 335, at 64 282 -> 269.  Four waves per workgroup, two workgroups per CU: eight waves that share each staged tile took
// 1255 dense.  64 rows per wave, one wave per SIMD: level at 32 768 tokens (MFMA busy 0.52 at 1.95 GHz), slower in short launches.
// What a block costs beside its tiles, clocks at head_dim 256 / 128: 26 000 / 15 000 when its segment was searched for one by one, q read where it lies
// (each load touches 32 rows), the first tiles waited for all together and the output stored 32 bytes of a row at a time.  Search by a prefix
// sum, q through LDS in whole rows, S(0) and S(1) as soon as K(0) and K(1) are there, output in whole rows.  Forward of 16 384 tokens, us,
// head_dim 128, 16 heads over 8, segments of 64 / 256 / 1024 / 2048: 215 / 68.6 / 95.7 / 164.8 -> 45 / 51.5 / 91 / 162; head_dim 256, 16 heads over 2, of 64 / 256 /
// 512 / 1024 / 2048: 227 / 151 / 165 / 214 / 316 -> 106 / 129 / 142 / 190 / 308, there most of the rest is q and the output at 3 to 5 TB/s, which one workgroup per CU
// does not hide.
// At head_dim 256 the sums lie in accumulation registers by name: left to the compiler the loops of three of the four instances read spilled
// registers, and such a read waits for every tile on its way into LDS (+ 20 %).
#include "dsa_tile.h"

template <int D, int NW>
constexpr size_t fwd_lds_bytes(bool has_idx) { return 8 * (size_t)DirectTile<D>::BYTES + (has_idx ? NW * 4 * 256 : 0); }

// NEG: the softmax scale is negative.  A masked key's logit is -inf in front of the scale, and the largest one is searched for there, so
// the kernel's scale is positive and the sign goes into q (an instance of its own: at head_dim 256 as little as a test of the sign in front
// of the loop made it spill).
// AGPR: the sums in accumulation registers, by name (mfma32_agpr_late).  ROUNDS: more than one round of workgroups; a launch of one reads q
// where it lies, beside the tiles, and stores the output so: each way through LDS is one more latency of the block, and nothing else uses the
// path to memory (197 tokens 8.8 against 9.2 us; from two rounds on 1.5 to 5 % less with them).
template <int D, bool HAS_IDX, int NW, bool NEG, bool CARRIED, bool AGPR, bool ROUNDS>
__global__ __launch_bounds__(NW * 64, (D <= 128 && NW == 4) ? 2 : 1) void dsa_tile_fwd_kernel(
    const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, int64_t q_tok, int64_t q_head,
    int64_t k_tok, int64_t k_head, int64_t v_tok, int64_t v_head, const uint32_t *__restrict__ bitmap, int ldw,
    const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv, int gshift, int d_real, float scale_log2, int pos_split, int split_len, int pos_short, int window, int causal,
    bf16_t *__restrict__ out, float *__restrict__ lse) {
    typedef DirectTile<D> TL;
    // MFMAs of S, of P V (head_dim 80: five and six) and pairs of a step (one of each while there are)
    constexpr int KS = CARRIED ? DSA_CARRIED_KS : D / 16, DT = CARRIED ? 4 : (D + 31) / 32, NP = 2 * DT, NS = KS > NP ? KS : NP;
    static_assert(KS <= NP || D > 128);
    constexpr int LPW = (TL::LOADS + NW - 1) / NW;          // wave loads per wave, step and operand
    constexpr int LPS = 2 * LPW + (HAS_IDX ? 1 : 0);        // everything a wave requests in a step
    static_assert(TL::LOADS % NW == 0, "every wave loads the same number of pieces");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];    // 4 K slots | 4 V slots | selection words

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv, kvh = blockIdx.x % Hkv, QBW = (NW * 32) >> gshift;
    int s0, L, blk;
    if (!LOCATE_QUERY_BLOCK(causal, gridDim.x, cu, N, blockIdx.x / Hkv, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = __builtin_amdgcn_readfirstlane(L);
    if (HAS_IDX) L = min(L, ldw * 32);                  // a bitmap row has ldw words whatever the caller's max_seqlen
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (qc0 >= min(L, tile_rows_end(L, pos_split, split_len, pos_short))) return;       // rows past the split are not the tile kernels'
    const int ntiles = (causal ? min(qc0 + QBW - 1, L - 1) : L - 1) / 32 + 1;

    const int r = wv * 32 + j;
    const int qcol = qc0 + (r >> gshift), head = r & ((1 << gshift) - 1);
    const bool row_ok = qcol < L && head < G;
    const int t = s0 + min(qcol, L - 1), hq = kvh * G + min(head, G - 1);
    const int klim = causal ? qcol : L - 1;             // last key column this row may attend (dense mode)

    // ---- requests ----
    const int chunks = CARRIED ? 2 * KS : d_real / 8;
    const int64_t k_step = 32 * k_tok * 2, v_step = 32 * v_tok * 2;      // bytes per tile
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k + (int64_t)s0 * k_tok + (int64_t)kvh * k_head);
    const unsigned char *vptr = reinterpret_cast<const unsigned char *>(v + (int64_t)s0 * v_tok + (int64_t)kvh * v_head);
    constexpr int NV = LPW < TL::SOURCES ? LPW : TL::SOURCES;   // the lane's source offsets repeat after that many pieces
    int kvoff[NV], vvoff[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        kvoff[i] = TL::source(wv * LPW + i, lane, (int)k_tok * 2, chunks);
        vvoff[i] = TL::source(wv * LPW + i, lane, (int)v_tok * 2, chunks);
    }
    const uint32_t lds0 = lds_address(dyn_lds);
    // Addresses of the next tile to request, in scalar registers (the asm statements keep them there); the bytes of its rows that exist
    // bound the buffer (the last row ends with its own elements: a token stride may be shorter than a row, or zero, in an expanded
    // tensor; rows past the segment are then bytes of live rows, and masked as ever)
    auto next = [](const unsigned char *&p, int64_t step) __attribute__((always_inline)) {
        p += step;
        asm volatile("" : "+s"(p));
    };
    const int gone = max(ntiles * 32 - L, 0);           // rows of the last tile that do not exist
    const uint32_t k_full = 31 * (int)k_tok * 2 + d_real * 2, v_full = 31 * (int)v_tok * 2 + d_real * 2;
    const uint32_t k_last = k_full - gone * (int)k_tok * 2, v_last = v_full - gone * (int)v_tok * 2;
    auto load_tile = [&](const unsigned char *&p, const int (&first)[NV], int tile, int slot, uint32_t full, uint32_t last, int64_t tile_b) __attribute__((always_inline)) {
        int voff[LPW];
#pragma unroll
        for (int i = 0; i < LPW; ++i) voff[i] = first[i % NV] + i / NV * NV * TL::LOAD_ROWS * (int)(tile_b / 32);
        constexpr int P1 = LPW > 1 ? 1 : 0, P2 = LPW > 2 ? 2 : P1, P3 = LPW > 2 ? 3 : P2;
        buffer_load_lds16_n<LPW, TL::load_lds(P1), TL::load_lds(P2) - TL::load_lds(P1), TL::load_lds(P3) - TL::load_lds(P2)>(
            scalar_buffer_rsrc(p, tile < ntiles - 1 ? full : tile == ntiles - 1 ? last : 0u), voff, lds0 + slot * TL::BYTES + TL::load_lds(wv * LPW));
        next(p, tile_b);
    };
    auto load_k = [&](int tile) __attribute__((always_inline)) { load_tile(kptr, kvoff, tile, tile & 3, k_full, k_last, k_step); };
    auto load_v = [&](int tile) __attribute__((always_inline)) { load_tile(vptr, vvoff, tile, 4 + (tile & 3), v_full, v_last, v_step); };
    unsigned char *const words = dyn_lds + 8 * TL::BYTES + wv * 1024;     // [tile % 4][lane]
    const int wq0 = __builtin_amdgcn_readfirstlane(min(qc0 + ((wv * 32) >> gshift), L - 1));   // the wave's first query
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + wq0) * ldw);
    const int wvoff = (t - s0 - wq0) * ldw * 4;         // (at most 31 rows of bitmap)
    auto load_w = [&](int tile) __attribute__((always_inline)) {
        if (HAS_IDX) {
            buffer_load_lds4(make_buffer_rsrc(wptr, 32 * ldw * 4), wvoff, lds0 + 8 * TL::BYTES + wv * 1024 + (tile & 3) * 256);
            next(wptr, tile + 1 < ntiles ? 4 : 0);       // (past the block's tiles: the last word again, never used)
        }
    };
    // The wave's rows of q, whole rows at a time into the V slot of its number and from there into registers (read where they lie, each load
    // would touch 32 rows); rows that are not on 16-byte boundaries or too far apart for an offset: where they lie
    bf16x8 qB[KS];
    TL tl;
    tl.init(lane);
    const bool staged = ROUNDS && !((reinterpret_cast<uintptr_t>(q) | (uintptr_t)(q_tok * 2) | (uintptr_t)(q_head * 2)) & 15) &&
                        31 * q_tok + (int64_t)(G - 1) * q_head < (1 << 30) - D;
    if (staged) {
        const buffer_rsrc rows = make_buffer_rsrc(q + (int64_t)(s0 + wq0) * q_tok + (int64_t)kvh * G * q_head, 0x7fffffff);
        const WaveRows<TL> wr(gshift, lane);
        const int there = L - (qc0 + ((wv * 32) >> gshift)), tok_b = (int)q_tok * 2, head_b = (int)q_head * 2, place = wr.place(tok_b, head_b);
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i) {
            const int c = (lane % TL::CPR) ^ TL::xor_of(i * TL::LOAD_ROWS + lane / TL::CPR);
            const int off[1] = {wr.query(i) < there && wr.head(i) < G && c < chunks ? place + wr.piece(i, tok_b, head_b) + c * 16 : (int)0x80000000};
            buffer_load_lds16_n<1, 0, 0, 0>(rows, off, lds0 + (4 + wv) * TL::BYTES + TL::load_lds(i));
        }
    }
    if (!staged) {
        const bf16_t *const qrow = q + (int64_t)t * q_tok + (int64_t)hq * q_head;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qB[ks] = row_ok && 2 * ks + h < chunks ? load_bf16x8(qrow + 16 * ks + 8 * h) : zero_bf16x8();
    }
    load_k(0); load_w(0); load_k(1); load_w(1);
    if (!staged) load_v(0);
    load_k(2); load_w(2);
    if (!staged) load_v(1);
    load_k(3); load_w(3);
    if (!staged) load_v(2);
    constexpr int AFTER_K1 = 2 * LPW + (HAS_IDX ? 2 : 0);
    if (staged) {
        wait_vmcnt<AFTER_K1>();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            qB[ks] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>((lds_u8 *)dyn_lds + (4 + wv) * TL::BYTES + tl.rowq[TL::row_q(ks)] + TL::row_imm(ks));
    }
    if (NEG) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qB[ks] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, qB[ks]) ^ 0x80008000u);
    }
    f32x16 oacc[DT], sE, sO;                            // S of even and of odd tiles
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        oacc[dt] = zero16();
        if (AGPR) settle(oacc[dt]);
    }
    uint32_t pE[8], pO[8];                              // P of even and of odd tiles, packed (keys 0-15 | 16-31)
    float mrun = -INFINITY, lsum = 0.f;
    auto meet_read = [&]() __attribute__((always_inline)) {               // (what this wave reads of LDS is read)
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
        barrier_only();
    };
    if (staged) wait_vmcnt<AFTER_K1>();                 // K(0) and K(1) are there
    else wait_vmcnt<0>();
    meet_read();
    if (staged) {
        load_v(0); load_v(1); load_v(2);
    }

    lds_u8 *ka_[4], *va_[4];                            // operand addresses: of the K tile of S(t+2) and of V(t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ka_[i] = (lds_u8 *)dyn_lds + tl.rowq[i];
        va_[i] = (lds_u8 *)dyn_lds + tl.trq[i] + 4 * TL::BYTES;
    }
    auto advance = [&](lds_u8 *(&a)[4], int tile) __attribute__((always_inline)) {         // from tile - 1 to tile
        const int by = tile & 3 ? TL::BYTES : -3 * TL::BYTES;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] += by;
            asm volatile("" : "+v"(a[i]));
        }
    };
    auto read_k = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8 *>(ka_[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto read_v = [&](int i) __attribute__((always_inline)) {             // MFMA i of P V: keys of half i / DT, d-tile i % DT
        const int pair = i / DT, dt = i % DT;
        return tr_pair(va_[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair), va_[TL::tr_q(dt)] + TL::tr_imm(dt, 2 * pair + 1));
    };
    // The keys of a tile this lane keeps, as they lie in memory; live(word): element vi then sits at bit 8*(vi/4) + vi%4
    const uint32_t row_mask = row_ok ? 0xffffffffu : 0u;
    auto live = [&](uint32_t w) __attribute__((always_inline)) { return (w >> (4 * h)) & row_mask; };
    auto word_of = [&](int tile) __attribute__((always_inline)) {
        return HAS_IDX ? *reinterpret_cast<const uint32_t *>(words + (tile & 3) * 256 + lane * 4) : causal_bits(klim - tile * 32);
    };
    // The row maximum is not searched in every tile: P is formed against the running reference first, and only when a
    // lane's sum says that some probability may have passed 2^8 - or a live row has not met a selected key yet - does the wave
    // look for the tile's maximum, move the reference, rescale the sums and form P again: the first tile of a block, then
    // rarely.  In between P stays below 2^8, exact in fp32 and safe in bf16, and never underflows as a whole, because the
    // reference is a maximum the row has really met.
    auto masked = [&](float s, uint32_t word, int vi) __attribute__((always_inline)) {
        return keep_or_neginf(s, bit_mask(word, 8 * (vi >> 2) + (vi & 3)));
    };
    auto settle = [&](const f32x16 &s, uint32_t word, uint32_t (&p)[8], float &psum) __attribute__((always_inline)) {
        if (__builtin_amdgcn_ballot_w64(row_ok && (mrun == -INFINITY || !(psum <= 256.f)))) {
            asm volatile("" : "+v"(word));              // (nothing of the fast path is kept alive for this one)
            float mloc = -INFINITY;
#pragma unroll
            for (int vi = 0; vi < 16; ++vi) mloc = fmaxf(mloc, masked(s[vi], word, vi));
            mloc = half_max_f(mloc) * scale_log2;
            if (mloc > mrun) {
                const float alpha = fast_exp2(mrun - mloc);   // mrun = -inf: 0, and the sums are 0
                lsum *= alpha;
                if (AGPR) asm volatile("s_nop 11" : : : "memory");
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    if (AGPR) ::settle(oacc[dt]);
                    oacc[dt] *= alpha;
                    if (AGPR) ::settle(oacc[dt]);
                }
                mrun = mloc;
            }
            const float mneg = (mrun == -INFINITY) ? 0.f : -mrun;
            psum = 0.f;
#pragma unroll
            for (int vi = 0; vi < 16; vi += 2) {
                const float a = fast_exp2(fmaf(masked(s[vi], word, vi), scale_log2, mneg));
                psum += a;
                const float b = fast_exp2(fmaf(masked(s[vi + 1], word, vi + 1), scale_log2, mneg));
                psum += b;
                p[vi >> 1] = pack2bf(a, b);
            }
        }
        lsum += psum;
    };
    // S of tiles 0 and 1, P of tile 0
    auto gemm_s = [&](f32x16 &s) __attribute__((always_inline)) {
        s = zero16();
        bf16x8 ka[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) ka[ks] = read_k(ks);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s = mfma32(ka[ks], qB[ks], s);
    };
    gemm_s(sE);
    advance(ka_, 1);
    if (ntiles > 1) gemm_s(sO);
    {
        float psum = INFINITY;                          // (no reference yet: the maximum is searched for)
        if (!row_ok) psum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) pE[i] = 0u;
        settle(sE, live(word_of(0)), pE, psum);
    }
    wait_vmcnt<LPW>();                                  // all but V(2): step 0 reads its first operands of V(1) itself
    meet_read();                                        // every wave is done with K(0) and K(1): their slots may be filled again
    load_k(4);
    constexpr int KA = KS % 5 == 0 ? 5 : KS % 4 ? 3 : 4, VA = NP % 4 ? 3 : 4;   // (divide KS and NP: an operand keeps its register from step to step)
    static_assert(KS % KA == 0 && NP % VA == 0);
    bf16x8 kr[KA], vr[VA];                              // operands of the next MFMA pairs
    advance(ka_, 2);
#pragma unroll
    for (int i = 0; i < KA; ++i) kr[i] = read_k(i);
#pragma unroll
    for (int i = 0; i < VA; ++i) vr[i] = read_v(i);
    uint32_t word_next = word_of(1);                    // (one-tile blocks never use it)

    // what step t requests: K(t+5), V(t+3), the selection words of tile t+4
    auto request = [&](int t_, int r_) __attribute__((always_inline)) {
        if (r_ == 0) load_k(t_ + 5);
        else if (r_ == 1) load_v(t_ + 3);
        else load_w(t_ + 4);
    };
    // Step t: O += P(t) V(t) with `p`; softmax of tile t+1 from `s` into `pn` (SM); S(t+2) into `sn` (NEXT).
    auto step = [&](auto masked_, auto sm_, auto next_, auto req_, int t_, const uint32_t (&p)[8], const f32x16 &s, uint32_t (&pn)[8],
                    f32x16 &sn) __attribute__((always_inline)) {
        constexpr bool MASKED = decltype(masked_)::value, SM = decltype(sm_)::value, NEXT = decltype(next_)::value, REQ = decltype(req_)::value;
        const u32x4 w0 = {p[0], p[1], p[2], p[3]}, w1 = {p[4], p[5], p[6], p[7]};
        const bf16x8 pB0 = __builtin_bit_cast(bf16x8, w0), pB1 = __builtin_bit_cast(bf16x8, w1);
        const uint32_t word = MASKED ? live(word_next) : 0xffffffffu;
        float psum = 0.f;
        const float mneg = (mrun == -INFINITY) ? 0.f : -mrun;
        f32x16 snew;
        // The softmax of an element is a chain of dependent instructions (mask, scale, exponential, sum, pack) and a wave
        // issues in order: behind each MFMA stand the first part of one element's chain, the exponential of the element before
        // and the sum of the one before that, so that no instruction waits for the one in front of it.
        constexpr int H = 2 * NS - 2;                   // half-steps an element can start in
        float y[16], e[16];
        auto behind = [&](int hs) __attribute__((always_inline)) {
#pragma unroll
            for (int vi = 16 * (hs - 2) / H; vi < 16 * (hs - 1) / H; ++vi)
                if (hs >= 2) {
                    psum += e[vi];
                    if (vi & 1) {
                        pn[vi >> 1] = pack2bf(e[vi - 1], e[vi]);
                        asm volatile("" : "+v"(pn[vi >> 1]));
                    }
                }
#pragma unroll
            for (int vi = 16 * (hs - 1) / H; vi < 16 * hs / H; ++vi)
                if (hs >= 1 && hs <= H) {
                    e[vi] = fast_exp2(y[vi]);
                    asm volatile("" : "+v"(e[vi]));
                }
#pragma unroll
            for (int vi = 16 * hs / H; vi < 16 * (hs + 1) / H; ++vi)
                if (hs < H) {
                    y[vi] = fmaf(MASKED ? masked(s[vi], word, vi) : s[vi], scale_log2, mneg);
                    asm volatile("" : "+v"(y[vi]));
                }
            asm volatile("" : "+v"(psum) : : "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < (NEXT ? NS : NP); ++i) {
            if (i < NP) {
                if (AGPR) mfma32_agpr_late(oacc[i % DT], vr[i % VA], i < DT ? pB0 : pB1, !SM);
                else oacc[i % DT] = mfma32(vr[i % VA], i < DT ? pB0 : pB1, oacc[i % DT]);
            }
            // this step's requests, spread over its first half: one after the other they would queue for the way into LDS
#pragma unroll
            for (int r_ = 0; r_ < (HAS_IDX ? 3 : 2); ++r_)
                if (REQ && r_ * (NP / 2) / 3 == i) request(t_, r_);
            // refill: the operand a few pairs on, of this step's tiles or, past their end, of the next step's
            if (i == NP - VA && SM) advance(va_, t_ + 1);
            if (i < NP && (i + VA < NP || SM)) vr[i % VA] = read_v((i + VA) % NP);
            if (SM) behind(2 * i);
            else __builtin_amdgcn_sched_barrier(0);
            if (NEXT && i < KS) {
                snew = mfma32(kr[i % KA], qB[i], i == 0 ? zero16() : snew);
                if (i == KS - KA) advance(ka_, t_ + 3);
                kr[i % KA] = read_k((i + KA) % KS);
                if (i == 0 && MASKED) word_next = word_of(t_ + 2);
            }
            if (SM) behind(2 * i + 1);
        }
        if (SM) settle(s, word, pn, psum);
        if (NEXT) sn = snew;
    };
    const std::true_type yes;
    const std::false_type no;
    auto meet = [&]() __attribute__((always_inline)) {
        wait_vmcnt<LPS>();                              // all but what this step requested
        barrier_only();
    };
    auto full_step = [&](auto masked_, int t_, const uint32_t (&p)[8], const f32x16 &s, uint32_t (&pn)[8], f32x16 &sn) __attribute__((always_inline)) {
        step(masked_, yes, yes, yes, t_, p, s, pn, sn);
        meet();
    };
    int tt = 0;
    {
        // tiles every row of the block attends whole: the softmax without mask arithmetic (a loop of its own, not a branch
        // in the loop: two bodies that meet again would keep two sets of accumulators)
        const int whole = (HAS_IDX && min(qc0 + QBW, L) > window ? 0 : causal ? qc0 : L) / 32;
        for (; tt + 3 < ntiles && tt + 2 < whole; tt += 2) {
            full_step(no, tt, pE, sO, pO, sE);
            full_step(no, tt + 1, pO, sE, pE, sO);
        }
        word_next = word_of(tt + 1);
    }
    if constexpr (D > 128) {
        // (S of up to two tiles past the end is formed for nothing: the exact tail below costs registers this head_dim lacks)
        for (; tt + 2 < ntiles; tt += 2) {
            full_step(yes, tt, pE, sO, pO, sE);
            full_step(yes, tt + 1, pO, sE, pE, sO);
        }
        if (tt + 1 < ntiles) {
            full_step(yes, tt, pE, sO, pO, sE);
            step(yes, no, no, no, tt + 1, pO, sE, pE, sO);
        } else {
            step(yes, no, no, no, tt, pE, sO, pO, sE);
        }
    } else {
        for (; tt + 3 < ntiles; tt += 2) {
            full_step(yes, tt, pE, sO, pO, sE);
            full_step(yes, tt + 1, pO, sE, pE, sO);
        }
        // at most three tiles are left
        if (tt + 2 < ntiles) {
            full_step(yes, tt, pE, sO, pO, sE);
            step(yes, yes, no, yes, tt + 1, pO, sE, pE, sO);
            meet();
            step(yes, no, no, no, tt + 2, pE, sO, pO, sE);
        } else if (tt + 1 < ntiles) {
            step(yes, yes, no, yes, tt, pE, sO, pO, sE);
            meet();
            step(yes, no, no, no, tt + 1, pO, sE, pE, sO);
        } else {
            step(yes, no, no, no, tt, pE, sO, pO, sE);
        }
    }
    wait_vmcnt<0>();                                    // no load is left on its way into LDS when the workgroup ends

    const float l = half_sum_f(lsum), inv = 1.f / l;
    if constexpr (!ROUNDS) {
        if (row_ok) {
            if (h == 0) lse[(int64_t)hq * T + t] = (mrun + log2f(l)) * LN2_F;
            bf16_t *const row = out + ((int64_t)t * Hq + hq) * d_real;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                if (AGPR) ::settle(oacc[dt]);
                store_c_tile(row + dt * 32, oacc[dt], inv, h, chunks - 4 * dt);
            }
            if (CARRIED) {                              // V's third part is its first one, the last one zeros
                store_c_tile(row + 128, oacc[0], inv, h, 4);
                store_c_tile(row + 160, oacc[1], inv, h, 4);
                store_c_tile(row + 192, zero16(), inv, h, 4);
                store_c_tile(row + 224, zero16(), inv, h, 4);
            }
        }
    } else {
        // (where the rows lie is formed again: the loop needs its registers)
        int tid_ = tid;
        asm volatile("" : "+v"(tid_));
        const int lane_ = tid_ & 63, h_ = lane_ >> 5, j_ = lane_ & 31;
        {
            const int qc = qc0 + ((wv * 32 + j_) >> gshift), hd = j_ & ((1 << gshift) - 1);
            if (qc < L && hd < G && h_ == 0) lse[(int64_t)(kvh * G + hd) * T + s0 + qc] = (mrun + log2f(l)) * LN2_F;
        }
        // whole rows per store, through LDS (as in dQ)
        barrier_only();                                     // the rings are read out
        unsigned char *const rows_out = dyn_lds + wv * (32 * TL::ROW_B);
        auto chunk_at = [&](int row, int c) __attribute__((always_inline)) {
            return row * TL::ROW_B + ((c ^ (D == 64 ? (row >> 1) & 7 : row & 15)) << 4);
        };
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i = 0; i < 2; ++i) {                   // (chunks 4 dt + 2 i + h, as in store_c_tile)
                f32x16 &a = oacc[dt];
                if (AGPR && i == 0) ::settle(a);
                const uint32_t a0 = pack2bf(a[8 * i] * inv, a[8 * i + 1] * inv), a1 = pack2bf(a[8 * i + 2] * inv, a[8 * i + 3] * inv);
                const uint32_t b0 = pack2bf(a[8 * i + 4] * inv, a[8 * i + 5] * inv), b1 = pack2bf(a[8 * i + 6] * inv, a[8 * i + 7] * inv);
                const auto x0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);
                const auto x1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
                *reinterpret_cast<u32x4 *>(rows_out + chunk_at(j_, 4 * dt + 2 * i + h_)) = u32x4{x0[0], x1[0], x0[1], x1[1]};
            }
        // (all of them read in front of the first store: a read and its store in turn would wait for the LDS each time)
        u32x4 x[TL::LOADS];
        const int c = lane_ % TL::CPR;
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i) {
            x[i] = *reinterpret_cast<const u32x4 *>(rows_out + chunk_at(i * TL::LOAD_ROWS + lane_ / TL::CPR, CARRIED ? c & 15 : c));
            if (CARRIED && c >= 24) x[i] = u32x4{0u, 0u, 0u, 0u};             // (V's third part is its first one, the last one zeros)
        }
        const WaveRows<TL> wr(gshift, lane_);
        const int q0 = qc0 + ((wv * 32) >> gshift), tok_b = Hq * d_real * 2, place = wr.place(tok_b, d_real * 2) + c * 16;
        unsigned char *const to = reinterpret_cast<unsigned char *>(out + ((int64_t)(s0 + q0) * Hq + kvh * G) * d_real);
#pragma unroll
        for (int i = 0; i < TL::LOADS; ++i)
            if (q0 + wr.query(i) < L && wr.head(i) < G && (CARRIED || c < chunks)) *reinterpret_cast<u32x4 *>(to + (place + wr.piece(i, tok_b, d_real * 2))) = x[i];
    }
}

template <int D, bool HAS_IDX, bool CARRIED = false, bool AGPR = (D > 128)>
static hipError_t launch_fwd_i(hipStream_t stream, const void *q, const void *k, const void *v, const int64_t *st, const uint32_t *bitmap, int ldw,
                               const int32_t *cu, int N, int T, int Hq, int Hkv, int gshift, int d_real, float scale, int pos_split, int split_len, int pos_short, int window, int causal,
                               void *out, float *lse) {
    constexpr int NW = 4;
    const dim3 grid((unsigned)(((int64_t)T / ((32 * NW) >> gshift) + N + 1) * Hkv));
    const bool rounds = grid.x > (D > 128 ? 256 : 512);     // (one or two workgroups per CU)
    const auto kernel = scale < 0.f ? &dsa_tile_fwd_kernel<D, HAS_IDX, NW, true, CARRIED, AGPR, true>
                        : rounds    ? &dsa_tile_fwd_kernel<D, HAS_IDX, NW, false, CARRIED, AGPR, true>
                                    : &dsa_tile_fwd_kernel<D, HAS_IDX, NW, false, CARRIED, AGPR, false>;
    constexpr size_t lds = fwd_lds_bytes<D, NW>(HAS_IDX);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), lds, stream, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, st[0], st[1], st[2], st[3],
                       st[4], st[5], bitmap, ldw, cu, N, T, Hq, Hkv, gshift, d_real, fabsf(scale) * LOG2E_F, pos_split, split_len, pos_short, window, causal, (bf16_t *)out, lse);
    return hipSuccess;
}
// d_real: the head_dim of the tensors, a multiple of 8 (the kernel of the next head_dim of 64, 80, 96, 128, 256 runs it; 80 and 96
// without a bitmap only); window: rows of a bitmap at positions below it attend all of their causal window (0: nothing is known); carried: see
// DSA_CARRIED_KS; st: token and head stride of q, k and v in elements (rows of 16-byte alignment).  The file is compiled twice, the second time
// (FWD_256) for head_dim 256, with results of MFMA builtins in vector registers: the sums have the accumulation registers.
#define FWD_LAUNCH_ARGS const void *q, const void *k, const void *v, const int64_t *st, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, \
    int Hq, int Hkv, int d_real, float scale, int pos_split, int split_len, int pos_short, int window, int carried, int causal, void *out, float *lse, hipStream_t stream
#define FWD_CASE(D_, ...) e = launch_fwd_i<D_, __VA_ARGS__>(stream, q, k, v, st, bitmap, ldw, cu, N, T, Hq, Hkv, group_shift(Hq, Hkv), d_real, logit_scale(scale), \
                                                            pos_split, split_len, pos_short, window, causal, out, lse)
extern "C" hipError_t dsa_launch_tile_fwd_256(FWD_LAUNCH_ARGS);
#if FWD_256
extern "C" hipError_t dsa_launch_tile_fwd_256(FWD_LAUNCH_ARGS) {
    hipError_t e;
    if (carried) {
        if (bitmap) FWD_CASE(256, true, true);
        else FWD_CASE(256, false, true);
    } else if (bitmap) FWD_CASE(256, true);
    else FWD_CASE(256, false);                           // (of a negative scale)
    return e != hipSuccess ? e : hipGetLastError();
}
#else
extern "C" hipError_t dsa_launch_tile_fwd(FWD_LAUNCH_ARGS) {
    if (d_real > 256) return hipErrorInvalidValue;
    if (d_real > 128 && (bitmap || carried || scale < 0.f)) return dsa_launch_tile_fwd_256(q, k, v, st, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, pos_split, split_len, pos_short, window, carried, causal, out, lse, stream);
    hipError_t e;
    if (bitmap) {
        if (d_real <= 64) FWD_CASE(64, true);
        else FWD_CASE(128, true);
    } else {
        if (d_real <= 64) FWD_CASE(64, false);
        else if (d_real <= 80) FWD_CASE(80, false);
        else if (d_real <= 96) FWD_CASE(96, false);
        else if (d_real <= 128) FWD_CASE(128, false);
        else FWD_CASE(256, false, false, false);         // (without a mask in its loop it spills nothing there, and takes 2 to 4 % less)
    }
    return e != hipSuccess ? e : hipGetLastError();
}
#endif
