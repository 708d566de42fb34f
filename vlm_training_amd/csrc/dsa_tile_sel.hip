// Attention forward and dQ of query rows whose selection is thin (late rows of long segments): blocks of keys staged whole, walked compacted.
//
// A workgroup holds 32*NW rows - a row is one (query, head of the kv group) - of one segment and kv head, as the tile kernels do, and
// stages the keys in blocks of 128.  Of each block a wave runs only the keys that one of its own queries selected: it forms, lane by
// key, the set of its queries that selected the key, ranks the keys of a set that is not empty and lists them, 32 to a step of
//   S^T = K Q^T, online softmax, O^T += V^T P^T            (forward)
//   S^T = K Q^T, dP^T = V dO^T - delta, dQ^T += K^T dS^T   (dQ)
// on 32x32 MFMA tiles whose operand rows are gathered from the staged block.  Every row leaves out the keys it did not select, as in the
// tile kernels.  At one selected key in forty, eight queries a wave (four heads per kv head) run 24 of 128 keys, one step where the dense
// walk takes four, and a block read from L2 serves all queries of the workgroup (the gather kernels read every row's keys on its own: 0.6 TB
// past L2 at 131 072 tokens).
//
// What bounds it: the LDS (operand rows of a list lie where they lie: 1.8 clocks a read instead of 1.0, dQ 2.1; busy 0.53 and 0.56 of the time at
// 131 072 tokens), the vector instructions (about 100 a step, 45 more a block for the list; 0.47 and 0.36 of a SIMD's time, MFMAs 0.33 and 0.37) and the
// spread of the waves' steps between two barriers.  Rows beyond
// 16 K of 131 072 tokens, K = 2048, 32 heads over 8 kv heads, the whole forward / backward, ms: gathered 94.5 / 299; here with eight waves and a step's
// chain of reads and MFMAs open to its latency 76 / 297, twelve waves, lists built a block ahead 65 / 293, operands read ahead and nothing spilled
// 56 / 280, exponentials behind the MFMAs of dP 57 / 275.  With twelve waves a spilled register read in the loop waits for the blocks on their way into LDS (+ 25 %).
#include "dsa_sel.h"

#define SEL_KEYS 128                                     // keys of a block
#define SEL_AHEAD 2                                      // operands read ahead
// waves of a workgroup: three to a SIMD (more hide more of a step's chain of reads and MFMAs), two for dQ
constexpr int sel_waves(bool bwd) { return bwd ? 8 : 12; }
// LDS: two blocks of K and V | of each wave: selection words of three blocks, two lists
constexpr int SEL_WORD_B = 256, SEL_LIST_B = SEL_KEYS * 4, SEL_WAVE_B = 3 * SEL_WORD_B + 2 * SEL_LIST_B;
constexpr size_t sel_lds_bytes(bool bwd) { return 4 * (size_t)SelBlock<SEL_KEYS>::BYTES + sel_waves(bwd) * SEL_WAVE_B; }

// One row, the same for all lanes, over its own keys alone: sixteen lanes to a key, four keys at a time, fp32 throughout.
template <bool BWD>
__device__ __forceinline__ void sel_redo_row(const bf16_t *q, const bf16_t *k, const bf16_t *v, const bf16_t *dout, const float *lse_in, const float *delta,
                                             const uint32_t *bitmap, int ldw, int T, int Hq, int Hkv, float scale, float scale_log2, int s0, int L, int kvh, int t, int hq,
                                             bf16_t *out, float *lse) {
    constexpr int D = 128;
    const int lane = threadIdx.x & 63, g = lane >> 4, sub = lane & 15;
    auto eight = [](const bf16_t *p, float (&x)[8]) __attribute__((always_inline)) {
        const u32x4 w = __builtin_bit_cast(u32x4, load_bf16x8(p));
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(i & 1 ? w[i >> 1] & 0xffff0000u : w[i >> 1] << 16);
    };
    auto over_key = [](float x) __attribute__((always_inline)) {          // sum over the sixteen lanes of a key
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        return x;
    };
    const int64_t at = ((int64_t)t * Hq + hq) * D + sub * 8;
    float qf[8], df[8], acc[8], m = -INFINITY, l = 0.f, lse2 = 0.f, dlt = 0.f;
    eight(q + at, qf);
    if (BWD) {
        eight(dout + at, df);
        lse2 = lse_in[(int64_t)hq * T + t] * LOG2E_F;
        dlt = delta[(int64_t)hq * T + t];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    bool keys = false;
    for (int w0 = 0; w0 * 32 < L; w0 += 64) {
        const uint32_t mine = w0 + lane < ldw ? bitmap[(int64_t)t * ldw + w0 + lane] : 0u;
        for (uint64_t some = __builtin_amdgcn_ballot_w64(mine != 0u); some; some &= some - 1) {
            const int wl = (int)__builtin_ctzll(some);
            uint32_t word = (uint32_t)__builtin_amdgcn_readlane((int)mine, wl);
            while (word) {                           // four keys, one to each sixteen lanes
                int col = -1;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (i == g && word) col = (w0 + wl) * 32 + (int)__builtin_ctz(word);
                    word &= word - 1;
                }
                if (col >= 0 && col < L) {
                    keys = true;
                    const int64_t key = ((int64_t)(s0 + col) * Hkv + kvh) * D + sub * 8;
                    float kf[8], vf[8], s = 0.f, dp = 0.f;
                    eight(k + key, kf);
                    eight(v + key, vf);
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        s = fmaf(kf[i], qf[i], s);
                        if (BWD) dp = fmaf(vf[i], df[i], dp);
                    }
                    s = over_key(s) * scale_log2;
                    if (BWD) {
                        const float ds = fast_exp2(s - lse2) * (over_key(dp) - dlt);
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[i] = fmaf(ds, kf[i], acc[i]);
                    } else {
                        const float top = fmaxf(m, s), alpha = m == top ? 1.f : fast_exp2(m - top), p = s == -INFINITY ? 0.f : fast_exp2(s - top);
                        m = top;
                        l = fmaf(l, alpha, p);
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[i] = fmaf(p, vf[i], acc[i] * alpha);
                    }
                }
            }
        }
    }
    auto over_groups = [](float x) __attribute__((always_inline)) {
        x += __shfl_xor(x, 16, 64);
        return x + __shfl_xor(x, 32, 64);
    };
    float mul = scale;
    if (!BWD) {                                      // the four sums under one reference (a group that met no logit above -inf has none)
        float top = fmaxf(m, __shfl_xor(m, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float to = m == top ? 1.f : fast_exp2(m - top);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] *= to;
        l = over_groups(l * to);
        mul = l != 0.f ? 1.f / l : __builtin_amdgcn_ballot_w64(keys) ? NAN : 0.f;         // no key: zero output, lse = -inf; none above -inf: no softmax
        if (lane == 0) lse[(int64_t)hq * T + t] = (top + log2f(l)) * LN2_F;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = over_groups(acc[i]) * mul;
    if (g == 0) *reinterpret_cast<u32x4 *>(out + at) = u32x4{pack2bf(acc[0], acc[1]), pack2bf(acc[2], acc[3]), pack2bf(acc[4], acc[5]), pack2bf(acc[6], acc[7])};
}

// BWD: dQ (acc, out = dq) instead of the forward (acc, out, lse)
template <int GSHIFT, bool BWD>
__global__ __launch_bounds__(sel_waves(BWD) * 64, 1) void dsa_tile_sel_kernel(
    const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, const bf16_t *__restrict__ dout,
    const float *__restrict__ lse_in, const float *__restrict__ delta, const uint32_t *__restrict__ bitmap, int ldw,
    const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv, float scale, float logit_scale_, int pos_min, int pos_max, int split_len, bf16_t *__restrict__ out,
    float *__restrict__ lse) {
    typedef SelBlock<SEL_KEYS> BL;
    constexpr int D = BL::D, KS = D / 16, DT = D / 32, QW = 32 >> GSHIFT, NW = sel_waves(BWD), QBW = NW * QW;
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv, kvh = blockIdx.x % Hkv;
    int s0, L, blk;
    if (!LOCATE_QUERY_BLOCK(true, gridDim.x, cu, N, blockIdx.x / Hkv, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = __builtin_amdgcn_readfirstlane(L);
    L = min(L, ldw * 32);                               // a bitmap row has ldw words whatever the caller's max_seqlen
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (L < split_len) return;                          // short segments belong to the tile kernel,
    L = min(L, pos_max);                                // rows from there on to the gather kernel, rows before pos_min to the tile kernel
    if (qc0 + QBW <= pos_min || qc0 >= L) return;
    const int nblocks = min(qc0 + QBW - 1, L - 1) / SEL_KEYS + 1;

    // ---- requests ----
    const int tok_b = Hkv * D * 2;                      // bytes from one key row to the next
    const uint32_t lds0 = lds_address(dyn_lds);
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k + ((int64_t)s0 * Hkv + kvh) * D);
    const unsigned char *vptr = reinterpret_cast<const unsigned char *>(v + ((int64_t)s0 * Hkv + kvh) * D);
    const int voff[1] = {BL::load_row(wv, lane) * tok_b + BL::load_chunk(wv, lane) * 16};       // (a wave's later loads lie whole rows of the buffer further on)
    const int q0 = qc0 + wv * QW, wq0 = min(q0, L - 1);                   // the wave's first query
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + wq0) * ldw);
    const int wave_at = 4 * BL::BYTES + wv * SEL_WAVE_B;
    auto request = [&](int b) __attribute__((always_inline)) {            // K and V of block b, in block order
        if (wv < SEL_LOADERS) {
            constexpr int STEP = SEL_LOADERS * BL::LOAD_ROWS;             // rows from one of the wave's loads to the next
            const uint32_t at = lds0 + (b & 1) * 2 * BL::BYTES + wv * 1024;
#pragma unroll
            for (int i = 0; i < BL::LPW; ++i) {
                const int rows = min(L - b * SEL_KEYS - i * STEP, SEL_KEYS);                    // (rows past the segment read as zero)
                const uint32_t bytes = rows > 0 ? (rows - 1) * tok_b + D * 2 : 0;
                buffer_load_lds16_n<1, 0, 0, 0>(scalar_buffer_rsrc(kptr, bytes), voff, at + i * SEL_LOADERS * 1024);
                buffer_load_lds16_n<1, 0, 0, 0>(scalar_buffer_rsrc(vptr, bytes), voff, at + i * SEL_LOADERS * 1024 + BL::BYTES);
                kptr += (int64_t)STEP * tok_b;
                vptr += (int64_t)STEP * tok_b;
                asm volatile("" : "+s"(kptr), "+s"(vptr));
            }
        }
    };
    int words_to = 0;                                   // slot of the next block's words
    auto request_words = [&](int b) __attribute__((always_inline)) {      // likewise
        // lane l loads word l % 4 of query l / 4; words past the row's end: none.  (Formed anew for each block: it would cost the loop a register.)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const bool there = b * 4 + (ln & 3) < ldw;
        const int woff = __mul24(min(q0 + min(ln >> 2, QW - 1), L - 1) - wq0, ldw * 4) + (ln & 3) * 4;
        buffer_load_lds4(make_buffer_rsrc(wptr, 16 * (int64_t)ldw * 4), there ? woff : (int)0x80000000, lds0 + wave_at + words_to);
        wptr += 16;
        asm volatile("" : "+s"(wptr));
        words_to = words_to == 2 * SEL_WORD_B ? 0 : words_to + SEL_WORD_B;
    };
    request(0);
    request_words(0);
    if (nblocks > 1) request_words(1);

    // row j of the wave: (query, head of the group); a lane holds half h of every 16 elements
    const int qcol = q0 + (j >> GSHIFT), head = j & ((1 << GSHIFT) - 1);
    const bool row_ok = qcol >= pos_min && qcol < L && head < G;
    const int t = s0 + min(qcol, L - 1), hq = kvh * G + min(head, G - 1);
    const int64_t row_off = ((int64_t)t * Hq + hq) * D;
    const uint32_t flip = !BWD && logit_scale_ < 0.f ? 0x80008000u : 0u;  // (the forward searches the maximum in front of a positive scale)
    bf16x8 qB[KS], doB[BWD ? KS : 1];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        qB[ks] = row_ok ? load_bf16x8(q + row_off + 16 * ks + 8 * h) : zero_bf16x8();
        qB[ks] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, qB[ks]) ^ flip);
        if (BWD) doB[ks] = row_ok ? load_bf16x8(dout + row_off + 16 * ks + 8 * h) : zero_bf16x8();
    }
    const float scale_log2 = (BWD ? logit_scale_ : fabsf(logit_scale_)) * LOG2E_F;
    // minus the softmax's reference: the forward's moves, and is not a number until the row has met a key (its sums then ask for one)
    float mneg = row_ok ? NAN : 0.f, lsum = 0.f, dlt = 0.f;
    if (BWD) {
        mneg = -lse_in[(int64_t)hq * T + t] * LOG2E_F;
        dlt = delta[(int64_t)hq * T + t];
    }
    f32x16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();

    // A list's entry: the set of the wave's queries that selected the key (bit i: query i), its row of the block in the upper half.  Lane l
    // stands for the keys r = 32 * (l % 4) + l / 4 and r + 16, so that the list goes by class; slots behind its end have an empty set.
    // Slot i of a step is rank 2 i (i < 16) or 2 (i - 16) + 1 of the list: keys of one class lie on either side.
    const int cls = lane >> 2;
    const uint32_t e0 = (uint32_t)BL::entry(32 * (lane & 3) + cls) << 16;
    uint32_t *const lists = reinterpret_cast<uint32_t *>(dyn_lds + wave_at + 3 * SEL_WORD_B);
    const int qi = j >> GSHIFT, trs = (lane & 15) >> 2;
    const int tr_in = (((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) << 4 | (lane & 1) << 3;
    int words_at = 0;
    // the keys of the next block that a query of the wave selected: the sets of the lane's two keys, query by query, then the list
    uint32_t both = 0u;
    auto gather_sets = [&](int from, int to) __attribute__((always_inline)) {
        const uint32_t *w = reinterpret_cast<const uint32_t *>(dyn_lds + wave_at + words_at) + (lane & 3);
#pragma unroll
        for (int i = QW - 1 - from; i > QW - 1 - to; --i) both = both << 1 | (w[i * 4] >> cls & 0x10001u);
    };
    auto build = [&](uint32_t *list) __attribute__((always_inline)) {
        words_at = words_at == 2 * SEL_WORD_B ? 0 : words_at + SEL_WORD_B;
        const uint32_t m0 = both & 0xffffu, m1 = both >> 16;
        both = 0u;
        const uint64_t b0 = __builtin_amdgcn_ballot_w64(m0 != 0u), b1 = __builtin_amdgcn_ballot_w64(m1 != 0u);
        const int r0 = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b1 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b1, __builtin_amdgcn_mbcnt_hi((uint32_t)(b0 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b0, 0))));
        list[lane] = e0;
        list[lane + 64] = e0;
        if (m0) list[r0] = e0 | m0;
        if (m1) list[r0 + (m0 ? 1 : 0)] = (e0 + ((uint32_t)BL::entry(16) << 16)) | m1;
        return (int)__popcll(b0) + (int)__popcll(b1);
    };
    wait_vmcnt<0>();
    barrier_only();
    gather_sets(0, QW);
    int n = build(lists);
    // Operands are read at LDS addresses that XORs form; the blocks start at address 0, for the kernel has no other LDS.  Of a list: the
    // lane's row (row-wise), its rows (transposed), the sets of its slots
    const uint32_t list0 = lds0 + wave_at + 3 * SEL_WORD_B;
    uint32_t er_at = list0 + 2 + 4 * ((j & 15) * 2 + (j >> 4)), et_at = list0 + 2 + 8 * (4 * h + trs), set_at = list0 + 32 * h;
    asm volatile("" : "+v"(er_at), "+v"(et_at), "+v"(set_at));

    for (int b = 0; b < nblocks; ++b) {
        if (b + 1 < nblocks) request(b + 1);
        if (b + 2 < nblocks) request_words(b + 2);
        const int at = (b & 1) * 2 * BL::BYTES, list_at = (b & 1) * SEL_LIST_B;
        int n_next = 0;
        auto step = [&](auto first_, int st) __attribute__((always_inline)) {
            constexpr bool FIRST = decltype(first_)::value;
            const int er = (lds_read<uint16_t>(er_at + list_at + 4 * st) | at) ^ (h << 4), er1 = er ^ 32;
            int et[4];
            const uint32_t ets = et_at + list_at + 4 * st, sets = set_at + list_at + 4 * st;
#pragma unroll
            for (int u = 0; u < 4; ++u) et[u] = (lds_read<uint16_t>(ets + 64 * (u & 1) + 4 * (u >> 1)) | at) ^ tr_in;
            u32x4 set[4];                                // of slots 8 u + 4 h + i: element (u / 2 + 2 i) % 4 of set[2 (u % 2) + i / 2]
            auto row_op = [&](int ks, int operand) __attribute__((always_inline)) {
                return lds_read<bf16x8>((ks & 1 ? er1 : er) + (ks >> 1) * BL::COLUMN_B + operand * BL::BYTES);
            };
            auto tr_op = [&](int i) __attribute__((always_inline)) {                    // keys of half i / DT, d-tile i % DT
                const int pair = i / DT, dt = i % DT;
                constexpr int OPERAND = BWD ? 0 : BL::BYTES;
                return tr_pair((lds_u8 *)(et[2 * pair] + dt * BL::COLUMN_B + OPERAND), (lds_u8 *)(et[2 * pair + 1] + dt * BL::COLUMN_B + OPERAND));
            };
            auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
            constexpr int NR = BWD ? 2 * KS : KS, NT = 2 * DT;
            bf16x8 op[SEL_AHEAD];
            auto fetch = [&](int m) __attribute__((always_inline)) { return m < NR ? row_op(m % KS, m / KS) : tr_op(m - NR); };
#pragma unroll
            for (int m = 0; m < SEL_AHEAD; ++m) op[m] = fetch(m);
            fence();
            f32x16 s = zero16(), dp;
#pragma unroll
            for (int m = 0; m < KS; ++m) {
                s = mfma32(op[m % SEL_AHEAD], qB[m], s);
                op[m % SEL_AHEAD] = fetch(m + SEL_AHEAD);
                if (FIRST) gather_sets(m * QW / KS, (m + 1) * QW / KS);
                fence();
            }
            if (FIRST) n_next = build(lists + ((b + 1) & 1) * SEL_KEYS);    // (behind the last block: of old words, never used)
            auto read_sets = [&](int half) __attribute__((always_inline)) {
                set[2 * half] = lds_read<u32x4>(sets + 64 * half);
                set[2 * half + 1] = lds_read<u32x4>(sets + 64 * half + 16);
            };
            read_sets(0);
            if (BWD) read_sets(1);
            auto keep = [&](int vi) __attribute__((always_inline)) {
                const int u = vi >> 2, i = vi & 3;
                return (uint32_t)__builtin_amdgcn_sbfe((int)set[2 * (u & 1) + (i >> 1)][(u >> 1) + 2 * (i & 1)], qi, 1);
            };
            uint32_t p[8];
            if (BWD) {
#pragma unroll
                for (int vi = 0; vi < 16; ++vi) dp[vi] = -dlt;
#pragma unroll
                for (int m = 0; m < KS; ++m) {           // the exponentials behind the MFMAs of dP
                    dp = mfma32(op[(KS + m) % SEL_AHEAD], doB[m], dp);
                    op[(KS + m) % SEL_AHEAD] = fetch(KS + m + SEL_AHEAD);
#pragma unroll
                    for (int vi = 16 * m / KS; vi < 16 * (m + 1) / KS; ++vi)
                        s[vi] = fast_exp2(keep_or_neginf(fmaf(s[vi], scale_log2, mneg), keep(vi)));
                    fence();
                }
#pragma unroll
                for (int vi = 0; vi < 16; vi += 2) p[vi >> 1] = pack2bf(s[vi] * dp[vi], s[vi + 1] * dp[vi + 1]);
            } else {
                float psum = 0.f;
#pragma unroll
                for (int half = 0; half < 2; ++half) {   // (half of the sets at a time: registers)
#pragma unroll
                    for (int vi = 0; vi < 16; ++vi)
                        if ((vi >> 2 & 1) == half) s[vi] = keep_or_neginf(s[vi], keep(vi));
                    if (half == 0) {
                        fence();
                        read_sets(1);
                    }
                }
#pragma unroll
                for (int vi = 0; vi < 16; vi += 2) {
                    const float a = fast_exp2(fmaf(s[vi], scale_log2, mneg)), c = fast_exp2(fmaf(s[vi + 1], scale_log2, mneg));
                    psum = vi ? psum + a : a;
                    psum += c;
                    p[vi >> 1] = pack2bf(a, c);
                }
                // the reference moves as in the tile kernel: when a sum says so, or no key has been met yet
                if (__builtin_amdgcn_ballot_w64(!(psum <= 256.f))) {
                    float mloc = -INFINITY, mrun = mneg == mneg ? -mneg : -INFINITY;
#pragma unroll
                    for (int vi = 0; vi < 16; ++vi) mloc = fmaxf(mloc, s[vi]);
                    mloc = half_max_f(mloc) * scale_log2;
                    if (mloc > mrun) {
                        const float alpha = fast_exp2(mrun - mloc);       // mrun = -inf: 0, and the sums are 0
                        lsum *= alpha;
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
                        mrun = mloc;
                    }
                    const float m2 = mrun == -INFINITY ? 0.f : -mrun;
                    mneg = mrun == -INFINITY ? NAN : -mrun;
                    psum = 0.f;
#pragma unroll
                    for (int vi = 0; vi < 16; vi += 2) {
                        const float a = fast_exp2(fmaf(s[vi], scale_log2, m2)), c = fast_exp2(fmaf(s[vi + 1], scale_log2, m2));
                        psum += a;
                        psum += c;
                        p[vi >> 1] = pack2bf(a, c);
                    }
                }
                lsum += psum;
            }
            const u32x4 w0 = {p[0], p[1], p[2], p[3]}, w1 = {p[4], p[5], p[6], p[7]};
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                acc[i % DT] = mfma32(op[(NR + i) % SEL_AHEAD], __builtin_bit_cast(bf16x8, i < DT ? w0 : w1), acc[i % DT]);
                if (i + SEL_AHEAD < NT) op[(NR + i) % SEL_AHEAD] = fetch(NR + i + SEL_AHEAD);
                fence();
            }
        };
        step(std::true_type(), 0);
        for (int st = 32; st < n; st += 32) step(std::false_type(), st);
        n = n_next;
        wait_vmcnt<0>();
        barrier_only();
    }

    // (where the row lies is formed again: the loop needs its registers)
    int j_ = j;
    asm volatile("" : "+v"(j_));
    const int qcol_ = q0 + (j_ >> GSHIFT), head_ = j_ & ((1 << GSHIFT) - 1), hq_ = kvh * G + head_, t_ = s0 + qcol_;
    const bool there = qcol_ >= pos_min && qcol_ < L && head_ < G;
    const float l = BWD ? 0.f : half_sum_f(lsum);
    float odd = 0.f;                                     // 0, of a row that is not finite NaN
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int vi = 0; vi < 16; ++vi) odd = fmaf(acc[dt][vi], 0.f, odd);
    odd = half_sum_f(odd);
    if (there && odd == odd) {
        const float mul = BWD ? scale : l > 0.f ? 1.f / l : 0.f;          // nothing selected: zero output, lse = -inf
        bf16_t *const row = out + ((int64_t)t_ * Hq + hq_) * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store_c_tile(row + dt * 32, acc[dt], mul, h);
        if (!BWD && h == 0) lse[(int64_t)hq_ * T + t_] = ((mneg == mneg ? -mneg : -INFINITY) + log2f(l)) * LN2_F;
    }
    // Rows that are not finite are formed again, over their own keys alone, so that what a key holds reaches nothing that did not select it (as when
    // such rows were gathered): the probabilities of keys that a row left out are 0, but a step multiplies them with the V (dQ: K) of keys that the
    // wave's other rows selected, and 0 times Inf or NaN is NaN.  (Here, and not by a launch behind the walk that looks for NaN: that took 4 to 5 us
    // each way whether there was one or not.  40 000 tokens, 32 heads over 8, K = 2048, forward / backward: 11 / 34 ms, one Inf in V 79 / 118, every row of q NaN 83 / 118.)
    for (uint32_t again = (uint32_t)__builtin_amdgcn_ballot_w64(there && !(odd == odd)); again; again &= again - 1) {
        const int r = (int)__builtin_ctz(again);
        sel_redo_row<BWD>(q, k, v, dout, lse_in, delta, bitmap, ldw, T, Hq, Hkv, scale, logit_scale_ * LOG2E_F, s0, L, kvh, s0 + q0 + (r >> GSHIFT),
                          kvh * G + (r & ((1 << GSHIFT) - 1)), out, lse);
    }
}

template <int GSHIFT, bool BWD>
static hipError_t launch_sel_i(hipStream_t stream, const void *q, const void *k, const void *v, const void *dout, const float *lse_in, const float *delta,
                               const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int pos_min,
                               int pos_max, int split_len, void *out, float *lse) {
    const auto kernel = &dsa_tile_sel_kernel<GSHIFT, BWD>;
    constexpr size_t lds = sel_lds_bytes(BWD);
    constexpr int NW = sel_waves(BWD);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(((int64_t)T / (NW * 32 >> GSHIFT) + N + 1) * Hkv));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), lds, stream, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (const bf16_t *)dout, lse_in,
                       delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, logit_scale(scale), pos_min, pos_max, split_len, (bf16_t *)out, lse);
    return hipGetLastError();
}
// rows at positions pos_min (a multiple of 256) to pos_max - 1 of segments of split_len tokens and more; head_dim 128, two to four heads per kv head
extern "C" hipError_t dsa_launch_sel_fwd(const void *q, const void *k, const void *v, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T,
                                         int Hq, int Hkv, float scale, int pos_min, int pos_max, int split_len, void *out, float *lse, hipStream_t stream) {
    const auto launch = group_shift(Hq, Hkv) == 1 ? &launch_sel_i<1, false> : &launch_sel_i<2, false>;
    return launch(stream, q, k, v, nullptr, nullptr, nullptr, bitmap, ldw, cu, N, T, Hq, Hkv, scale, pos_min, pos_max, split_len, out, lse);
}
extern "C" hipError_t dsa_launch_sel_dq(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                                        const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int pos_min,
                                        int pos_max, int split_len, void *dq, hipStream_t stream) {
    const auto launch = group_shift(Hq, Hkv) == 1 ? &launch_sel_i<1, true> : &launch_sel_i<2, true>;
    return launch(stream, q, k, v, dout, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, pos_min, pos_max, split_len, dq, nullptr);
}
