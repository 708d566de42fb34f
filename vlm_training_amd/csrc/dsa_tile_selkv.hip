// dK, dV of long segments whose selection is thin: blocks of queries staged whole, walked compacted (the key side of dsa_tile_sel.hip).
//
// A workgroup owns 192 keys of one segment and kv head, 16 to a wave, and walks the queries from the segment's end down in blocks of 128 rows
// - a row is one (query, head of the kv group).  Of each block a wave runs only the queries that selected one of its own keys - those whose
// word of the selection bitmap has one of its 16 bits -, 32 rows to a step of
//   S = Q K^T, dP = dO V^T              (A = q / dO rows gathered from the staged block, B = the wave's K / V rows in registers; the sums
//                                        start from -lse/scale and -delta)
//   dV^T += dO^T P, dK^T += Q^T dS      (A = the same rows transposed, B = P / dS from the C layout)
// on 16x16x32 MFMA tiles.  At one selected key in forty two thirds of the queries are left out.  Every key row is reduced by one wave in a
// fixed query order: no atomics, bit-reproducible.
//
// What bounds it: nothing alone - at 131 072 tokens and one selected key in forty the LDS is busy for 0.52 of the time (0.13 of it bank conflicts), vector
// instructions (98 a step beside 32 MFMAs) take 0.43, the matrix cores 0.37 - but their sum, 0.87 of a SIMD's issue slots, and the spread of the waves'
// steps between two barriers.  Backward of 131 072
// tokens, K = 2048, ms: tile kernel 281; here with 32 keys a wave, eight waves and V in LDS (twice the queries per wave, two waves to a SIMD) 258,
// 16 keys and twelve waves 238, rows of a step picked by class (1.7 -> 1.1 clocks a read) 226.  An odd tile as a step of its own (half the reads):
// two step bodies share the sums badly, 20 spilled registers.
#include "dsa_sel.h"

#define SELKV_AHEAD 3                                    // operands read ahead
#define SELKV_NW 12
#define SELKV_KEYS 16                                    // of a wave
#define SELKV_ROWS 128                                   // rows of a block
// LDS: two blocks of q and dO | row data of two blocks (-lse / scale | -delta) and, as loaded, of the next | of each wave two lists and the
// selection words of two blocks
constexpr int SELKV_DATA_B = SELKV_ROWS * 8, SELKV_DATA = 4 * SelBlock<SELKV_ROWS>::BYTES, SELKV_RAW = SELKV_DATA + 2 * SELKV_DATA_B,
              SELKV_WAVES = SELKV_RAW + SELKV_DATA_B;
template <int GSHIFT> constexpr int selkv_list_bytes() { return (SELKV_ROWS >> GSHIFT) * 8; }
template <int GSHIFT> constexpr int selkv_wave_bytes() { return 2 * selkv_list_bytes<GSHIFT>() + 2 * 128; }
template <int GSHIFT> constexpr size_t selkv_lds_bytes() { return SELKV_WAVES + SELKV_NW * (size_t)selkv_wave_bytes<GSHIFT>(); }

template <int GSHIFT>
__global__ __launch_bounds__(SELKV_NW * 64, 1) void dsa_tile_selkv_kernel(
    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v,
    const float *__restrict__ lse, const float *__restrict__ delta, const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu,
    int N, int T, int Hq, int Hkv, float scale, float logit_scale, int split_len, bf16_t *__restrict__ dk, bf16_t *__restrict__ dv) {
    typedef SelBlock<SELKV_ROWS> BL;
    constexpr int D = BL::D, KS = D / 32, DT = D / 16, Gp = 1 << GSHIFT, QB = SELKV_ROWS >> GSHIFT, NC = 16 >> GSHIFT, WAVE_B = selkv_wave_bytes<GSHIFT>();
    constexpr int LIST_B = selkv_list_bytes<GSHIFT>();
    static_assert(GSHIFT >= 2 && GSHIFT <= 4, "four neighbouring rows of a lane are one query's");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, j = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = Hq / Hkv, kvh = blockIdx.x % Hkv;
    int s0, L, blk;
    if (!locate_block(cu, N, blockIdx.x / Hkv, SELKV_NW * SELKV_KEYS, false, s0, L, blk)) return;     // (a segment's first keys, which all its queries see, first)
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = __builtin_amdgcn_readfirstlane(L);
    L = min(L, ldw * 32);                               // a bitmap row has ldw words whatever the caller's max_seqlen
    const int c0 = __builtin_amdgcn_readfirstlane(blk) * (SELKV_NW * SELKV_KEYS), kc = c0 + wv * SELKV_KEYS;    // the workgroup's and the wave's first key
    if (L < split_len || c0 >= L) return;               // short segments belong to the tile kernel
    const int last = (L - 1) / QB, nblocks = last - c0 / QB + 1;           // block b of the walk: queries (last - b) QB ..

    // ---- requests ----
    const int tok_b = Hq * D * 2;                       // bytes from one query to the next
    const uint32_t lds0 = lds_address(dyn_lds);
    const int64_t first = ((int64_t)(s0 + last * QB) * Hq + kvh * G) * D;
    const unsigned char *qptr = reinterpret_cast<const unsigned char *>(q + first), *dptr = reinterpret_cast<const unsigned char *>(dout + first);
    const int lrow = BL::load_row(wv, lane), lhead = lrow & (Gp - 1);
    const int voff[1] = {lhead < G ? (lrow >> GSHIFT) * tok_b + lhead * BL::ROW_B + BL::load_chunk(wv, lane) * 16 : (int)0x80000000};
    auto request = [&](int b) __attribute__((always_inline)) {            // q and dO of block b, in block order; rows that do not exist read as zero
        constexpr int STEP = SEL_LOADERS * BL::LOAD_ROWS >> GSHIFT;       // queries from one of the wave's loads to the next
        const uint32_t at = lds0 + (b & 1) * 2 * BL::BYTES + wv * 1024;
        if (wv >= SEL_LOADERS) return;
#pragma unroll
        for (int i = 0; i < BL::LPW; ++i) {
            const int n = min(L - (last - b) * QB - i * STEP, QB);
            const uint32_t bytes = n > 0 ? (n - 1) * tok_b + G * BL::ROW_B : 0;
            buffer_load_lds16_n<1, 0, 0, 0>(scalar_buffer_rsrc(qptr, bytes), voff, at + i * SEL_LOADERS * 1024);
            buffer_load_lds16_n<1, 0, 0, 0>(scalar_buffer_rsrc(dptr, bytes), voff, at + i * SEL_LOADERS * 1024 + BL::BYTES);
            const int64_t by = i + 1 < BL::LPW ? (int64_t)STEP * tok_b : (int64_t)((BL::LPW - 1) * -STEP - QB) * tok_b;
            qptr += by;
            dptr += by;
            asm volatile("" : "+s"(qptr), "+s"(dptr));
        }
    };
    // (what a lane loads beside the blocks is placed anew for each: the addresses would cost the loop its registers)
    auto opaque_lane = [&]() __attribute__((always_inline)) {
        int x = lane;
        asm volatile("" : "+v"(x));
        return x;
    };
    // row data: 64 rows a wave, of waves 0 and 1 the log-sum-exps, of 2 and 3 delta; heads that pad a group get values that make P vanish
    auto request_rowdata = [&](int b) __attribute__((always_inline)) {
        const int ln = opaque_lane(), row = (wv & 1) * (SELKV_ROWS / 2) + ln;
        if (wv < 4 && ln < SELKV_ROWS / 2)
            global_load_lds4((wv < 2 ? lse : delta) + (int64_t)(kvh * G + min(row & (Gp - 1), G - 1)) * T + s0 + min((last - b) * QB + (row >> GSHIFT), L - 1),
                             lds0 + SELKV_RAW + wv * (SELKV_ROWS * 2));
    };
    auto put_rowdata = [&](int b) __attribute__((always_inline)) {
        const int ln = opaque_lane(), row = (wv & 1) * (SELKV_ROWS / 2) + ln;
        if (wv < 4 && ln < SELKV_ROWS / 2) {
            const float x = *reinterpret_cast<const float *>(dyn_lds + SELKV_RAW + wv * (SELKV_ROWS * 2) + ln * 4);
            *reinterpret_cast<float *>(dyn_lds + SELKV_DATA + (b & 1) * SELKV_DATA_B + wv * (SELKV_ROWS * 2) + ln * 4) =
                (row & (Gp - 1)) >= G ? (wv < 2 ? (logit_scale < 0.f ? 1e30f : -1e30f) : 0.f) : x * (wv < 2 ? -1.f / logit_scale : -1.f);
        }
    };
    // Selection words: lane l < QB stands for query NC (l % (QB / NC)) + l / (QB / NC) of a block, so that a list goes by the classes of its rows
    static_assert(QB % NC == 0 && QB <= 32, "");
    auto query_of = [&](int l) __attribute__((always_inline)) { return NC * (l % (QB / NC)) + l / (QB / NC); };
    const int wave_at = SELKV_WAVES + wv * WAVE_B;
    auto request_words = [&](int b) __attribute__((always_inline)) {
        const int ln = opaque_lane(), t = (last - b) * QB + query_of(ln);
        if (ln < QB) {
            const bool there = t >= 0 && t < L && (kc >> 5) < ldw;
            buffer_load_lds4(make_buffer_rsrc(bitmap + (int64_t)(s0 + max((last - b) * QB, 0)) * ldw + (kc >> 5), (int64_t)QB * ldw * 4),
                             there ? (t - max((last - b) * QB, 0)) * ldw * 4 : (int)0x80000000, lds0 + wave_at + 2 * LIST_B + (b & 1) * 128);
        }
    };
    request(0);
    request_rowdata(0);
    request_words(0);
    request_words(1);

    // the wave's keys: a lane holds quarter g of every 32 elements of key j
    bf16x8 kB[KS], vB[KS];
    {
        const int64_t off = ((int64_t)(s0 + min(kc + j, L - 1)) * Hkv + kvh) * D + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            kB[ks] = load_bf16x8(k + off + 32 * ks);
            vB[ks] = load_bf16x8(v + off + 32 * ks);
        }
    }
    f32x4 dkacc[DT], dvacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) dkacc[dt] = dvacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float scale_log2 = logit_scale * LOG2E_F;

    // A list's entry: the query's bits of the wave's keys, where its first row lies in the block (BL::entry), in the upper half where its row data does
    auto build = [&](int b) __attribute__((always_inline)) {              // the list of block b: its tiles
        u32x2 *const list = reinterpret_cast<u32x2 *>(dyn_lds + wave_at + (b & 1) * LIST_B);
        const int ln = opaque_lane(), row = query_of(ln) * Gp;
        const uint32_t w = ln < QB ? *reinterpret_cast<const uint32_t *>(dyn_lds + wave_at + 2 * LIST_B + (b & 1) * 128 + ln * 4) >> (kc & 16) & 0xffffu : 0u;
        const uint32_t e = (uint32_t)BL::entry(row) | (uint32_t)(row * 4) << 16;
        const uint32_t some = (uint32_t)__builtin_amdgcn_ballot_w64(w != 0u);
        const int tiles = (__builtin_popcount(some) + NC - 1) / NC;       // of sixteen rows, two to a step
        // The k-th query of class c goes to place c of tile k, where the rows are of different classes; those of a class that has more than there
        // are tiles go to the places left over
        const int c = ln >> 3, k = (int)__builtin_amdgcn_mbcnt_lo(some & 0xffu << (8 * c & 31), 0);
        int at = k < tiles ? k * NC + c : -1;
        const uint64_t over = __builtin_amdgcn_ballot_w64(w != 0u && at < 0);
        if (over) {
            const int o = (int)__builtin_amdgcn_mbcnt_lo((uint32_t)over, 0);
            int cc = 0, kk = 0, left = 0;                // the o-th place left over: class and number
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int n = __builtin_popcount(some >> 8 * i & 0xffu);
                if (o >= left) {
                    cc = i;
                    kk = n + o - left;
                }
                left += max(tiles - n, 0);
            }
            if (at < 0) at = kk * NC + cc;
        }
        if (ln < QB) list[ln] = u32x2{0u, (uint32_t)BL::entry((ln & (NC - 1)) * Gp)};       // (nobody's: a row of the class that its place would have)
        if (w) list[at] = u32x2{w, e};
        return tiles;
    };
    // of the head of the lane's row (row-wise, transposed) and its chunk
    const int er_x = BL::entry(j & (Gp - 1)) ^ g << 4, et_x = BL::entry((4 * g + (j >> 2)) & (Gp - 1)) ^ (j >> 1 & 1) << 4 ^ (j & 1) << 3;
    const uint32_t list0 = lds0 + wave_at;
    wait_vmcnt<0>();
    put_rowdata(0);
    int tiles = build(0);
    __syncthreads();

    // Entries of the step ahead: of the lane's rows (row-wise), of rows 16 m + 4 g ..
    uint32_t row_entry[2];
    u32x2 entry[2];
    auto read_entries = [&](uint32_t list) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            row_entry[m] = lds_read<uint16_t>(list + 4 + ((16 * m + j) >> GSHIFT) * 8);
            entry[m] = lds_read<u32x2>(list + ((16 * m + 4 * g) >> GSHIFT) * 8);
        }
    };
    read_entries(list0);

    for (int b = 0; b < nblocks; ++b) {
        const int next = build(b + 1);               // (behind the last block: an empty list or an old one, never used)
        if (b + 1 < nblocks) {
            request(b + 1);
            request_rowdata(b + 1);
        }
        request_words(b + 2);
        const int at = (b & 1) * 2 * BL::BYTES;
        const uint32_t rd0 = lds0 + SELKV_DATA + (b & 1) * SELKV_DATA_B;
        for (int tile = 0; tile < tiles; tile += 2) {
            int er[2], et[2];
            uint32_t mine[2], data[2];                   // rows 16 m + 4 g ..: one query's; its bits, where its row data lies
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                er[m] = ((int)row_entry[m] ^ er_x ^ BL::entry(16 * m & (Gp - 1))) + at;
                mine[m] = entry[m][0];
                et[m] = ((int)(entry[m][1] & 0xffffu) ^ et_x ^ BL::entry(16 * m & (Gp - 1))) + at;
                data[m] = rd0 + (entry[m][1] >> 16) + ((16 * m + 4 * g) & (Gp - 1)) * 4;
            }
            auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
            // operands in the order of their MFMAs: q and dO rows (tiles of 16 rows in turn), dO and q transposed
            constexpr int TR = 4 * KS;
            auto fetch = [&](int i) __attribute__((always_inline)) {
                return lds_read<bf16x8>(er[i % 2] + i / 2 % KS * BL::COLUMN_B + i / 2 / KS * BL::BYTES);
            };
            auto fetch_tr = [&](int i) __attribute__((always_inline)) {
                const int dt = i % DT, by = (dt >> 1) * BL::COLUMN_B + (i < DT ? BL::BYTES : 0);
                return tr_pair((lds_u8 *)((et[0] ^ (dt & 1) << 5) + by), (lds_u8 *)((et[1] ^ (dt & 1) << 5) + by));
            };
            auto words = [](const uint32_t (&w)[4]) __attribute__((always_inline)) { return __builtin_bit_cast(bf16x8, u32x4{w[0], w[1], w[2], w[3]}); };
            bf16x8 op[SELKV_AHEAD], tr[SELKV_AHEAD];
#pragma unroll
            for (int m = 0; m < SELKV_AHEAD; ++m) op[m] = fetch(m);
            f32x4 s[2], dp[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                s[m] = lds_read<f32x4>(data[m]);
                dp[m] = lds_read<f32x4>(data[m] + SELKV_ROWS * 4);
            }
            fence();
            auto refill = [&](int i) __attribute__((always_inline)) {
                if (i + SELKV_AHEAD < TR) op[i % SELKV_AHEAD] = fetch(i + SELKV_AHEAD);
                else tr[i + SELKV_AHEAD - TR] = fetch_tr(i + SELKV_AHEAD - TR);
            };
            auto refill_tr = [&](int i) __attribute__((always_inline)) {
                if (i + SELKV_AHEAD < 2 * DT) tr[i % SELKV_AHEAD] = fetch_tr(i + SELKV_AHEAD);
            };
#pragma unroll
            for (int i = 0; i < 2 * KS; ++i) {
                s[i % 2] = mfma16(op[i % SELKV_AHEAD], kB[i / 2], s[i % 2]);
                refill(i);
                fence();
            }
            float pm = 0.f;
            uint32_t p[4], ds[4];
#pragma unroll
            for (int i = 0; i < 2 * KS; ++i) {          // P behind the MFMAs of dP
                dp[i % 2] = mfma16(op[(2 * KS + i) % SELKV_AHEAD], vB[i / 2], dp[i % 2]);
                refill(2 * KS + i);
                const int m = i >> 2, e = i & 3;
                s[m][e] = fast_exp2(keep_or_neginf(s[m][e] * scale_log2, (uint32_t)__builtin_amdgcn_sbfe((int)mine[m], j, 1)));
                pm = fmaxf(pm, s[m][e]);
                fence();
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = pack2bf(s[i >> 1][2 * (i & 1)], s[i >> 1][2 * (i & 1) + 1]);
#pragma unroll
            for (int i = 0; i < 4; ++i) ds[i] = pack2bf(s[i >> 1][2 * (i & 1)] * dp[i >> 1][2 * (i & 1)], s[i >> 1][2 * (i & 1) + 1] * dp[i >> 1][2 * (i & 1) + 1]);
            // dV also takes what bf16 rounds off the larger probabilities, as in the tile kernel: the same MFMAs once more (a loop, for behind
            // a branch around them the sums would have to come together again, and spill).  From 2^-7 on, half of the tile kernel's: a step holds
            // fewer probabilities than its blocks, one of which decides (error of dV against 64 bits, K = 128, 3500 tokens: tile kernel 2.08e-3,
            // here from 2^-6 on 2.19e-3, from 2^-7 on 1.66e-3, which is the rounding of the result).
            for (bool more = __builtin_amdgcn_ballot_w64(pm >= 0x1p-7f) != 0ull;; more = false) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    dvacc[dt] = mfma16(tr[dt % SELKV_AHEAD], words(p), dvacc[dt]);
                    refill_tr(dt);
                    fence();
                }
                if (!more) break;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    p[i] = pack2bf(s[i >> 1][2 * (i & 1)] - __uint_as_float(p[i] << 16), s[i >> 1][2 * (i & 1) + 1] - __uint_as_float(p[i] & 0xffff0000u));
#pragma unroll
                for (int m = 0; m < SELKV_AHEAD; ++m) tr[m] = fetch_tr(m);
            }
            read_entries(list0 + (tile + 2 < tiles ? (b & 1) * LIST_B + (tile + 2) * NC * 8 : (~b & 1) * LIST_B));
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                dkacc[dt] = mfma16(tr[(DT + dt) % SELKV_AHEAD], words(ds), dkacc[dt]);
                refill_tr(DT + dt);
                fence();
            }
        }
        if (tiles == 0) read_entries(list0 + (~b & 1) * LIST_B);
        wait_vmcnt<0>();
        put_rowdata(b + 1);
        tiles = next;
        __syncthreads();
    }
    int j_ = j;                                          // (where the row lies is formed again: the loop needs its registers)
    asm volatile("" : "+v"(j_));
    if (kc + j_ < L) {                                   // a lane holds elements 16 dt + 4 g .. of key j
        const int64_t off = ((int64_t)(s0 + kc + j_) * Hkv + kvh) * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const f32x4 a = dkacc[dt] * scale, c = dvacc[dt];
            *reinterpret_cast<u32x2 *>(dk + off + 16 * dt) = u32x2{pack2bf(a[0], a[1]), pack2bf(a[2], a[3])};
            *reinterpret_cast<u32x2 *>(dv + off + 16 * dt) = u32x2{pack2bf(c[0], c[1]), pack2bf(c[2], c[3])};
        }
    }
}

template <int GSHIFT>
static hipError_t launch_selkv(hipStream_t stream, const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                               const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int split_len, void *dk, void *dv) {
    const auto kernel = &dsa_tile_selkv_kernel<GSHIFT>;
    constexpr size_t lds = selkv_lds_bytes<GSHIFT>();
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(((int64_t)T / (SELKV_NW * SELKV_KEYS) + N) * Hkv));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * SELKV_NW), lds, stream, (const bf16_t *)dout, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, lse, delta,
                       bitmap, ldw, cu, N, T, Hq, Hkv, scale, logit_scale(scale), split_len, (bf16_t *)dk, (bf16_t *)dv);
    return hipGetLastError();
}
// the keys of segments of split_len tokens and more; head_dim 128, three to sixteen heads per kv head, all operands on 16-byte boundaries
extern "C" hipError_t dsa_launch_selkv(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                                       const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int split_len,
                                       void *dk, void *dv, hipStream_t stream) {
    const int gs = group_shift(Hq, Hkv);
    const auto launch = gs == 2 ? &launch_selkv<2> : gs == 3 ? &launch_selkv<3> : &launch_selkv<4>;
    return launch(stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, split_len, dk, dv);
}
