// Attention mass over 32x32 MFMA tiles with the selection applied as a bitmap mask, and the launch of dK / dV (the forward:
// dsa_tile_fwd.hip, dQ: dsa_tile_dq.hip, dK / dV: dsa_tile_dkv.hip, the indexer backward: dsa_tile_idx.hip).  They do the same
// arithmetic as the gather kernels but visit every (query block, key
// tile) pair of the causal triangle, so they win wherever the selection is dense: one selected pair
// costs the gather kernels 2*D*e bytes of L2 traffic per kv head, a causal pair costs these kernels
// 4*G*D flop on the matrix cores - on MI355X the tile walk is cheaper down to a few percent density.
//
// Common scheme (wave64, v_mfma_f32_32x32x16_bf16):
//   rows of the problem are (query, head-in-group) pairs, `Gp` (power of two >= G) rows per query;
//   the mask depends on the query only.  Operands that move (K,V tiles for the query-stationary
//   kernels, q,dO blocks for the key-stationary one) are staged once per workgroup in LDS, row-major
//   with an XOR swizzle of the 16-byte chunks, and read either row-wise (16-byte reads, contraction
//   over D) or transposed with ds_read_b64_tr_b16 (contraction over rows/keys) - both conflict-free.
//   The second GEMM of each chain takes its B operand straight from the C layout of the first
//   (the contraction order over the 32 keys/rows of a tile is permuted identically on both operands).
#include "dsa_tile.h"

// ==================================================================================================
// attention mass: the indexer's training target.  Same walk and S^T = K Q^T as the forward, with the
// saved log-sum-exp instead of the online softmax and no V: P = exp(S*scale - lse) on the selected
// keys, summed over the heads of a query that share the kv head (lanes of one query are adjacent:
// DPP adds), and written to the slot the key has in the query's ascending selection list
// (slot = selected keys of earlier tiles + selected keys below it in the tile's word).
// ==================================================================================================
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
// sum over the aligned group of 2^GSHIFT adjacent lanes, on every lane of the group
template <int GSHIFT>
__device__ __forceinline__ float group_sum(float x) {
    if (GSHIFT >= 1) x += dpp_f<0xB1>(x);               // quad_perm [1,0,3,2]
    if (GSHIFT >= 2) x += dpp_f<0x4E>(x);               // quad_perm [2,3,0,1]
    if (GSHIFT >= 3) x += dpp_f<0x141>(x);              // row_half_mirror: the other quad's total
    if (GSHIFT >= 4) x += dpp_f<0x140>(x);              // row_mirror: the other half row's total
    return x;
}
// The heads of a query meet in one workgroup: a wave's 32 rows are (query, head of one kv group) pairs as in the
// forward, and the workgroup takes its HPG kv heads *inside* each key tile - all their K tiles are staged together,
// all their q rows stay in registers - and adds their probabilities up in registers.  With two or more kv heads the
// workgroup has two sets of four waves on the same queries, each set taking half of the kv heads (two waves per
// SIMD: one's exponentials run beside the other's matrix work; a wave holds up to 128 registers of q rows); the
// second set hands its sums to the first through LDS once per tile.  A slot of the result is therefore written
// once, by one lane, with the finished sum: no table per kv head, nothing read back.  Only a batch with more kv
// heads than a workgroup holds is cut into groups with one table each.
// A slot depends on its own tile alone, so a walk can be cut anywhere: launches that leave the chip idle (one workgroup
// per CU: 64 queries of a 2B stack's 8192 tokens are 128 workgroups for 256 CUs) run pieces of `chunk` tiles as workgroups
// of their own, each counting the selected keys in front of its piece first (there 189 -> 89 us).
// Each wave runs two heads at once: the MFMAs of S for the next (tile, head) with the exponentials of this one behind them.  Key
// tiles of all the heads go from memory straight into LDS, two slots: at the last head of tile t - every wave has read tile t by
// then - the wave waits for tile t+1, meets the one barrier per tile and requests tile t+2.  The second set leaves its sums, added
// up over the heads of a query first, in LDS in front of that barrier and the first set finishes tile t behind the next one.
// What bounds it: the vector pipe, 16 exponentials of 16 clocks and 32 other instructions per head, tile and wave (384 clocks
// against 256 of MFMA).  32 768 tokens, 32 heads of 128: 1110 -> 875 us (operands staged through registers, S and exponentials
// one after the other, two barriers per tile before).
template <int D> constexpr int mass_heads_max() { return 1024 / D; }      // 16 / 8 / 4 kv heads at head_dim 64 / 128 / 256
template <int HPG> constexpr int mass_sets() { return HPG >= 2 ? 2 : 1; }
template <int D, int GSHIFT, int HPG> constexpr size_t mass_lds_bytes() {
    return 2 * (size_t)HPG * DirectTile<D>::BYTES + 4 * 4 * 256 + (mass_sets<HPG>() == 2 ? 2 * 4 * 64 * (16 >> GSHIFT) * sizeof(float) : 0);
}
template <int D, int GSHIFT, int HPG>
__global__ __launch_bounds__(256 * mass_sets<HPG>(), 1) void dsa_tile_mass_kernel(
    const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const float *__restrict__ lse,
    const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv,
    float scale_log2, int K, int ngroups, int chunk, float final_mul, float *__restrict__ table) {
    typedef DirectTile<D> TL;
    constexpr int NS = mass_sets<HPG>(), HPW = HPG / NS;       // wave sets; kv heads per wave
    constexpr int KS = D / 16, NT = 256 * NS, Gp = 1 << GSHIFT, QBW = (4 * 32) >> GSHIFT, U = 16 / Gp;
    constexpr int LPW = HPG * TL::LOADS / (4 * NS);            // wave loads per wave and tile
    static_assert(HPG * TL::LOADS % (4 * NS) == 0 && LPW >= 1 && (LPW % 2 == 0 || TL::SOURCES == 1), "every wave loads the same number of pieces");
    extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_lds[];   // [2][HPG] K tiles | words [quarter][tile % 4] | sums of the second set
    constexpr int SLOT = HPG * TL::BYTES;
    unsigned char *const words = dyn_lds + 2 * SLOT;
    float *const xbuf = reinterpret_cast<float *>(words + 4 * 4 * 256);

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = wv & 3, set = wv >> 2;                // query quarter of the block; wave set
    const int G = Hq / Hkv;
    const int grp = blockIdx.x % ngroups, kvh0 = grp * HPG;
    int s0, L, blk;
    // (heaviest block first over the whole batch: 1.21 against 1.37 ms for the segment-by-segment order at 32 768 tokens)
    if (!locate_block_heaviest_first(cu, N, blockIdx.x / ngroups, QBW, s0, L, blk)) return;
    s0 = __builtin_amdgcn_readfirstlane(s0);
    L = min(__builtin_amdgcn_readfirstlane(L), ldw * 32);      // a bitmap row has ldw words whatever the caller's max_seqlen
    const int qc0 = __builtin_amdgcn_readfirstlane(blk) * QBW;
    if (qc0 >= L) return;

    const int r = wq * 32 + j;
    const int qcol = qc0 + (r >> GSHIFT), head = r & (Gp - 1);
    const bool row_ok = qcol < L && head < G;
    const int t = s0 + min(qcol, L - 1);
    // this workgroup's piece of the walk: tiles [it0, ntiles)
    const int it0 = (int)blockIdx.y * chunk, ntiles = min((min(qc0 + QBW - 1, L - 1) / 32 + 1), it0 + chunk);
    if (it0 >= ntiles) return;

    // ---- requests ----
    const uint32_t lds0 = lds_address(dyn_lds);
    const int tok_b = Hkv * D * 2;                       // bytes from one key row to the next
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k + (int64_t)(s0 + it0 * 32) * Hkv * D);
    int koff[TL::SOURCES];
#pragma unroll
    for (int i = 0; i < TL::SOURCES; ++i) koff[i] = TL::source(i, lane, tok_b, D / 8);
    const int wq0 = min(qc0 + ((wq * 32) >> GSHIFT), L - 1);   // the wave's first query
    const unsigned char *wptr = reinterpret_cast<const unsigned char *>(bitmap + (int64_t)(s0 + wq0) * ldw + it0);
    const int wvoff = (t - s0 - wq0) * ldw * 4;
    // the tiles of all heads (kv heads past the last one, in a short last group, repeat it and count for nothing: lse = +inf
    // below; rows past the segment read as zero) and the selection words; called for tile it0, it0+1, ... in turn
    auto request = [&](int tile) __attribute__((always_inline)) {
        const buffer_rsrc keys = make_buffer_rsrc(kptr, (int64_t)max(min(L - tile * 32, 32), 0) * tok_b);
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            const int g = wv * LPW + i, hh = g / TL::LOADS, p = g % TL::LOADS;
            buffer_load_lds16(keys, koff[i % TL::SOURCES] + (p / TL::SOURCES * TL::SOURCES) * TL::LOAD_ROWS * tok_b + min(kvh0 + hh, Hkv - 1) * D * 2,
                              lds0 + (tile & 1) * SLOT + hh * TL::BYTES + TL::load_lds(p));
        }
        kptr += (int64_t)32 * tok_b;
        if (set == 0) {
            buffer_load_lds4(make_buffer_rsrc(wptr, tile < ntiles ? 32 * (int64_t)ldw * 4 : 0), wvoff, lds0 + 2 * SLOT + wq * 1024 + (tile & 3) * 256);
            wptr += 4;
        }
    };
    request(it0);
    request(it0 + 1);
    const uint32_t *wrow = bitmap + (int64_t)t * ldw;
    float *prow = table + ((int64_t)grp * T + t) * K;
    if (ngroups == 1 && it0 == 0) {
        // the table is the result itself: slots past a row's selection (rows shorter than K keys) are zero
        for (int qq = 0; qq < QBW && qc0 + qq < L; ++qq) {
            float *zr = table + (int64_t)(s0 + qc0 + qq) * K;
            for (int jj = qc0 + qq + 1 + tid; jj < K; jj += NT) zr[jj] = 0.f;
        }
    }
    bf16x8 qB[HPW][KS];
    float lse2[HPW];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int kv_rel = set * HPW + hh;
        const int kvh = min(kvh0 + kv_rel, Hkv - 1);
        const int hq = kvh * G + min(head, G - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            qB[hh][ks] = row_ok ? load_bf16x8(q + ((int64_t)t * Hq + hq) * D + 16 * ks + 8 * h) : zero_bf16x8();
        // padding rows (head >= G, query past the segment, kv head past the last) get lse = +inf: their P is
        // exp2(-inf) = 0 in the sums.  Keys that are not selected need no masking: their sums are never stored.
        const float lse_row = lse[(int64_t)hq * T + t];
        lse2[hh] = (row_ok && kvh0 + kv_rel < Hkv) ? lse_row * LOG2E_F : INFINITY;
    }
    int seen = 0;                                        // selected keys of this row in the tiles before this one
    for (int w = 0; w < it0; w += 8)                     // (it0 is a multiple of 8)
#pragma unroll
        for (int u = 0; u < 8; ++u) seen += __popc(wrow[w + u]);
    TL tl;
    tl.init(lane);
    wait_vmcnt<0>();
    barrier_only();

    int ka[4];                                           // operand addresses in the tile of the next S
    bf16x8 kr[4];
    auto read_k = [&](int ks) __attribute__((always_inline)) {
        return *reinterpret_cast<const bf16x8 *>(dyn_lds + ka[TL::row_q(ks)] + TL::row_imm(ks));
    };
    auto first_reads = [&](int tile, int hh) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ka[i] = tl.rowq[i] + (tile & 1) * SLOT + (set * HPW + hh) * TL::BYTES;
#pragma unroll
        for (int i = 0; i < 4; ++i) kr[i] = read_k(i);
    };
    float val[U];                                        // the elements u * Gp + head of the last tile's sums
    // tile's sums finished and stored: the lanes of a query share the stores, lane `head` has the elements vi = u*Gp + head
    auto finish = [&](int tile) __attribute__((always_inline)) {
        if (set != 0) return;
        const uint32_t wl = *reinterpret_cast<const uint32_t *>(words + wq * 1024 + (tile & 3) * 256 + lane * 4);
        const uint32_t word = qcol < L ? wl : 0u;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float x = val[u];
            if (NS == 2) x += xbuf[(((tile & 1) * 4 + wq) * U + u) * 64 + lane];
            const int vi = u * Gp + head;
            const int bit = 8 * (vi >> 2) + (vi & 3) + 4 * h;    // the key's column in the tile
            if ((word >> bit) & 1u) prow[seen + __popc(word & ((1u << bit) - 1u))] = x * final_mul;
        }
        seen += __popc(word);
    };
    float p[16];
    // exponentials of (this tile, head hh) from `s` behind the MFMAs of the next S into `sn` (NEXT: with `qn`)
    auto stage = [&](auto next_, int hh, const f32x16 &s, const bf16x8 (&qn)[KS], f32x16 &sn) __attribute__((always_inline)) {
        constexpr bool NEXT = decltype(next_)::value;
        const float neg = -lse2[hh];
        f32x16 snew;
        auto behind = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int vi = 16 * i / KS; vi < 16 * (i + 1) / KS; ++vi) {
                const float e = fast_exp2(fmaf(s[vi], scale_log2, neg));
                p[vi] = hh == 0 ? e : p[vi] + e;
                asm volatile("" : "+v"(p[vi]));
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            if (NEXT) {
                snew = mfma32(kr[i & 3], qn[i], i == 0 ? zero16() : snew);
                if (i + 4 < KS) kr[i & 3] = read_k(i + 4);
            }
            behind(i);
        }
        if (NEXT) sn = snew;
    };
    const std::true_type yes;
    const std::false_type no;
    f32x16 sA, sB;
    // one tile: S of its first head in sA; leaves S of the next tile's first head there (LAST: there is none)
    auto tile_step = [&](auto last_, int it) __attribute__((always_inline)) {
        constexpr bool LAST = decltype(last_)::value;
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
            f32x16 &s = hh & 1 ? sB : sA, &sn = hh & 1 ? sA : sB;
            if (hh + 1 < HPW) {
                first_reads(it, hh + 1);
                stage(yes, hh, s, qB[hh + 1 < HPW ? hh + 1 : 0], sn);
            } else {
                // every wave has read this tile; the sums of the one before are in place
                wait_vmcnt<0>();
                asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
                barrier_only();
                if (it > it0) finish(it - 1);
                if (!LAST) {
                    request(it + 2);
                    first_reads(it + 1, 0);
                    stage(yes, hh, s, qB[0], sn);
                    if (hh % 2 == 0) sA = sB;            // (an odd number of heads)
                } else {
                    stage(no, hh, s, qB[0], sn);
                }
            }
        }
#pragma unroll
        for (int vi = 0; vi < 16; ++vi) p[vi] = group_sum<GSHIFT>(p[vi]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            val[u] = p[u * Gp];
#pragma unroll
            for (int g = 1; g < Gp; ++g) val[u] = head == g ? p[u * Gp + g] : val[u];
            if (NS == 2 && set == 1) xbuf[(((it & 1) * 4 + wq) * U + u) * 64 + lane] = val[u];
        }
    };
    first_reads(it0, 0);
    sA = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        sA = mfma32(kr[ks & 3], qB[0][ks], sA);
        if (ks + 4 < KS) kr[ks & 3] = read_k(ks + 4);
    }
    for (int it = it0; it + 1 < ntiles; ++it) tile_step(no, it);
    tile_step(yes, ntiles - 1);
    wait_vmcnt<0>();                                    // no load is left on its way into LDS when the workgroup ends
    __syncthreads();
    finish(ntiles - 1);
}

// mass[t,j] = inv_hq * sum over the tables of partial[g][t][j] for j < n[t], else 0.  One workgroup per query row
// and blockIdx.y-th part of it, four columns per thread (16-byte accesses when K is a multiple of four).
__global__ __launch_bounds__(256) void dsa_mass_reduce_kernel(const float *__restrict__ partial,
                                                               const int32_t *__restrict__ nsel, int T, int K, int Hkv,
                                                               float inv_hq, float *__restrict__ mass) {
    const int t = blockIdx.x, nt = nsel[t];
    const int64_t row = (int64_t)t * K, plane = (int64_t)T * K;
    if ((K & 3) == 0) {
        for (int j4 = blockIdx.y * 256 + threadIdx.x; j4 < (K >> 2); j4 += gridDim.y * 256) {
            float4 acc = {0.f, 0.f, 0.f, 0.f};
            if (4 * j4 < nt)
                for (int kvh = 0; kvh < Hkv; ++kvh) {
                    const float4 x = *reinterpret_cast<const float4 *>(partial + kvh * plane + row + 4 * j4);
                    acc.x += x.x; acc.y += x.y; acc.z += x.z; acc.w += x.w;
                }
            // slots at and beyond n[t] were never written
            acc.x = 4 * j4 < nt ? acc.x * inv_hq : 0.f;
            acc.y = 4 * j4 + 1 < nt ? acc.y * inv_hq : 0.f;
            acc.z = 4 * j4 + 2 < nt ? acc.z * inv_hq : 0.f;
            acc.w = 4 * j4 + 3 < nt ? acc.w * inv_hq : 0.f;
            *reinterpret_cast<float4 *>(mass + row + 4 * j4) = acc;
        }
    } else {
        for (int jj = blockIdx.y * 256 + threadIdx.x; jj < K; jj += gridDim.y * 256) {
            float acc = 0.f;
            if (jj < nt)
                for (int kvh = 0; kvh < Hkv; ++kvh) acc += partial[kvh * plane + row + jj];
            mass[row + jj] = acc * inv_hq;
        }
    }
}

// ==================================================================================================
// Launch order of the key-stationary workgroups.  A key tile's walk is as long as the part of its segment
// behind it, and the hardware starts workgroups in grid order: handed out segment by segment, the long
// walks of a late long segment start late and the launch ends on them.  This kernel (one workgroup) lists
// the 128-key tiles of all segments longest walk first -
//   mode 0: by the number of tiles behind them, across segments (32 768 tokens in eight segments, segment by segment in order
//           of length: 2380 instead of 2297 us - CUs busy 0.83 instead of 0.91 of the launch; octave by octave of the walk's
//           length, segments together within one: level),
//   mode 1: the segments by length, each one's tiles together, without a causal mask: walks are equally long within a
//           segment, and workgroups that run side by side walk the same q / dO rows and share them in L2 (4000 patches,
//           forward and backward, 170 -> 154 us),
//   mode 2: long walks cut into equal pieces of at most `pb` steps (a step = `qb` queries), listed by length, for launches of up
//           to three rounds of workgroups: a launch then ends with its longest walk, however few the workgroups.  A tile in
//           pieces leaves one fp32 partial dK / dV per piece, added in piece order by dsa_dkv_pieces_reduce_kernel.  pb (see
//           below) depends on cu_seqlens and the parameters of the launch only.
// Table:
//   order[0] = number of entries (or -1: too many segments or tiles for the table, use the plain order),
//   order[1] = queries of a piece, pb steps of qb (0: no walk is cut), order[2] = number of tiles that are cut,
//   order[4 + 4 s .. 7 + 4 s] = first row and length of the segment, tile | piece << 13, first partial slot of the tile (-1: not
//   cut) of entry s,
//   behind the `cap` entries: the entry of the first piece of every cut tile.
// The pieces of a tile are counted from the walk's length bound 128 r / qb of its rank r (tiles behind it,
// itself included); a tile whose own walk is shorter leaves its last pieces empty (the kernels and the
// reduction count the pieces from the walk itself).
// The order changes the schedule only; every tile is still reduced in a fixed order.
// ==================================================================================================
#define DSA_ORDER_MAX_TILES 8192                         // tiles of the longest segment
#define DSA_ORDER_EXTRA 4096                             // entries beyond one per tile (pieces)
#define DSA_ORDER_SPLIT_MAX_TILES 1024                   // mode 2: one thread per rank
static_assert(DSA_ORDER_MAX_TILES + 1 >= 2 * DSA_ORDER_MAX_SEGS, "the rank tables of the by-segment order share cnt[]");
__device__ __forceinline__ void order_entry(int32_t *order, const int32_t *cu, int slot, int seg, int tile, int piece, int mslot) {
    const int s0 = cu[seg];
    *reinterpret_cast<int4 *>(order + 4 + 4 * slot) = make_int4(s0, cu[seg + 1] - s0, tile | piece << 13, mslot);
}
struct TileOrder { int cap, mode, qb, wg_per_tile, item_cap, slot_cap, slots, share8, extra; };
__device__ __forceinline__ void tile_order(const int32_t *__restrict__ cu, int N, const TileOrder &o_, int32_t *__restrict__ order) {
    const int cap = o_.cap, mode = o_.mode, qb = o_.qb, wg_per_tile = o_.wg_per_tile, item_cap = o_.item_cap, slot_cap = o_.slot_cap;
    __shared__ int nt[DSA_ORDER_MAX_SEGS];               // tiles per segment
    __shared__ int cnt[DSA_ORDER_MAX_TILES + 1];         // cnt[r]: segments with at least r tiles; then: slots before rank r
    __shared__ int part[1024];
    __shared__ int maxnt_s, sum_a;
    const int tid = threadIdx.x;
    if (N > DSA_ORDER_MAX_SEGS) {
        if (tid == 0) { order[0] = -1; order[1] = 0; order[2] = 0; }
        return;
    }
    if (tid == 0) { maxnt_s = 0; order[1] = 0; order[2] = 0; }
    __syncthreads();
    int mx = 0;
    for (int i = tid; i < N; i += 1024) {
        const int L = cu[i + 1] - cu[i];
        nt[i] = L > 0 ? (L + 127) / 128 : 0;
        mx = max(mx, nt[i]);
    }
    atomicMax(&maxnt_s, mx);
    __syncthreads();
    const int maxnt = maxnt_s;
    if (maxnt > DSA_ORDER_MAX_TILES) {
        if (tid == 0) order[0] = -1;
        return;
    }
    if (mode == 1) {
        // rank of a segment = segments that are longer, or as long and earlier; cnt[rank] = segment, then its first slot
        int *seg_of = cnt, *first = cnt + DSA_ORDER_MAX_SEGS;     // (both fit: DSA_ORDER_MAX_TILES + 1 >= 2 * DSA_ORDER_MAX_SEGS)
        for (int i = tid; i < N; i += 1024) {
            int rk = 0;
            for (int o = 0; o < N; ++o) rk += nt[o] > nt[i] || (nt[o] == nt[i] && o < i);
            seg_of[rk] = i;
        }
        __syncthreads();
        if (tid == 0) {                                  // N <= 4096 additions
            int run = 0;
            for (int rk = 0; rk < N; ++rk) {
                first[rk] = run;
                run += nt[seg_of[rk]];
            }
            maxnt_s = run;
        }
        __syncthreads();
        const int total = maxnt_s;
        if (total > cap) {
            if (tid == 0) order[0] = -1;
            return;
        }
        if (tid == 0) order[0] = total;
        for (int rk = 0; rk < N; ++rk) {
            const int seg = seg_of[rk], f = first[rk];
            for (int j = tid; j < nt[seg]; j += 1024) order_entry(order, cu, f + j, seg, j, 0, -1);
        }
        return;
    }
    for (int r = 1 + tid; r <= maxnt; r += 1024) {
        int c = 0;
        for (int i = 0; i < N; ++i) c += nt[i] >= r;
        cnt[r] = c;
    }
    __syncthreads();
    if (mode == 2 && maxnt <= DSA_ORDER_SPLIT_MAX_TILES) {
        // A tile of rank r is cut into ceil((128 r / qb) / pb) pieces of equal length.  pb = `share8` eighths of the steps
        // that a balanced launch gives each of its `slots` concurrent workgroups, and `extra` (a piece costs as much as 7 to 9 steps
        // besides its own, and its partial sums), or the first of the larger candidates (an eighth of an octave apart) whose entries and
        // partial sums fit.  Launches of one workgroup per CU start from a quarter of `extra`, up to the usual pb only with candidates
        // whose pieces all run at once.  Key side with the list and the sum over pieces, us, against the usual pb alone and candidates a
        // quarter of an octave apart: 2048 tokens in four segments at head_dim 256 70 -> 57, 16 384 in 33 330 -> 310, 4000 in three 114 ->
        // 98; one segment of 4000: level; two workgroups per CU (8192 tokens in seven segments at 128): 131 -> 143, so not there.
        if (tid == 0) sum_a = 0;
        __syncthreads();
        const int spt = 128 / qb, longest = maxnt * spt;          // steps of a rank
        {
            int mine = 0;
            for (int r = 1 + tid; r <= maxnt; r += 1024) mine += cnt[r] * r * spt;
            if (mine) atomicAdd(&sum_a, mine);
        }
        __syncthreads();
        const int64_t ideal = ((int64_t)sum_a * wg_per_tile + o_.slots - 1) / o_.slots;
        const int64_t even = ideal * o_.share8 / 8 + o_.extra;
        const int pb0 = max((int)min(ideal * o_.share8 / 8 + (o_.slots > 256 ? o_.extra : o_.extra / 4), (int64_t)longest), max(8, 32 / qb));
        auto candidate = [&](int k) { return (pb0 * (8 + (k & 7)) << (k >> 3)) / 8; };
        {
            const int k = tid >> 4, pbk = candidate(k);              // 16 threads a candidate
            const float inv = 1.f / (float)pbk;
            int ni = 0, nm = 0;
            for (int r = 1 + (tid & 15); r <= maxnt; r += 16) {
                const int up = r * spt + pbk - 1;                    // (below 2^24: a float holds it)
                int np = (int)((float)up * inv);
                np += (np + 1) * pbk <= up;
                np -= np * pbk > up;
                ni += cnt[r] * np;
                if (np > 1) nm += cnt[r] * np;
            }
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) {
                ni += __shfl_xor(ni, off, 64);
                nm += __shfl_xor(nm, off, 64);
            }
            if ((tid & 15) == 0)
                part[k] = ni <= item_cap && ni <= cap && nm <= slot_cap && (pbk >= min(even, (int64_t)longest) || (int64_t)ni * wg_per_tile <= o_.slots);
        }
        __syncthreads();
        const uint64_t fits = __ballot(part[tid & 63] != 0);
        const int pb = fits ? candidate(__ffsll((unsigned long long)fits) - 1) : 1 << 30;
        __syncthreads();
        // thread tid owns rank r = tid + 1.  Entries are listed by length (then by rank, then by segment): its entries, partial slots
        // and cut tiles start behind those of the ranks in front of it.
        const int r = 1 + tid, c = r <= maxnt ? cnt[r] : 0, steps = r * spt, np = (steps + pb - 1) / pb;
        if (r <= maxnt) part[tid] = ((steps + np - 1) / np << 13) | np;         // at most 2^16 steps, 2^13 pieces
        __syncthreads();
        int slot = 0, ms = 0, mt = 0, total = 0, cuts = 0;
        const int me = r <= maxnt ? part[tid] : 0;
        for (int o = maxnt; o >= 1; --o) {
            const int it = part[o - 1], no = it & 8191, co = cnt[o];
            total += co * no;
            if (no > 1) cuts += co;
            if ((it >> 13) > (me >> 13) || ((it >> 13) == (me >> 13) && o > r)) {
                slot += co * no;
                if (no > 1) { ms += co * no; mt += co; }
            }
        }
        if (total > cap || total > item_cap) {           // (only when even whole walks do not fit)
            if (tid == 0) order[0] = -1;
            return;
        }
        if (tid == 0) { order[0] = total; order[1] = pb >= longest ? 0 : pb * qb; order[2] = cuts; }
        if (c) {
            int32_t *cut = order + 4 + 4 * cap;          // entries of the first pieces of the cut tiles, for the reduction
            for (int i = 0; i < N; ++i)
                if (nt[i] >= r) {
                    if (np > 1) cut[mt++] = slot;
                    for (int pc = 0; pc < np; ++pc) order_entry(order, cu, slot++, i, nt[i] - r, pc, np > 1 ? ms : -1);
                    if (np > 1) ms += np;
                }
        }
        return;
    }
    // slots before rank r = sum of cnt[r'] over r' > r: ranks are cut into 1024 runs (run t = the ranks
    // maxnt - t per .. downwards), a scan over the runs' sums, then each thread finishes its run
    const int per = (maxnt + 1023) / 1024;
    int sum = 0;
    for (int u = 0; u < per; ++u) {
        const int r = maxnt - (tid * per + u);
        if (r >= 1) sum += cnt[r];
    }
    part[tid] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int add = tid >= d ? part[tid - d] : 0;
        __syncthreads();
        part[tid] += add;
        __syncthreads();
    }
    int before = part[tid] - sum;                        // slots of the runs with larger ranks
    const int total = part[1023];
    __syncthreads();
    for (int u = 0; u < per; ++u) {
        const int r = maxnt - (tid * per + u);
        if (r >= 1) {
            const int c = cnt[r];
            cnt[r] = before;
            before += c;
        }
    }
    __syncthreads();
    if (total > cap) {
        if (tid == 0) order[0] = -1;
        return;
    }
    if (tid == 0) order[0] = total;
    for (int r = 1 + tid; r <= maxnt; r += 1024) {
        int slot = cnt[r];
        for (int i = 0; i < N; ++i)
            if (nt[i] >= r) order_entry(order, cu, slot++, i, nt[i] - r, 0, -1);
    }
}
__global__ __launch_bounds__(1024) void dsa_tile_order_kernel(const int32_t *__restrict__ cu, int N, TileOrder o, int32_t *__restrict__ order) {
    tile_order(cu, N, o, order);
}
// the list by the first workgroup and delta, 64 rows each, by the others: the two things the passes of a backward on two streams
// wait for, in one launch (the list alone takes 8 to 14 us, most of it latency)
__global__ __launch_bounds__(1024) void dsa_tile_order_delta_kernel(const int32_t *__restrict__ cu, int N, TileOrder o, int32_t *__restrict__ order,
                                                                    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ out, int T,
                                                                    int Hq, int D, float *__restrict__ delta) {
    if (blockIdx.x == 0) tile_order(cu, N, o, order);
    else delta_row(dout, out, T, Hq, D, (int64_t)(blockIdx.x - 1) * 64 + (threadIdx.x >> 4), threadIdx.x & 15, delta);
}
static inline int order_entries_cap(int T) { return T / 128 + DSA_ORDER_MAX_SEGS + 1 + DSA_ORDER_EXTRA; }
extern "C" size_t dsa_tile_order_bytes(int T) { return ((size_t)order_entries_cap(T) * 5 + 4) * sizeof(int32_t); }
// Adds the pieces of every tile that was cut, in piece order, and writes its dK (times the softmax scale) and dV
// rows of D elements (`pitch` in the partial sums).  Grid: (cut tiles at most, kv heads, pitch / 8 slices of 256 units).
__global__ __launch_bounds__(256) void dsa_dkv_pieces_reduce_kernel(const int32_t *__restrict__ order, int cap,
                                                                    const float *__restrict__ partial, const int32_t *__restrict__ cu,
                                                                    int N, int Hkv, int D, int pitch, int qb, int seq_clamp, float scale, int carried,
                                                                    bf16_t *__restrict__ dk, bf16_t *__restrict__ dv) {
    if ((int)blockIdx.x >= __builtin_amdgcn_readfirstlane(order[2])) return;
    const int entry = __builtin_amdgcn_readfirstlane(order[4 + 4 * cap + blockIdx.x]);
    int s0, L, blk, piece, mslot, pb;
    if (!locate_key_tile(order, cu, N, entry, s0, L, blk, piece, mslot, pb)) return;
    if (piece != 0 || mslot < 0 || pb <= 0) return;
    L = min(L, seq_clamp);
    const int c0 = blk * 128;
    if (c0 >= L) return;
    pb /= qb;
    const int nblocks = (L - c0 + qb - 1) / qb;          // (pieces only exist for causal launches: the walk starts at the tile)
    if (nblocks <= pb) return;                           // (its walk fits one piece after all: piece 0 wrote the rows itself)
    const int np = (nblocks + pb - 1) / pb, kvh = blockIdx.y;
    // a thread's unit: eight columns of a row, in the two halves of a wave's store
    const int DT = pitch / 32, unit = blockIdx.z * 256 + threadIdx.x, j = unit & 31, part = unit >> 5;     // part: [dK | dV][key group][d-tile][8 columns]
    const int m = part / (16 * DT), grp = part / (4 * DT) % 4, col = part % (4 * DT) * 8, key = grp * 32 + j;
    if (m > 1 || key >= min(128, L - c0) || col >= D || (carried && !carried_chunk(col / 8, m))) return;
    const int64_t slot_f = 2 * 128 * (int64_t)pitch;         // floats per (slot, kv head)
    const float *src = partial + ((int64_t)mslot * Hkv + kvh) * slot_f + part * 256 + j * 4;
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
    constexpr int U = 4;                                 // pieces whose loads are in flight together
    for (int pc = 0; pc < np; pc += U) {                 // piece order: the sum does not depend on the schedule
        f32x4 x0[U], x1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float *p = src + (int64_t)min(pc + u, np - 1) * Hkv * slot_f;
            x0[u] = *reinterpret_cast<const f32x4 *>(p);
            x1[u] = *reinterpret_cast<const f32x4 *>(p + 128);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (pc + u < np) { a0 += x0[u]; a1 += x1[u]; }
    }
    const float mul = m ? 1.f : scale;
    const u32x4 w = {pack2bf(a0[0] * mul, a0[1] * mul), pack2bf(a0[2] * mul, a0[3] * mul), pack2bf(a1[0] * mul, a1[1] * mul), pack2bf(a1[2] * mul, a1[3] * mul)};
    *reinterpret_cast<u32x4 *>((m ? dv : dk) + ((int64_t)(s0 + c0 + key) * Hkv + kvh) * D + col) = w;
}

// ==================================================================================================
// launchers: instantiate per head_dim, mask kind and (power-of-two padded) group size
// ==================================================================================================

#define GS_SWITCH(FN, DD, HI, ...)                                    \
    switch (gs) {                                                     \
        case 0: launch_status = FN<DD, HI, 0>(__VA_ARGS__); break;    \
        case 1: launch_status = FN<DD, HI, 1>(__VA_ARGS__); break;    \
        case 2: launch_status = FN<DD, HI, 2>(__VA_ARGS__); break;    \
        case 3: launch_status = FN<DD, HI, 3>(__VA_ARGS__); break;    \
        default: launch_status = FN<DD, HI, 4>(__VA_ARGS__); break;   \
    }
#define TILE_SWITCH(FN, ...)                                                              \
    hipError_t launch_status = hipSuccess;                                                \
    switch (D) {                                                                          \
        case 64: if (bitmap) { GS_SWITCH(FN, 64, true, __VA_ARGS__) } else { GS_SWITCH(FN, 64, false, __VA_ARGS__) } break;    \
        case 128: if (bitmap) { GS_SWITCH(FN, 128, true, __VA_ARGS__) } else { GS_SWITCH(FN, 128, false, __VA_ARGS__) } break; \
        case 256: if (bitmap) { GS_SWITCH(FN, 256, true, __VA_ARGS__) } else { GS_SWITCH(FN, 256, false, __VA_ARGS__) } break; \
        default: return hipErrorInvalidValue;                                             \
    }                                                                                     \
    if (launch_status != hipSuccess) return launch_status;

// kv heads a workgroup of the attention-mass kernel takes (a power of two, at most what its registers hold; with
// one query head per kv head a lane also holds all sixteen sums of a tile to itself, which costs the top size)
template <int D>
static int mass_hpg(int Hq, int Hkv) {
    const int most = Hq == Hkv ? mass_heads_max<D>() / 2 : mass_heads_max<D>();
    int hpg = 1;
    while (hpg * 2 <= most && hpg < Hkv) hpg *= 2;
    return hpg;
}
extern "C" int dsa_mass_groups(int Hq, int Hkv, int D) {
    const int hpg = D == 64 ? mass_hpg<64>(Hq, Hkv) : D == 128 ? mass_hpg<128>(Hq, Hkv) : mass_hpg<256>(Hq, Hkv);
    return (Hkv + hpg - 1) / hpg;
}
template <int D, int GS, int HPG>
static hipError_t launch_mass_h(dim3 grid, hipStream_t stream, const void *q, const void *k, const float *lse,
                                const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float sl2,
                                int K, int ngroups, int chunk, float final_mul, float *table) {
    if constexpr (HPG > (GS == 0 ? mass_heads_max<D>() / 2 : mass_heads_max<D>())) {     // (mass_hpg asks for no more)
        return hipErrorInvalidValue;
    } else {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&dsa_tile_mass_kernel<D, GS, HPG>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)mass_lds_bytes<D, GS, HPG>());
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((dsa_tile_mass_kernel<D, GS, HPG>), grid, dim3(256 * mass_sets<HPG>()), (mass_lds_bytes<D, GS, HPG>()), stream,
                           (const bf16_t *)q, (const bf16_t *)k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk,
                           final_mul, table);
        return hipSuccess;
    }
}
template <int D, bool HAS_IDX, int GS>
static hipError_t launch_mass_i(dim3 grid, hipStream_t stream, const void *q, const void *k, const float *lse,
                          const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float sl2,
                          int K, int ngroups, int chunk, float final_mul, float *table) {
    switch (mass_hpg<D>(Hq, Hkv)) {
        case 1: return launch_mass_h<D, GS, 1>(grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk, final_mul, table);
        case 2: return launch_mass_h<D, GS, 2>(grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk, final_mul, table);
        case 4: return launch_mass_h<D, GS, 4>(grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk, final_mul, table);
        case 8: return launch_mass_h<D, GS, 8>(grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk, final_mul, table);
        default: return launch_mass_h<D, GS, 16>(grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, sl2, K, ngroups, chunk, final_mul, table);
    }
}
// attention mass of the selected keys: the heads of a query summed in registers, scaled by 1/Hq and written into
// mass (T,K); batches with more kv heads than one workgroup holds leave one (T,K) table per group in `partial`,
// which dsa_mass_reduce_kernel adds in group order
extern "C" hipError_t dsa_launch_tile_mass(const void *q, const void *k, const float *lse, const uint32_t *bitmap,
                                           int ldw, const int32_t *n, const int32_t *cu, int N, int T, int Hq, int Hkv,
                                           int D, int K, float scale, float *partial, float *mass, hipStream_t stream) {
    const int gs = group_shift(Hq, Hkv);
    const int ngroups = dsa_mass_groups(Hq, Hkv, D);
    const int64_t blocks = ((int64_t)T / ((32 * 4) >> gs) + N + 1) * ngroups;
    // walks (ldw tiles at most) stay whole from four workgroups per CU on; below, pieces of at least 8 tiles (a tile takes
    // about 3 us, the q rows of a piece as long as one or two tiles), as many as give the chip about four rounds
    const int64_t chunk_fit = blocks * ldw / (2 * 4 * 256) / 8 * 8;
    const int chunk = blocks >= 4 * 256 ? ldw : (int)std::max<int64_t>(chunk_fit, 8);
    const dim3 grid((unsigned)blocks, (unsigned)((ldw + chunk - 1) / chunk));
    const float inv_hq = 1.f / (float)Hq;
    float *table = ngroups == 1 ? mass : partial;
    const float final_mul = ngroups == 1 ? inv_hq : 1.f;
    TILE_SWITCH(launch_mass_i, grid, stream, q, k, lse, bitmap, ldw, cu, N, T, Hq, Hkv, scale * LOG2E_F, K, ngroups, chunk, final_mul, table)
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ngroups == 1) return e;
    const unsigned parts = (unsigned)((K / 4 + 255) / 256 > 0 ? (K / 4 + 255) / 256 : 1);
    hipLaunchKernelGGL(dsa_mass_reduce_kernel, dim3(T, parts < 8 ? parts : 8), dim3(256), 0, stream, partial, n, T, K, ngroups,
                       inv_hq, mass);
    return hipGetLastError();
}
// bytes of fp32 partial sums a launch of T tokens may use for key-tile walks in pieces (0: launches of this size are
// never cut); a slot = the dK and dV of one 128-key tile and kv head
extern "C" size_t dsa_tile_dkv_partial_bytes(int T) {
    if (T <= 0 || T > 131072) return 0;
    const size_t b = (size_t)T * 16384;
    return b < ((size_t)128 << 20) ? b : ((size_t)128 << 20);
}
// How the key-side launch of these sizes hands out its tiles.  `order` (dsa_tile_order_bytes(T) bytes, or null): the tiles are
// listed longest walk first before the launch.  A launch of at most four workgroups per CU may also cut long walks into pieces
// (`partial`: fp32 partial sums), so that it does not end on a few long walks with most of the chip idle.
struct DkvPlan { int tiles_ub, pitch; bool listed, pieces; TileOrder o; };
static DkvPlan dkv_plan(int T, int N, int Hq, int Hkv, int d_real, bool has_idx, int causal, const void *order, const void *partial, size_t partial_bytes) {
    DkvPlan p;
    p.tiles_ub = T / 128 + N;                            // 128-key tiles of all segments, at most
    p.pitch = has_idx ? d_real : (dense_kernel_dim(d_real) + 31) / 32 * 32;             // row of a partial sum
    const int wg_per_tile = Hkv, kg = dkv_key_groups(d_real, T, N, Hq, Hkv, causal);
    const int64_t slot_pairs = partial ? (int64_t)(partial_bytes / ((size_t)2 * 128 * p.pitch * sizeof(float))) : 0;
    p.pieces = order && causal && slot_pairs >= Hkv && (int64_t)p.tiles_ub * wg_per_tile <= dkv_pieces_max_wg(d_real);
    p.listed = order && (N > 1 || p.pieces);             // (one segment: its tiles are in order already)
    const int cap = order_entries_cap(T), item_cap = p.pieces ? std::min(cap, p.tiles_ub + (1024 + wg_per_tile - 1) / wg_per_tile) : cap;
    p.o = TileOrder{cap, p.pieces ? 2 : (causal ? 0 : 1), 32 >> group_shift(Hq, Hkv), wg_per_tile, item_cap,
                    (int)(slot_pairs / Hkv < (1 << 20) ? slot_pairs / Hkv : (1 << 20)),       // (sums stay below 2^21)
                    dkv_slots(kg), kg == 1 ? 8 : 6, kg == 1 ? 16 : 32};          // see tile_order
    return p;
}
// delta and, where the key-side launch of the same sizes will want it, its list
extern "C" hipError_t dsa_launch_tile_order_delta(const void *dout, const void *out, const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real,
                                                  int has_idx, int causal, int32_t *order, const float *partial, size_t partial_bytes,
                                                  float *delta, hipStream_t stream) {
    const DkvPlan p = dkv_plan(T, N, Hq, Hkv, d_real, has_idx != 0, causal, order, partial, partial_bytes);
    if (!p.listed) return hipErrorNotReady;
    hipLaunchKernelGGL(dsa_tile_order_delta_kernel, dim3((unsigned)(1 + ((int64_t)T * Hq + 63) / 64)), dim3(1024), 0, stream, cu, N, p.o, order,
                       (const bf16_t *)dout, (const bf16_t *)out, T, Hq, d_real, delta);
    return hipGetLastError();
}
extern "C" hipError_t dsa_launch_dkv_tiles(unsigned grid, hipStream_t stream, const void *dout, const void *q, const void *k, const void *v,
                                           const float *lse, const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N,
                                           int T, int Hq, int Hkv, int d_real, float scale, int carried, int causal, int skip_len, const int32_t *order,
                                           float *partial, void *dk, void *dv);
extern "C" hipError_t dsa_launch_dkv_dq_tiles(unsigned key_blocks, hipStream_t stream, const void *dout, const void *q, const void *k, const void *v,
                                              const float *lse, const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N,
                                              int T, int Hq, int Hkv, float scale, int carried, int causal, const int32_t *order, float *partial,
                                              void *dk, void *dv, int window, void *dq);
// listed: dsa_launch_tile_order_delta has left the list in `order`.  beside: null, or dQ in the same launch (head_dim 256)
extern "C" hipError_t dsa_launch_tile_dkv(const void *dout, const void *q, const void *k, const void *v,
                                          const float *lse, const float *delta, const uint32_t *bitmap, int ldw,
                                          const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real, float scale, int carried, int causal, int skip_len,
                                          int32_t *order, int listed, float *partial, size_t partial_bytes, void *dk, void *dv,
                                          const DqBeside *beside, hipStream_t stream) {
    const int gs = group_shift(Hq, Hkv);
    const DkvPlan p = dkv_plan(T, N, Hq, Hkv, d_real, bitmap != nullptr, causal, order, partial, partial_bytes);
    dim3 grid((unsigned)((p.pieces ? p.o.item_cap : p.tiles_ub + 1) * Hkv));
    if (!p.listed) order = nullptr;
    else if (!listed) hipLaunchKernelGGL(dsa_tile_order_kernel, dim3(1), dim3(1024), 0, stream, cu, N, p.o, order);
    if (!p.pieces) partial = nullptr;
    const hipError_t e = beside ? dsa_launch_dkv_dq_tiles(grid.x, stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, carried, causal,
                                                          order, partial, dk, dv, beside->window, beside->dq) :
                         dsa_launch_dkv_tiles(grid.x, stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, carried,
                                              causal, skip_len, order, partial, dk, dv);
    if (e != hipSuccess) return e;
    if (p.pieces)
        hipLaunchKernelGGL(dsa_dkv_pieces_reduce_kernel, dim3(p.tiles_ub, Hkv, p.pitch / 8), dim3(256), 0, stream, order,
                           p.o.cap, partial, cu, N, Hkv, d_real, p.pitch, 32 >> gs, bitmap ? ldw * 32 : 0x7fffffff, scale, carried,
                           (bf16_t *)dk, (bf16_t *)dv);
    return hipGetLastError();
}
