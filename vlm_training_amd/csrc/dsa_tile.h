// Helpers shared by the tile kernels (32x32 MFMA tiles over packed segments): LDS tiles, masks, the hand-out of blocks.
#pragma once
#include "dsa_common.h"
#include <type_traits>

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }   // v_exp_f32; exp2(-inf) = 0

// all-ones if bit `b` of `word` is set, else 0 (v_bfe_i32 when b is a compile-time constant)
__device__ __forceinline__ uint32_t bit_mask(uint32_t word, int b) {
    return (uint32_t)(((int32_t)(word << (31 - b))) >> 31);
}
// x where keep is all-ones, -inf where it is 0 (one v_bfi_b32 / v_bitop3_b32)
__device__ __forceinline__ float keep_or_neginf(float x, uint32_t keep) {
    return __uint_as_float((keep & __float_as_uint(x)) | (~keep & 0xff800000u));
}
// bits j <= d of a 32-key tile (keys at or before the diagonal when d = query column - tile start)
__device__ __forceinline__ uint32_t causal_bits(int d) { return d >= 31 ? 0xffffffffu : (d < 0 ? 0u : ((2u << d) - 1u)); }
// A transposed operand of mfma32: ds_read_b64_tr_b16 - within 16 lanes, lane s supplies the address of 4 consecutive elements of row
// R + s/4 at column m0 + 4*(s%4) and receives rows R..R+3 of column m0 + s - twice
typedef __attribute__((address_space(3))) unsigned char lds_u8;
__device__ __forceinline__ bf16x8 tr_pair(lds_u8 *p0, lds_u8 *p1) {
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)p0);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)p1);
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 r = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(bf16x8, r);
}
__device__ __forceinline__ bf16x8 pack8(const float *x) {
    const u32x4 w = {pack2bf(x[0], x[1]), pack2bf(x[2], x[3]), pack2bf(x[4], x[5]), pack2bf(x[6], x[7])};
    return __builtin_bit_cast(bf16x8, w);
}
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.f;
    return z;
}

// Write one 32-column d-tile of a C-layout accumulator as bf16 (lane = row j; a lane holds the four
// columns 8*g4 + 4*h + {0..3} of every group g4, so a 16-byte chunk of the row is split over the two
// lanes 32 apart).  The halves of the wave exchange 8-byte pieces - lane (j,0) takes chunk 2m whole,
// lane (j,1) chunk 2m+1 - and every lane stores 16 bytes.  Both lanes of a row must be active.
// `chunks`: 16-byte chunks of the row that exist from this d-tile on (4 and more: all of it).
__device__ __forceinline__ void store_c_tile(bf16_t *row_dt, const f32x16 &acc, float mul, int h, int chunks = 4) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const uint32_t a0 = pack2bf(acc[8 * m] * mul, acc[8 * m + 1] * mul), a1 = pack2bf(acc[8 * m + 2] * mul, acc[8 * m + 3] * mul);
        const uint32_t b0 = pack2bf(acc[8 * m + 4] * mul, acc[8 * m + 5] * mul), b1 = pack2bf(acc[8 * m + 6] * mul, acc[8 * m + 7] * mul);
        const auto r0 = __builtin_amdgcn_permlane32_swap(a0, b0, false, false);   // upper lanes of a <-> lower lanes of b
        const auto r1 = __builtin_amdgcn_permlane32_swap(a1, b1, false, false);
        const u32x4 w = {r0[0], r1[0], r0[1], r1[1]};
        if (2 * m + h < chunks) *reinterpret_cast<u32x4 *>(row_dt + 8 * (2 * m + h)) = w;
    }
}

// Sum / maximum (of values >= 0) over the wave, wave-uniform: DPP steps inside the rows of sixteen lanes, then across them -
// no LDS round trips (the search below takes about ten of these sums in front of a workgroup's first load; by lane
// shuffles they cost it 2 us).
template <class F>
__device__ __forceinline__ int wave_fold_i(int x, F f) {
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));      // row_shr:1
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));      // row_shr:2
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));      // row_shr:4
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));      // row_shr:8: lane 15 of a row has the row
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));      // row_bcast:15 into rows 1 and 3
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));      // row_bcast:31 into rows 2 and 3
    return __builtin_amdgcn_readlane(x, 63);
}
__device__ __forceinline__ int wave_sum_i(int x) { return wave_fold_i(x, [](int a, int b) { return a + b; }); }
__device__ __forceinline__ int wave_max_i(int x) { return wave_fold_i(x, [](int a, int b) { return max(a, b); }); }
// Sums over the lanes up to and with one's own, the same way
__device__ __forceinline__ int wave_prefix_i(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return x;
}

// slot -> (segment, block) for blocks of `blk` columns handed out segment by segment; within a segment
// the blocks are numbered from the end when `reverse` (heaviest causal blocks first).  Returns false
// for spare slots.  The segments are searched 64 at a time, one per lane: where one's blocks begin is a sum over the lanes in front (a walk from
// segment to segment took a workgroup 3100 clocks with 16 of them, 8200 with 64).
__device__ __forceinline__ bool locate_block(const int32_t *cu, int N, int slot, int blk, bool reverse, int &s0, int &L,
                                             int &b) {
    const int lane = threadIdx.x & 63;
    for (int base = 0; base < N; base += 64) {
        const int seg = min(base + lane, N - 1);
        const int lo = cu[seg], len = cu[seg + 1] - lo;
        const int nb = base + lane < N ? (len + blk - 1) / blk : 0, upto = wave_prefix_i(nb);
        const uint64_t past = __builtin_amdgcn_ballot_w64(upto > slot);
        if (past) {
            const int w = (int)__builtin_ctzll(past);
            s0 = __builtin_amdgcn_readlane(lo, w);
            L = __builtin_amdgcn_readlane(len, w);
            const int n = __builtin_amdgcn_readlane(nb, w), at = slot - (__builtin_amdgcn_readlane(upto, w) - n);
            b = reverse ? n - 1 - at : at;
            return true;
        }
        slot -= __builtin_amdgcn_readlane(upto, 63);
    }
    return false;
}

// The same hand-out, heaviest block first over the whole batch: slot 0 takes the last block of the longest segment,
// then every block with the next lower index in segment order, and so on - a block's walk grows with its index, so
// long walks start first wherever their segment lies in the batch (with the segment-by-segment order the long
// walks of a late segment start late and the launch ends on them).  For up to 64 segments (their lengths live in
// one wave's lanes); larger batches fall back to the segment-by-segment order.
__device__ __forceinline__ bool locate_block_heaviest_first(const int32_t *cu, int N, int slot, int blk, int &s0, int &L,
                                                            int &b) {
    if (N > 64) return locate_block(cu, N, slot, blk, true, s0, L, b);
    const int lane = threadIdx.x & 63;
    const int seg = min(lane, N - 1);
    const int lo = cu[seg], len = cu[seg + 1] - lo;
    const int nb = lane < N ? (len + blk - 1) / blk : 0;
    const int most = wave_max_i(nb);
    // blocks with index >= x over all segments
    auto count_ge = [&](int x) { return wave_sum_i(max(nb - x, 0)); };
    if (slot >= count_ge(0)) return false;
    int lo_b = 0, hi_b = most;                           // count_ge(lo_b) > slot >= count_ge(hi_b)
    while (hi_b - lo_b > 1) {
        const int mid = (lo_b + hi_b) >> 1;
        if (count_ge(mid) > slot) lo_b = mid; else hi_b = mid;
    }
    b = lo_b;
    const int rank = slot - count_ge(b + 1);             // among the segments that have a block b, in segment order
    const uint64_t has = __builtin_amdgcn_ballot_w64(nb > b);
    // the rank-th set bit of `has`
    const int below = (int)__popcll(has & ((1ull << lane) - 1ull));
    const uint64_t me = __builtin_amdgcn_ballot_w64(nb > b && below == rank);
    const int w = (int)__builtin_ctzll(me);
    s0 = __builtin_amdgcn_readlane(lo, w);
    L = __builtin_amdgcn_readlane(len, w);
    return true;
}

// Query blocks are handed out heaviest first: over the whole batch for launches of a few rounds of workgroups (they
// would otherwise end on the long walks of a late segment: forward -11 %, dQ -15 % on 8192 tokens in seven
// segments), segment by segment for larger ones, where the blocks of a segment that run side by side share their
// K / V tiles in L2 (the batch-wide order is 2-3 % slower there).
// Without a causal mask the walks of a segment are equally long and there is nothing to balance inside it: segment by segment
// (12 288 patches of 13 images, forward and backward: 485 us, in the batch-wide order 549).
#define DSA_BATCH_ORDER_MAX_BLOCKS (6 * 256)
#define LOCATE_QUERY_BLOCK(causal, blocks, cu, N, slot, blk, s0, L, b)                                           \
    ((causal) && (blocks) <= DSA_BATCH_ORDER_MAX_BLOCKS ? locate_block_heaviest_first(cu, N, slot, blk, s0, L, b)          \
                                             : locate_block(cu, N, slot, blk, true, s0, L, b))

// ---- LDS tiles filled straight from memory ------------------------------------------------------------------------------
// 32 rows of D bf16 (head_dim 80 and 96: of 128, columns past the true head_dim zero).  A load puts 1 KiB of one wave at consecutive addresses, so
// rows cannot be padded one by one; instead groups of rows (1 KiB at head_dim 64, four rows else) are 16 bytes apart, and the
// 16-byte chunk c of row r sits at position c ^ x(r), x = 4 (r & 3) (head_dim 64: 4 (bit 1 of r) + 2 (bit 2)): sixteen
// consecutive rows at one chunk (row-wise operand) and four consecutive rows at four neighbouring chunks (transposed operand,
// 32 lanes) each cover the 64 banks once.  The XOR is applied to the source address of a load.
template <int D>
struct DirectTile {
    static constexpr int ROW_B = D == 96 || D == 80 ? 256 : 2 * D;                  // bytes per row
    static constexpr int CPR = ROW_B / 16;                               // chunks per row
    static constexpr int GROUP = D == 64 ? 8 : 4;                        // rows between two gaps
    static constexpr int GROUP_B = GROUP * ROW_B + 16;
    static constexpr int BYTES = 32 / GROUP * GROUP_B;
    static constexpr int LOADS = 32 * ROW_B / 1024;                      // wave loads of a tile
    static constexpr int LOAD_ROWS = 1024 / ROW_B;                       // rows of one of them (1 at most for head_dim 512)
    static constexpr int SOURCES = D == 256 ? 2 : 1;                     // pieces after which x repeats (from an even piece on)
    __device__ __forceinline__ static constexpr int load_lds(int p) {              // LDS offset of wave load p
        return p * LOAD_ROWS / GROUP * GROUP_B + p * LOAD_ROWS % GROUP * ROW_B;
    }
    __device__ __forceinline__ static int xor_of(int row) { return D == 64 ? ((row >> 1) & 1) * 4 + ((row >> 2) & 1) * 2 : (row & 3) << 2; }
    // byte offset, from the first row of the tile, that `lane` reads in wave load p; chunks at and past `chunks` read as zero
    __device__ __forceinline__ static int source(int p, int lane, int row_stride_b, int chunks) {
        const int row = p * LOAD_ROWS + lane / CPR, c = (lane % CPR) ^ xor_of(row);
        return c < chunks ? row * row_stride_b + c * 16 : (int)0x80000000;
    }
    int rowq[4], trq[4];
    __device__ __forceinline__ void init(int lane) {
        const int h = lane >> 5, j = lane & 31, s = lane & 15, i = s >> 2;
        const int low = ((lane >> 4) & 1) * 2 + ((s & 3) >> 1), sub = (s & 1) << 3;
        const int rb = j / GROUP * GROUP_B + j % GROUP * ROW_B;
        const int tr_row = 4 * h + i, tb = tr_row / GROUP * GROUP_B + tr_row % GROUP * ROW_B;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            rowq[q] = D == 64 ? rb + (((2 * q + h) ^ xor_of(j)) << 4) : rb + ((q ^ (j & 3)) << 6) + h * 16;
            trq[q] = D == 64 ? tb + (((4 * (q & 1) + low) ^ xor_of(tr_row)) << 4) + sub : tb + ((q ^ i) << 6) + low * 16 + sub;
        }
    }
    // k-step ks of a row-wise operand: which of rowq, and what to add
    static constexpr int row_q(int ks) { return D == 64 ? ks : (ks >> 1) & 3; }
    static constexpr int row_imm(int ks) { return D == 64 ? 0 : (ks >> 3) * 256 + (ks & 1) * 32; }
    static constexpr int tr_q(int dt) { return dt & 3; }
    static constexpr int tr_imm(int dt, int v) { return (D == 64 ? 0 : (dt >> 2) * 256) + v * (8 / GROUP) * GROUP_B; }
};

// Where the rows of a wave lie that a piece of a tile holds, a row being a (query, head of the kv group): rows first + p * LOAD_ROWS + l of the
// wave's first query on, l = lane / CPR.  A piece never splits a query's heads unevenly, so that a row's place is a sum of what the piece
// and what the lane says.
template <class TL>
struct WaveRows {
    int gshift, lane_query, lane_head;
    __device__ __forceinline__ WaveRows(int gshift_, int lane) : gshift(gshift_), lane_query((lane / TL::CPR) >> gshift_), lane_head((lane / TL::CPR) & ((1 << gshift_) - 1)) {}
    // of row first + p * LOAD_ROWS + l: the query behind the wave's first one, the head
    __device__ __forceinline__ int query(int p, int first = 0) const { return ((first + p * TL::LOAD_ROWS) >> gshift) + lane_query; }
    __device__ __forceinline__ int head(int p, int first = 0) const { return ((first + p * TL::LOAD_ROWS) & ((1 << gshift) - 1)) + lane_head; }
    // its byte offset from the first query's first head: tok_b, head_b bytes from one query, one head to the next
    __device__ __forceinline__ int place(int tok_b, int head_b) const { return lane_query * tok_b + lane_head * head_b; }
    __device__ __forceinline__ int piece(int p, int tok_b, int head_b, int first = 0) const {
        return ((first + p * TL::LOAD_ROWS) >> gshift) * tok_b + ((first + p * TL::LOAD_ROWS) & ((1 << gshift) - 1)) * head_b;
    }
};

// ---- one wave per SIMD: sums in accumulation registers, phases of mixed operands ----
// c += a b with c in accumulation registers, named here: left to itself the compiler keeps 128 to 256 registers of sums where the
// vector instructions need them, and spills.  It does not see an MFMA in this statement, so its hazards are held by hand: an operand
// that a vector instruction wrote needs two wait states (operands come from LDS or are formed many MFMAs ahead), a result that one
// reads eleven; the last MFMA on a tuple in front of a join or of the stores (`last`) waits itself.  tests/test_key_side.py looks for both in the compiled kernels (a copy of a tuple
// that the compiler placed a wait state too close was enough to spoil dK).
__device__ __forceinline__ void mfma32_agpr(f32x16 &c, bf16x8 a, bf16x8 b, bool last) {
    if (last) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\ts_nop 11" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    __builtin_amdgcn_sched_barrier(0);                   // (nor does it see where the vector instructions behind it belong)
}
// the same behind operands that the compiler may have just moved or formed: it waits for them itself
__device__ __forceinline__ void mfma32_agpr_late(f32x16 &c, bf16x8 a, bf16x8 b, bool last) {
    if (last) asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\ts_nop 11" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    __builtin_amdgcn_sched_barrier(0);
}
// the tuple's value lies in accumulation registers here; in front of its uses: the tuples leave them one by one
__device__ __forceinline__ void settle(f32x16 &c) { asm volatile("" : "+a"(c)); }
// a wave's N pieces of a tile, one behind the other; N0, N1, N2 = LDS bytes from one to the next (see buffer_load_lds16)
template <int N, int N0, int N1, int N2>
__device__ __forceinline__ void buffer_load_lds16_n(buffer_rsrc rsrc, const int (&voff)[N], uint32_t lds) {
    static_assert(N == 1 || N == 2 || N == 4, "");
    if constexpr (N == 1)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(voff[0]), "s"(rsrc), "s"(lds) : "memory", "m0");
    if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %2, 0 offen lds\n\ts_add_u32 m0, m0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     : : "v"(voff[0]), "v"(voff[1]), "s"(rsrc), "s"(lds), "n"(N0) : "memory", "m0", "scc");
    if constexpr (N == 4)
        asm volatile("s_mov_b32 m0, %5\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %4, 0 offen lds\n\ts_add_u32 m0, m0, %6\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %4, 0 offen lds"
                     "\n\ts_add_u32 m0, m0, %7\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %4, 0 offen lds\n\ts_add_u32 m0, m0, %8\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, 0 offen lds"
                     : : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(rsrc), "s"(lds), "n"(N0), "n"(N1), "n"(N2) : "memory", "m0", "scc");
}
// fp32 tensors of head_dim 64 come as rows of 256, four parts of 64 (dsa_split_bf16_stack): the last part is zeros, and of a result two
// parts are read.  `CARRIED` kernels of head_dim 256 run 12 of the 16 k-steps and the four 32-wide d-tiles that are read: parts 0 and 1
// (out, dK) or 0 and 2 (dQ, dV), the same bits.  2048 tokens in four segments, 8 heads over 2, us, all of a row -> those: forward 34 -> 28.7,
// dQ 41 -> 31, dK/dV 42 -> 29.5 (of it 5 to 10 a fixed start and end).
#define DSA_CARRIED_KS 12
__host__ __device__ constexpr int carried_tile(int dt) { return dt < 2 ? dt : dt + 2; }      // d-tile of parts 0 | 2
__device__ __forceinline__ bool carried_chunk(int c, bool second) { return second ? !(c & 8) && c < 24 : c < 16; }   // 16-byte chunk c of parts 0 | 2 (second), 0 | 1
// Order of a phase's NR row-wise and NT transposed operands: `PRE` transposed ones, then both kinds evenly mixed.
template <int NR, int NT, int PRE>
struct PhaseOrder {
    static constexpr int M = NR + NT;
    static constexpr int rows_before(int m) { return m <= PRE || M == PRE ? 0 : (m - PRE) * NR / (M - PRE); }
    static constexpr bool is_row(int m) { return rows_before(m + 1) > rows_before(m); }
    static constexpr int index(int m) { return is_row(m) ? rows_before(m) : m - rows_before(m); }
};

// ---- walks of key tiles (dK, dV) ----
#define DSA_ORDER_MAX_SEGS 4096
// the tile (and the piece of its walk) of workgroup slot `slot`: from the order table when there is one, else
// segment by segment
__device__ __forceinline__ bool locate_key_tile(const int32_t *order, const int32_t *cu, int N, int slot, int &s0, int &L, int &blk,
                                                int &piece, int &mslot, int &pb) {
    piece = 0;
    mslot = -1;
    pb = 0;
    if (order && N <= DSA_ORDER_MAX_SEGS) {
        // (every lane reads the same words; the lane reads tell the compiler that the results are wave-uniform.  The table has room
        // for every slot of a launch of that many segments: header and entry come in one round trip.)
        const int4 hd = *reinterpret_cast<const int4 *>(order), e = *reinterpret_cast<const int4 *>(order + 4 + 4 * slot);
        const int total = __builtin_amdgcn_readfirstlane(hd.x);
        if (total >= 0) {
            if (slot >= total) return false;
            const int tp = __builtin_amdgcn_readfirstlane(e.z);
            s0 = __builtin_amdgcn_readfirstlane(e.x);
            L = __builtin_amdgcn_readfirstlane(e.y);
            blk = tp & 8191;
            piece = tp >> 13;
            mslot = __builtin_amdgcn_readfirstlane(e.w);
            pb = max(__builtin_amdgcn_readfirstlane(hd.y), 0);
            return true;
        }
    }
    return locate_block(cu, N, slot, 128, false, s0, L, blk);
}
// A walk of `nblocks` steps (block nblocks-1-b at step b, `QB` queries each, the queries q0 .. Lq-1) cut into equal pieces of
// at most `pb` steps: narrows q0, Lq and nblocks to piece `piece` and returns the number of pieces (1: the whole walk,
// 0: this piece is empty).  Block boundaries stay where they are, so a piece's blocks are the walk's own.
__device__ __forceinline__ int walk_piece(int pb, int piece, int QB, int &q0, int &Lq, int &nblocks) {
    if (pb <= 0 || nblocks <= pb) return piece == 0 ? 1 : 0;
    const int np = (nblocks + pb - 1) / pb, len = (nblocks + np - 1) / np;
    if (piece >= np) return 0;
    const int b_lo = min(piece * len, nblocks), b_hi = min(b_lo + len, nblocks);
    if (b_lo > 0) Lq = q0 + (nblocks - b_lo) * QB;
    q0 += (nblocks - b_hi) * QB;
    nblocks = b_hi - b_lo;
    return np;
}
// fp32 partial dK / dV of piece `piece` of a tile in pieces: [slot][kv head][dK | dV][key group][d-tile][8 columns][lane][4], as
// the accumulators lie in a wave, so that its stores are whole
__device__ __forceinline__ float *piece_partial(float *partial, int mslot, int piece, int Hkv, int kvh, int DT) {
    return partial + ((int64_t)(mslot + piece) * Hkv + kvh) * (2 * 128 * 32 * (int64_t)DT);
}
__device__ __forceinline__ void store_c_tile_f32(float *p, const f32x16 &acc, int lane) {
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
        const f32x4 w = {acc[4 * g4], acc[4 * g4 + 1], acc[4 * g4 + 2], acc[4 * g4 + 3]};
        *reinterpret_cast<f32x4 *>(p + g4 * 256 + lane * 4) = w;
    }
}

// ---- indexer backward ----
// The query side over the selected keys alone (dsa_tile_idxg.hip) instead of over every causal tile (dsa_tile_idx.hip): a segment this much
// longer than the selection.  Whole backward, us, tiles against gather, 64 heads of 128: selection of 2048 keys in segments of 2048
// 609 / 646, 3072: 1246 / 1200, 4096: 2146 / 1951, 5120: 2351 / 2016; 16 384 tokens in one 7441 / 4805; 512 keys in segments of 1536
// 518 / 426; 256 keys in segments of 300 197 / 250.  32 heads (a tile is half the matrix work for the same keys) of 64: 1024 keys in
// segments of 2048 193 / 196, 3072: 393 / 353, 4096: 646 / 529; of 700 to 1800: 146 / 163; of 128, in 2048: 331 / 362.
// Each segment by its own length: a launch whose bound of the longest one reaches the line runs both kernels, and the workgroups of the
// other's segments leave at once.  Against one kernel by that bound: segments of 680 to 1799, 512 keys 157 -> 150 (64 heads: 371 -> 381); one
// of 4096 beside 24 of 256 523 -> 490; four of 2048, 512 keys, under a bound of 8192 680 -> 570; 32 768 tokens level.
__host__ __device__ inline bool idx_segment_gathers(int Hi, int K, int L) { return 2 * (int64_t)L >= (Hi > 32 ? 3 : 6) * (int64_t)K; }

// ---- launches ----
// log2 of the rows a query takes: its group's heads, padded to a power of two
static inline int group_shift(int Hq, int Hkv) {
    const int G = Hq / Hkv;
    int gshift = 0;
    while ((1 << gshift) < G) ++gshift;
    return gshift;
}
// The factor of the logits for a softmax scale: kernels that divide by it, or mask in front of it, cannot take one at or next to zero.  At
// 2^-80 instead a logit below 2^40 is below 2^-40, which the exponential takes for zero as well; gradients take the scale itself.
static inline float logit_scale(float scale) { return scale > -0x1p-80f && scale < 0x1p-80f ? 0x1p-80f : scale; }
// Rows of d_real elements, a multiple of 8: without a selection the kernel of the next head_dim of 64, 80, 96, 128 reads and writes
// such rows where they lie (80: five k-steps instead of six for the S and dP of 72- and 80-wide vision heads)
static inline int dense_kernel_dim(int d_real) { return d_real <= 64 ? 64 : d_real <= 80 ? 80 : d_real <= 96 ? 96 : d_real <= 128 ? 128 : d_real; }
