// Stage D1: lightning-indexer scores on bf16 MFMA.
//
//   score[t,s] = scale * sum_j w[t,j] * relu( q_idx[t,j,:] . k_idx[s,:] ),   s in [seg_start(t), t]
//
// GEMM view: rows = (query, indexer head), columns = keys, contraction = Di.  One wave owns one query:
// its Hi x Di index-query block stays in registers as the A operand of v_mfma_f32_32x32x16_bf16
// (32 heads per tile), key rows stream through LDS in 64-key tiles shared by the four waves of the
// workgroup.  The epilogue applies ReLU and the per-head weight to the fp32 tiles in registers and
// reduces over heads (in-lane, then one cross-lane add), so only one fp32 per (query,key) pair reaches
// HBM.  Key tiles outside the query's own segment or above its diagonal are skipped per wave; queries
// whose causal window is not longer than top-k are skipped altogether.
//
// What bounds it is the matrix cores and the power they draw: on operands of this kind a register-only
// loop of these MFMAs sustains 1.83 PFLOP/s, on zeros 2.46 (the clock follows the power).  Hence as little
// besides the MFMAs as possible: keys go from memory straight into LDS, no vector address arithmetic in the
// loop.  32 768 tokens in eight segments, 64 x 128 indexer: 1040 -> 851 us (1.28 PFLOP/s); with zeros for
// queries 681; the same loop without its sums 782, without its LDS reads 797, without the key loads 798.
// (The 16x16x32 MFMA, which sustains 2.07 PFLOP/s in registers, was no faster here: 864 us.)
#include "dsa_common.h"

__device__ __forceinline__ f32x16 zero_acc() {
    f32x16 z;
#pragma unroll
    for (int v = 0; v < 16; ++v) z[v] = 0.f;
    return z;
}

#define IDX_WAVES 4
#define IDX_BK 64
#define IDX_BUFS 4

// The loop is pipelined inside each wave, sub-tile (32 keys) by sub-tile: behind every MFMA of sub-tile i stand the ReLU,
// weight and sum of 16 / KS elements of sub-tile i-1 (two vector instructions each), and the key operands an MFMA group has
// just consumed are re-read for sub-tile i+1, so that no MFMA waits for LDS and the vector work hides in the MFMAs' shadow
// (every MFMA step ends in an empty asm statement its results pass through, which fixes that order; left to itself the
// scheduler sinks every read next to its use).  Tile it+3 is requested at the start of step it (buffer_load ... lds: no
// registers, no LDS write instructions) and waited for in the middle of step it+1, in front of that step's score stores, so
// that one exact vmcnt covers it whether or not a wave stores; the barrier at the end of step it+1 publishes it, and its
// first operands are read in the second half of step it+2.
template <int HT, int DI>
__global__ __launch_bounds__(IDX_WAVES * 64, 2) void dsa_indexer_scores_kernel(
    const bf16_t *__restrict__ q_idx, const bf16_t *__restrict__ k_idx, const bf16_t *__restrict__ w_idx,
    const int32_t *__restrict__ cu, int N, int Hi, float scale, int row_begin, int row_end, int skip_dense_k,
    float *__restrict__ scores, int64_t ld) {
    constexpr int KS = DI / 16;                 // MFMA k-steps
    constexpr int ROW_B = DI * 2, CPR = DI / 8; // bytes and 16-byte chunks per key row
    constexpr int TILE_B = IDX_BK * ROW_B;
    constexpr int LOADS = TILE_B / (IDX_WAVES * 1024);   // 1 KiB per wave and load
    constexpr int NM = HT * KS, EL = 16 * HT / NM;       // MFMAs per sub-tile; elements of the one before behind each
    static_assert(LOADS >= 1 && LOADS * IDX_WAVES * 1024 == TILE_B, "tile must split evenly");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[IDX_BUFS][TILE_B];
    // the waves' ranges of keys: in the last buffer, which nothing is loaded into before the first barrier of the pipeline
    int *const range_lo = reinterpret_cast<int *>(&lds[IDX_BUFS - 1][0]), *const range_hi = range_lo + IDX_WAVES;

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, j = lane & 31, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // last rows first: the longest windows of a segment start first
    const int t = row_begin + (int)(gridDim.x - 1 - blockIdx.x) * IDX_WAVES + wv;
    bool active = t < row_end;
    int s0 = 0;
    if (active) {
        s0 = __builtin_amdgcn_readfirstlane(cu[find_segment_wave(cu, N, t)]);
        if (t - s0 + 1 <= skip_dense_k) active = false;
    }
    if (lane == 0) { range_lo[wv] = active ? s0 : 0x7fffffff; range_hi[wv] = active ? t : -1; }
    __syncthreads();
    int lo = range_lo[0], hi = range_hi[0];
#pragma unroll
    for (int i = 1; i < IDX_WAVES; ++i) { lo = min(lo, range_lo[i]); hi = max(hi, range_hi[i]); }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    if (hi < 0) return;                          // uniform: nothing to do in this workgroup

    const int kt0 = lo & ~(IDX_BK - 1);
    const int ntiles = (hi - kt0) / IDX_BK + 1;
    // Keys in LDS: unpadded rows (a load writes 1 KiB of consecutive LDS per wave), chunk c of row r at position
    // c ^ swizzle(r), so that the sixteen rows of an operand read fall on sixteen different 16-byte columns of the banks;
    // the swizzle is applied to the source address.  A tile's buffer starts at its first key and ends behind the last key any of
    // the workgroup's queries sees: rows past that, and tiles past the last one, read as zero without touching memory.
    auto swizzle = [](int row) { return DI == 128 ? (row & 15) : DI == 64 ? ((row >> 1) & 7) : ((row >> 2) & 3); };
    const int src_row = tid / CPR;               // (every later load of a tile starts a multiple of 16 rows further)
    const int voff = src_row * ROW_B + (((tid % CPR) ^ swizzle(src_row)) << 4);
    const uint32_t lds0 = lds_address(&lds[0][0]) + wv * 1024;
    const unsigned char *kptr = reinterpret_cast<const unsigned char *>(k_idx + (int64_t)kt0 * DI);
    int rows_left = hi + 1 - kt0;
    auto load_tile = [&](int buf) __attribute__((always_inline)) {   // the next tile, into the buffer at byte offset buf
        const buffer_rsrc keys = make_buffer_rsrc(kptr, max(min(rows_left, IDX_BK), 0) * ROW_B);
#pragma unroll
        for (int r = 0; r < LOADS; ++r) buffer_load_lds16(keys, voff + r * (IDX_WAVES * 1024), lds0 + buf + r * (IDX_WAVES * 1024));
        kptr += TILE_B;
        rows_left -= IDX_BK;
        asm volatile("" : "+s"(kptr), "+s"(rows_left));
    };
    load_tile(0);
    load_tile(TILE_B);
    load_tile(2 * TILE_B);
    // A operand: this wave's query, heads 32*ht + lane%32, k = 16*ks + 8*(lane/32) + e
    bf16x8 a[HT][KS];
    float wreg[HT][16];
    const int tq = active ? t : row_begin;
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
        const bf16_t *qrow = q_idx + ((int64_t)tq * Hi + min(ht * 32 + j, Hi - 1)) * DI + h * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a[ht][ks] = load_bf16x8(qrow + ks * 16);
#pragma unroll
        for (int v = 0; v < 16; ++v) {           // heads past Hi repeat the last one and weigh nothing
            const int hrow = ht * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
            const float w = (float)w_idx[(int64_t)tq * Hi + min(hrow, Hi - 1)];
            wreg[ht][v] = hrow < Hi ? w : 0.f;
        }
    }
    wait_vmcnt<0>();
    barrier_only();

    float *orow = scores + (int64_t)(tq - row_begin) * ld - s0;
    // this wave's own tiles of the walk, and the columns it stores
    const int my_last = active ? min(t, (int)min((int64_t)s0 + ld - 1, (int64_t)0x7fffffff)) : -1;   // ld bounds the row whatever the caller's max_seqlen
    const int it_lo = (s0 - kt0) / IDX_BK, it_hi = active ? (t - kt0) / IDX_BK : -1;
    int lane_b[KS];                              // operand address of key lane%32 of a sub-tile, k-step ks
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) lane_b[ks] = j * ROW_B + (((ks * 2 + h) ^ swizzle(j)) << 4);
    bf16x8 b[KS];
    f32x16 acc[2][HT];                           // [sub-tile parity][head tile]
    float sum = 0.f;
    auto read_b = [&](int buf, int sub, int ks) __attribute__((always_inline)) {
        b[ks] = *reinterpret_cast<const bf16x8 *>(&lds[0][buf + lane_b[ks] + sub * 32 * ROW_B]);
    };
    auto element = [&](const f32x16 (&p)[HT], int el) __attribute__((always_inline)) {
        // ReLU as one integer max on the bit pattern: negative floats are negative integers (fmaxf would cost a second
        // instruction to quiet NaNs)
        sum = fmaf(wreg[el >> 4][el & 15], __int_as_float(max(__float_as_int(p[el >> 4][el & 15]), 0)), sum);
    };
    // store the finished sums of the sub-tile of keys kb .. kb + 31
    auto finish = [&](int kb) __attribute__((always_inline)) {
        const float total = half_sum_f(sum) * scale;
        const int s = kb + j;
        if (h == 0 && s >= s0 && s <= my_last) orow[s] = total;
        sum = 0.f;
    };
    // MFMAs of the sub-tile whose operands are in b, with the elements of `prev` behind them and the operands of the next
    // sub-tile (nbuf, nsub) read as they fall free
    auto substep = [&](f32x16 (&cur)[HT], const f32x16 (&prev)[HT], int nbuf, int nsub) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int ks = m / HT, ht = m % HT;
            cur[ht] = mfma32(a[ht][ks], b[ks], ks == 0 ? zero_acc() : cur[ht]);
            if (ht == HT - 1) read_b(nbuf, nsub, ks);
#pragma unroll
            for (int e = 0; e < EL; ++e) element(prev, m * EL + e);
            asm volatile("" : "+v"(sum) : : "memory");
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // byte offsets of the buffers of tiles it .. it+3, taking turns (opaque, so that no address becomes an induction
    // variable of its own)
    int cb = 0, nb = TILE_B, n2 = 2 * TILE_B, sb = 3 * TILE_B;
    for (int it = 0; it < ntiles; ++it) {
        load_tile(sb);                           // tile it+3; its buffer was last read before the previous barrier
        const bool mine = it >= it_lo && it <= it_hi;    // wave-uniform
        const int kt = kt0 + it * IDX_BK;
        if (mine) {
            if (it == it_lo) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) read_b(cb, 0, ks);
#pragma unroll
                for (int ht = 0; ht < HT; ++ht) acc[1][ht] = zero_acc();
            }
            substep(acc[0], acc[1], cb, 1);
        }
        wait_vmcnt<LOADS>();                     // everything but the tile just requested
        if (mine) {
            if (it != it_lo) finish(kt - 32);
            sum = 0.f;
            substep(acc[1], acc[0], nb, 0);
            finish(kt);
            if (it == it_hi) {
#pragma unroll
                for (int el = 0; el < 16 * HT; ++el) element(acc[1], el);
                finish(kt + 32);
            }
        }
        barrier_only();
        const int ob = cb;
        cb = nb; nb = n2; n2 = sb; sb = ob;
        asm volatile("" : "+s"(cb), "+s"(nb), "+s"(n2), "+s"(sb));
    }
    wait_vmcnt<0>();                             // no load is left on its way into LDS when the workgroup ends
}

template <int HT, int DI>
static hipError_t launch_indexer(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int N,
                                 int Hi, float scale, int row_begin, int row_end, int skip_dense_k,
                                 float *scores, int64_t ld, hipStream_t stream) {
    const int rows = row_end - row_begin;
    const int grid = (rows + IDX_WAVES - 1) / IDX_WAVES;
    hipLaunchKernelGGL((dsa_indexer_scores_kernel<HT, DI>), dim3(grid), dim3(IDX_WAVES * 64), 0, stream,
                       (const bf16_t *)q_idx, (const bf16_t *)k_idx, (const bf16_t *)w_idx, cu, N, Hi, scale,
                       row_begin, row_end, skip_dense_k, scores, ld);
    return hipGetLastError();
}

// returns hipErrorInvalidValue for geometries the kernel does not cover
extern "C" hipError_t dsa_launch_indexer(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu,
                                         int N, int Hi, int Di, float scale, int row_begin, int row_end,
                                         int skip_dense_k, float *scores, int64_t ld, hipStream_t stream) {
    if (row_end <= row_begin) return hipSuccess;
    const int HT = (Hi + 31) / 32;
#define IDX_CASE(ht, di) \
    if (HT == ht && Di == di) \
        return launch_indexer<ht, di>(q_idx, k_idx, w_idx, cu, N, Hi, scale, row_begin, row_end, skip_dense_k, scores, ld, stream);
    IDX_CASE(1, 32) IDX_CASE(1, 64) IDX_CASE(1, 128)
    IDX_CASE(2, 32) IDX_CASE(2, 64) IDX_CASE(2, 128)
#undef IDX_CASE
    return hipErrorInvalidValue;
}
