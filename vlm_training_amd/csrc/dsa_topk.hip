// Stage D2: per-query top-k over one row of fp32 scores, total order (score descending, column
// ascending).  One 256-thread workgroup per query row.
//
//   1. rows with pos+1 <= K are the whole causal window: write the range, done;
//   2. MSB-first radix select (3 passes of 11, 11 and 10 bits) over order-preserving uint32 keys finds the
//      K-th largest key tau and how many keys equal to tau are still wanted (need_eq); the first histogram
//      is filled while the row is read;
//   3. an index-ordered compaction keeps key > tau, plus the first need_eq keys == tau.  The row is
//      split into four contiguous quarters (one per wave); per-quarter counts give every wave its
//      output offset, so the result comes out ascending and deterministic without sorting.
//
// Rows up to TOPK_LDS_CAP keys are read from HBM once and kept in LDS as keys.  Longer ones are swept once, by dsa_topk_long_kernel below,
// or, where that does not hold them, five times.
// With a sel_out pointer the kernel also writes the scores of the selected keys beside their indices (the key it ranks
// by is the score, bit for bit, but for the sign of a zero).
//
// With a bitmap pointer the kernel also leaves the row's inverted selection (bit c of the row's ldw words = "key column c
// of the segment is selected", what dsa_bitmap_kernel builds from the finished list): the compaction's ballots are those
// words already, so the list need not be read back.
#include "dsa_common.h"
#include <algorithm>

#define TOPK_THREADS 256
#define TOPK_LDS_CAP 8192
#define TOPK_BINS 2048                                  // 11-bit digits (the last pass uses 1024 of them)
#define TOPK_CAND 256                                   // see topk_tau
#define TOPK_LIST 6144                                  // most scores of a long row that are held
#define TOPK_LONG_MAX 131072                            // longest row swept once (a bit per column in LDS, whatever the launch's bound), and most keys selected of it
#define TOPK_LONG_K 4096

// the score a key stands for (-0.0 comes back as +0.0: score_key folds the two)
__device__ __forceinline__ float key_score(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ uint32_t score_key(float x) {
    uint32_t u = __float_as_uint(x);
    if (u == 0x80000000u) u = 0u;                       // -0.0 ties with +0.0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // larger float <=> larger key
}
struct TopkShared {
    __attribute__((aligned(16))) uint32_t hist[TOPK_BINS];
    uint32_t wave_tot[4], cnt_gt[4], cnt_eq[4];
    uint32_t sel_digit, sel_remaining, sel_count;
};
// where a row's results go (orow null: into the bitmap alone)
struct TopkRow { const float *row; int32_t *orow; float *srow; uint32_t *brow; int nvalid, s0, K, ldw; };

// The bin of `hist` in which the `remaining`-th largest count lies (largest bins first), what of it is still wanted and how many counts
// it has: sel_digit, sel_remaining, sel_count.  `per` consecutive bins per thread.  hist is complete behind a barrier.
__device__ __forceinline__ void topk_find_bin(TopkShared &sh, int per, uint32_t remaining) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t own[8], h = 0u;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        own[b] = b < per ? sh.hist[per * tid + b] : 0u;
        h += own[b];
    }
    uint32_t v = h;                                     // inclusive suffix sum over threads
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_down(v, off, 64);
        if (lane + off < 64) v += u;
    }
    if (lane == 0) sh.wave_tot[wv] = v;
    __syncthreads();
    for (int w2 = wv + 1; w2 < 4; ++w2) v += sh.wave_tot[w2];
    uint32_t above = v - h;                             // counts beyond this thread's bins
    if (above < remaining && remaining <= v) {          // exactly one thread satisfies this; walk its bins from the top
#pragma unroll
        for (int b = 7; b >= 0; --b) {
            if (b < per && above < remaining) {
                if (remaining <= above + own[b]) {
                    sh.sel_digit = (uint32_t)(per * tid + b);
                    sh.sel_remaining = remaining - above;
                    sh.sel_count = own[b];
                }
                above += own[b];
            }
        }
    }
    __syncthreads();
}

// Index-ordered compaction of 64 columns of a wave: the keys beyond tau and the first need_eq equal ones.  column: that of lane 0
__device__ __forceinline__ void topk_compact(const TopkRow &r, int column, bool is_gt, bool is_eq, float score, uint32_t need_eq,
                                             uint32_t &out_pos, uint32_t &eq_seen) {
    const int lane = threadIdx.x & 63;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint64_t b_eq = __ballot(is_eq);
    const uint32_t eq_rank = eq_seen + (uint32_t)__popcll(b_eq & lt_mask);
    const bool take = is_gt || (is_eq && eq_rank < need_eq);
    const uint64_t b_take = __ballot(take);
    // exactly K keys are taken when every score orders; NaN scores can break the count, hence the bound on the slot
    const uint32_t slot = out_pos + (uint32_t)__popcll(b_take & lt_mask);
    if (r.orow && take && slot < (uint32_t)r.K) {
        r.orow[slot] = r.s0 + column + lane;
        if (r.srow) r.srow[slot] = score;
    }
    if (r.brow && lane < 2) {                           // the ballot is the two bitmap words of these 64 columns
        const int w = (column >> 5) + lane;
        if (w < r.ldw) r.brow[w] = (uint32_t)(b_take >> (32 * lane));
    }
    out_pos += (uint32_t)__popcll(b_take);
    eq_seen += (uint32_t)__popcll(b_eq);
}
// the wave's first output slot and the equal keys before it, from every wave's counts in cnt_gt, cnt_eq (behind a barrier)
__device__ __forceinline__ void topk_wave_start(const TopkShared &sh, uint32_t need_eq, uint32_t &out_pos, uint32_t &eq_seen) {
    out_pos = eq_seen = 0u;
    for (int w2 = 0; w2 < (int)(threadIdx.x >> 6); ++w2) {
        out_pos += sh.cnt_gt[w2] + (need_eq > eq_seen ? min(need_eq - eq_seen, sh.cnt_eq[w2]) : 0u);
        eq_seen += sh.cnt_eq[w2];
    }
}

// The bitmap words of a wave's columns [c_begin, c_end) of a row, c_begin a multiple of 64: take(i) says whether column i is selected, asked in
// column order.  A lane keeps every 64th ballot, so that words leave 64 columns per lane in one store.
// A selection whose list nobody reads ends here: no pass that counts what is taken of each quarter, no slots, no (row, K) integers in memory.  The
// whole step with the list -> without, us: 8 192 tokens, K = 512: 305.5 -> 300.2; forward of 16 384, K = 2048: 695.6 -> 673.4; 32 768: 6586 -> 6526.
template <class Take>
__device__ __forceinline__ void topk_words(const TopkRow &r, int c_begin, int c_end, Take take) {
    const int lane = threadIdx.x & 63;
    for (int base = c_begin; base < c_end; base += 64 * 64) {
        uint64_t mine = 0ull;
#pragma unroll 4
        for (int u = 0; u < 64; ++u) {
            const int column = base + u * 64;
            if (column >= c_end) break;                 // wave-uniform
            const uint64_t b = __ballot(take(column + lane));
            if (u == lane) mine = b;
        }
        const int w = (base >> 5) + 2 * lane;
        if (base + 64 * lane < c_end) {
            if (w + 1 < r.ldw && !(reinterpret_cast<uintptr_t>(r.brow) & 7)) *reinterpret_cast<uint64_t *>(r.brow + w) = mine;
            else {
                if (w < r.ldw) r.brow[w] = (uint32_t)mine;
                if (w + 1 < r.ldw) r.brow[w + 1] = (uint32_t)(mine >> 32);
            }
        }
    }
}

// Radix select of a row; any scores.  key_at(i): key of column i; counted: the first histogram is there (in front of a barrier)
template <class KeyAt>
__device__ __forceinline__ void topk_radix(TopkShared &sh, const TopkRow &r, bool counted, KeyAt key_at) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int nvalid = r.nvalid;
    uint32_t prefix = 0u, pmask = 0u, remaining = (uint32_t)r.K;
    for (int pass = 0; pass < 3; ++pass) {
        const int shift = pass == 0 ? 21 : (pass == 1 ? 10 : 0);
        const uint32_t dmask = pass == 2 ? 1023u : 2047u;
        if (pass > 0 || !counted) {
            __syncthreads();
            for (int i = tid; i < TOPK_BINS; i += TOPK_THREADS) sh.hist[i] = 0u;
            __syncthreads();
            // eight keys per thread in flight (rows that are not cached come from memory on every sweep)
            for (int base = tid; base < nvalid; base += 8 * TOPK_THREADS) {
                uint32_t kk[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) kk[u] = key_at(min(base + u * TOPK_THREADS, nvalid - 1));
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (base + u * TOPK_THREADS < nvalid && (kk[u] & pmask) == prefix) atomicAdd(&sh.hist[(kk[u] >> shift) & dmask], 1u);
            }
        }
        __syncthreads();
        topk_find_bin(sh, pass == 2 ? 4 : 8, remaining);
        prefix |= sh.sel_digit << shift;
        pmask |= dmask << shift;
        remaining = sh.sel_remaining;
    }
    const uint32_t tau = prefix, need_eq = remaining, n_eq = sh.sel_count;
    const bool words_only = r.orow == nullptr && n_eq == need_eq;         // every key equal to tau is taken: nothing to rank
    __syncthreads();

    // contiguous quarter of the row per wave, multiple of 64 columns
    const int per = (((nvalid + 3) >> 2) + 63) & ~63;
    const int c_begin = min(wv * per, nvalid), c_end = min(c_begin + per, nvalid);
    if (words_only) {
        topk_words(r, c_begin, c_end, [&](int i) { return i < c_end && key_at(min(i, nvalid - 1)) >= tau; });
        for (int w = 2 * ((nvalid + 63) >> 6) + tid; w < r.ldw; w += TOPK_THREADS) r.brow[w] = 0u;
        return;
    }
    uint32_t g = 0, e = 0;
    for (int base = c_begin + lane; base < c_end; base += 8 * 64) {
        uint32_t kk[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) kk[u] = key_at(min(base + u * 64, nvalid - 1));
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (base + u * 64 < c_end) {
                g += kk[u] > tau;
                e += kk[u] == tau;
            }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        g += __shfl_xor(g, off, 64);
        e += __shfl_xor(e, off, 64);
    }
    if (lane == 0) { sh.cnt_gt[wv] = g; sh.cnt_eq[wv] = e; }
    __syncthreads();
    uint32_t eq_seen, out_pos;
    topk_wave_start(sh, need_eq, out_pos, eq_seen);
    for (int base = c_begin; base < c_end; base += 4 * 64) {
        uint32_t kk[4];                                 // four chunks of 64 columns fetched, then ranked in index order
#pragma unroll
        for (int u = 0; u < 4; ++u) kk[u] = key_at(min(base + u * 64 + lane, nvalid - 1));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = base + u * 64 + lane;
            if (base + u * 64 >= c_end) break;          // wave-uniform
            topk_compact(r, base + u * 64, i < c_end && kk[u] > tau, i < c_end && kk[u] == tau, key_score(kk[u]), need_eq, out_pos, eq_seen);
        }
    }
    if (r.brow)                                         // the words behind the window: the quarters end on 64 columns
        for (int w = 2 * ((nvalid + 63) >> 6) + tid; w < r.ldw; w += TOPK_THREADS) r.brow[w] = 0u;
}

// the row of a workgroup; false: nothing is left to do for it (only rows of min_row to max_row columns are looked at: a launch whose
// bound on the longest row exceeds what a kernel holds is split, as the bound may be far above the real longest row - max_seqlen = the
// packed length when the caller holds no better one)
__device__ __forceinline__ bool topk_row(const float *scores, int64_t ld, int row_begin, const int32_t *cu, int N, int K, int min_row,
                                         int max_row, int32_t *idx_out, int32_t *n_out, uint32_t *bitmap, int ldw, float *sel_out,
                                         TopkRow &r) {
    const int tid = threadIdx.x, t = row_begin + blockIdx.x;
    const int s0 = cu[find_segment_wave(cu, N, t)];
    // a row never reaches past its ld columns: with a max_seqlen below the longest segment (a caller's mistake) the
    // selection of the long rows is wrong, but nothing outside the score rows is read
    const int nvalid = (int)min((int64_t)(t - s0 + 1), ld);
    if (nvalid < min_row || nvalid > max_row) return false;
    r = TopkRow{scores + (int64_t)(t - row_begin) * ld, idx_out ? idx_out + (int64_t)t * K : nullptr, sel_out ? sel_out + (int64_t)t * K : nullptr,
                bitmap ? bitmap + (int64_t)t * ldw : nullptr, nvalid, s0, K, ldw};
    if (n_out && tid == 0) n_out[t] = min(nvalid, K);
    if (nvalid > K) return true;
    if (r.orow)
        for (int i = tid; i < K; i += TOPK_THREADS) r.orow[i] = (i < nvalid) ? (s0 + i) : -1;
    if (r.srow)                                         // the scores of the selected keys, slot by slot (0 past n)
        for (int i = tid; i < K; i += TOPK_THREADS) r.srow[i] = (i < nvalid) ? r.row[i] : 0.f;
    if (r.brow)
        for (int w = tid; w < ldw; w += TOPK_THREADS) {
            const int left = nvalid - 32 * w;           // columns of this word inside the window
            r.brow[w] = left >= 32 ? ~0u : (left > 0 ? (1u << left) - 1u : 0u);
        }
    return false;
}

template <bool CACHED>
__global__ __launch_bounds__(TOPK_THREADS) void dsa_topk_rows_kernel(
    const float *__restrict__ scores, int64_t ld, int row_begin, const int32_t *__restrict__ cu, int N, int K, int min_row, int max_row,
    int32_t *__restrict__ idx_out, int32_t *__restrict__ n_out, uint32_t *__restrict__ bitmap, int ldw, float *__restrict__ sel_out) {
    __shared__ TopkShared sh;
    extern __shared__ __attribute__((aligned(16))) uint32_t keys_lds[];   // CACHED: the launch's longest row (max_row); the fewer bytes, the more rows per CU
    TopkRow r;
    if (!topk_row(scores, ld, row_begin, cu, N, K, min_row, max_row, idx_out, n_out, bitmap, ldw, sel_out, r)) return;
    if (!CACHED) return topk_radix(sh, r, false, [&](int i) -> uint32_t { return score_key(r.row[i]); });
    const int tid = threadIdx.x;
    for (int i = tid; i < TOPK_BINS; i += TOPK_THREADS) sh.hist[i] = 0u;
    __syncthreads();
    // 16-byte loads, four per thread in flight: one load per loop iteration would pay the memory latency
    // nvalid / 256 times over
    const float4 *row4 = reinterpret_cast<const float4 *>(r.row);
    const int n4 = (reinterpret_cast<uintptr_t>(r.row) & 15) ? 0 : r.nvalid >> 2;   // a caller's own rows may not be aligned
    for (int base = 0; base < n4; base += 4 * TOPK_THREADS) {
        float4 x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i4 = base + u * TOPK_THREADS + tid;
            x[u] = row4[min(i4, n4 - 1)];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i4 = base + u * TOPK_THREADS + tid;
            if (i4 < n4) {
                const uint4 kk = {score_key(x[u].x), score_key(x[u].y), score_key(x[u].z), score_key(x[u].w)};
                *reinterpret_cast<uint4 *>(&keys_lds[4 * i4]) = kk;
                atomicAdd(&sh.hist[kk.x >> 21], 1u);    // first digit: the top 11 bits
                atomicAdd(&sh.hist[kk.y >> 21], 1u);
                atomicAdd(&sh.hist[kk.z >> 21], 1u);
                atomicAdd(&sh.hist[kk.w >> 21], 1u);
            }
        }
    }
    for (int i = (n4 << 2) + tid; i < r.nvalid; i += TOPK_THREADS) {
        const uint32_t key = score_key(r.row[i]);
        keys_lds[i] = key;
        atomicAdd(&sh.hist[key >> 21], 1u);
    }
    topk_radix(sh, r, true, [&](int i) -> uint32_t { return keys_lds[i]; });
}

// ---- long rows ----
struct TopkLong {
    TopkShared sh;
    uint32_t ncand, need_eq, odd[4], some_odd, nlist;
    float tau, lo[4], hi[4], cand_x[TOPK_CAND];
    int cand_i[TOPK_CAND];
};
// A score's bin never falls as the score rises: 2048 bins of equal width between the smallest and the largest score are counted, the one
// that holds the K-th largest found, its few scores ranked exactly against each other.  A crowded bin (more than TOPK_CAND scores) is
// counted again by itself, from its smallest to its largest score, until it is not.
// tau = the K-th largest of the scores x[u] with in(u), need_eq = how many scores equal to it are among the K largest.  index(u): the
// score's column; any(u): whether a lane of the wave has a u-th score (wave-uniform).  False: some score is not finite (or the spread
// overflows).  Every thread gets the answer; called by the whole workgroup.
template <int R, class Any, class In, class Index>
__device__ __forceinline__ bool topk_tau(TopkLong &m, float (&x)[R], Any any, In in, Index index, uint32_t remaining, float &tau,
                                         uint32_t &need_eq) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    auto again = [&]() {                                // (a score's bin and its tests are formed again: kept, they cost more registers than the scores)
#pragma unroll
        for (int u = 0; u < R; ++u) asm volatile("" : "+v"(x[u]));
    };
    float mn = INFINITY, mx = -INFINITY, finite = 0.f;  // (a sum of zeros, unless a score is infinite or not a number)
#pragma unroll
    for (int u = 0; u < R; ++u)
        if (any(u) && in(u)) {
            mn = fminf(mn, x[u]);
            mx = fmaxf(mx, x[u]);
            finite = fmaf(x[u], 0.f, finite);
        }
    for (bool first = true;; first = false) {
        again();
#pragma unroll
        for (int i = 0; i < TOPK_BINS / TOPK_THREADS; ++i) m.sh.hist[i * TOPK_THREADS + tid] = 0u;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, off, 64));
            mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        }
        const uint64_t odd = __ballot(!(finite == 0.f));
        if (lane == 0) {
            m.lo[wv] = mn;
            m.hi[wv] = mx;
            m.odd[wv] = odd != 0ull;
        }
        if (tid == 0) m.ncand = 0u;
        __syncthreads();
        // the scores that are still in question: from lo to hi
        const float lo = fminf(fminf(m.lo[0], m.lo[1]), fminf(m.lo[2], m.lo[3]));
        const float hi = fmaxf(fmaxf(m.hi[0], m.hi[1]), fmaxf(m.hi[2], m.hi[3]));
        if (first && (m.odd[0] | m.odd[1] | m.odd[2] | m.odd[3])) return false;
        if (lo == hi) {
            tau = lo;
            need_eq = remaining;
            return true;
        }
        const float bins = (float)(TOPK_BINS - 1) / (hi - lo);
        if (!(bins > 0.f && bins <= 3.402823466e38f)) return false;
        auto bin = [&](float v) -> uint32_t { return (uint32_t)fminf((v - lo) * bins, (float)(TOPK_BINS - 1)); };
#pragma unroll
        for (int u = 0; u < R; ++u)
            if (any(u) && in(u) && x[u] >= lo && x[u] <= hi) atomicAdd(&m.sh.hist[bin(x[u])], 1u);
        __syncthreads();
        topk_find_bin(m.sh, TOPK_BINS / TOPK_THREADS, remaining);
        again();
        const uint32_t mid = m.sh.sel_digit, c = m.sh.sel_count;
        remaining = m.sh.sel_remaining;
        if (c <= TOPK_CAND) {
#pragma unroll
            for (int u = 0; u < R; ++u)
                if (any(u) && in(u) && x[u] >= lo && x[u] <= hi && bin(x[u]) == mid) {
                    const uint32_t slot = atomicAdd(&m.ncand, 1u);
                    m.cand_x[slot] = x[u];
                    m.cand_i[slot] = index(u);
                }
            __syncthreads();
            if (tid < (int)c) {
                const float xi = m.cand_x[tid];
                const int ii = m.cand_i[tid];
                uint32_t above = 0u, before = 0u;       // larger ones; equal ones of lower columns
                for (int j = 0; j < (int)c; ++j) {
                    above += m.cand_x[j] > xi;
                    before += m.cand_x[j] == xi && m.cand_i[j] < ii;
                }
                if (above + before + 1u == remaining) {
                    m.tau = xi;
                    m.need_eq = remaining - above;
                }
            }
            __syncthreads();
            again();
            tau = m.tau;
            need_eq = m.need_eq;
            return true;
        }
        mn = INFINITY;
        mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < R; ++u)
            if (any(u) && in(u) && x[u] >= lo && x[u] <= hi && bin(x[u]) == mid) {
                mn = fminf(mn, x[u]);
                mx = fmaxf(mx, x[u]);
            }
    }
}

__device__ __noinline__ void topk_radix_memory(TopkShared &sh, const TopkRow &r) {
    topk_radix(sh, r, false, [&](int i) -> uint32_t { return score_key(r.row[i]); });
}
// words of a row's bit per column, as many for every thread
__host__ __device__ inline int topk_long_words(int columns) { return (columns + 32 * TOPK_THREADS - 1) / (32 * TOPK_THREADS) * TOPK_THREADS; }
// Rows of min_row to TOPK_LONG_MAX scores, one sweep over memory: the scores from a threshold on that a sample of 4096 puts at about 1.75 K of them
// go into a list in LDS, as many as `cap` (another sweep, the threshold moved, when fewer than K or more than cap passed); tau and
// need_eq come from the list, the selected columns are marked in a bit each and the bits compacted.  What does not fit - scores that are
// not finite, two moved thresholds that did not help, hundreds of scores equal to tau - takes the radix select.
//
// What bounds it: memory, and a fixed 20 us a row around the sweep (the sample's scattered reads, two selections of seven barriers), three
// workgroups a CU.  Same box, us, against five sweeps of the radix select, rows at the end of one segment: 2048 rows of 20 480 columns
// 140 -> 94, 32 768: 225 -> 110, 65 536: 506 -> 203, 131 072: 1020 -> 322, and under a bound of 131 104
// 20 480: 141 -> 120, 65 536: 514 -> 204; all 16 384 rows of one segment 438 -> 407, all 12 288: level.
// Held in registers and selected this way, rows of up to 8192 scores took 309 us where the radix select over LDS takes 261 (32 768 tokens).
__global__ __launch_bounds__(TOPK_THREADS, 3) void dsa_topk_long_kernel(
    const float *__restrict__ scores, int64_t ld, int row_begin, const int32_t *__restrict__ cu, int N, int K, int min_row, int cap,
    int32_t *__restrict__ idx_out, int32_t *__restrict__ n_out, uint32_t *__restrict__ bitmap, int ldw, float *__restrict__ sel_out) {
    extern __shared__ __attribute__((aligned(16))) unsigned char long_lds[];     // TopkLong | cap scores | their columns | a bit per column
    TopkLong &m = *reinterpret_cast<TopkLong *>(long_lds);
    float *const list_x = reinterpret_cast<float *>(long_lds + sizeof(TopkLong));
    int *const list_i = reinterpret_cast<int *>(list_x + cap);
    uint32_t *const words = reinterpret_cast<uint32_t *>(list_i + cap);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    TopkRow r;
    if (!topk_row(scores, ld, row_begin, cu, N, K, min_row, TOPK_LONG_MAX, idx_out, n_out, bitmap, ldw, sel_out, r)) return;
    const int nvalid = r.nvalid, nwords = topk_long_words(nvalid);

    // a sample: 256 runs of 16 columns over the row
    constexpr int SR = 16;
    float s[SR];
#pragma unroll
    for (int u = 0; u < SR; ++u) s[u] = r.row[(int64_t)(u * 16 + (tid >> 4)) * (nvalid - 16) / 255 + (tid & 15)];
    auto all = [](int) { return true; };
    int rank = (int)((int64_t)min(K + K / 2 + 512, (K + cap) / 2) * (SR * TOPK_THREADS) / nvalid);
    uint32_t n = 0u;
    for (int attempt = 0;; ++attempt) {
        if (attempt == 3) return topk_radix_memory(m.sh, r);
        float from;
        uint32_t unused;
        if (!topk_tau<SR>(m, s, all, all, [&](int u) { return u * TOPK_THREADS + tid; }, (uint32_t)max(rank, 1), from, unused)) return topk_radix_memory(m.sh, r);
        __syncthreads();
        if (tid == 0) { m.nlist = 0u; m.some_odd = 0u; }
        __syncthreads();
        // one sweep: eight 16-byte loads per thread in flight, one place in the list asked for per wave and sweep of 8192 columns
        const float4 *row4 = reinterpret_cast<const float4 *>(r.row);
        const int n4 = (nvalid + 3) >> 2;               // (the last one is read by elements: a row ends where its columns do)
        float finite = 0.f;
        for (int base = 0; base < n4; base += 8 * TOPK_THREADS) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = row4[min(base + u * TOPK_THREADS + tid, (nvalid >> 2) - 1)];
            if ((nvalid & 3) && base + 8 * TOPK_THREADS >= n4)
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (base + u * TOPK_THREADS + tid == n4 - 1) {
                        const float *p = r.row + 4 * (n4 - 1);
                        v[u] = make_float4(p[0], (nvalid & 3) > 1 ? p[1] : p[0], (nvalid & 3) > 2 ? p[2] : p[0], p[0]);
                    }
            uint32_t mine = 0u, total = 0u;             // bit 4 u + c: element c of load u passes
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int col = 4 * (base + u * TOPK_THREADS + tid);
                const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    finite = fmaf(e[c], 0.f, finite);
                    const bool pass = e[c] >= from && col + c < nvalid;
                    mine |= (uint32_t)pass << (4 * u + c);
                    total += (uint32_t)__popcll(__ballot(pass));
                }
            }
            uint32_t before = (uint32_t)__popc(mine);   // exclusive prefix sum over the lanes
            const uint32_t own = before;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t o = __shfl_up(before, off, 64);
                if (lane >= off) before += o;
            }
            uint32_t place = 0u;
            if (lane == 0) place = atomicAdd(&m.nlist, total);
            place = (uint32_t)__builtin_amdgcn_readfirstlane((int)place) + before - own;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if ((mine >> (4 * u + c)) & 1u) {
                        if (place < (uint32_t)cap) {
                            list_x[place] = e[c];
                            list_i[place] = 4 * (base + u * TOPK_THREADS + tid) + c;
                        }
                        ++place;
                    }
            }
        }
        if (!(finite == 0.f)) m.some_odd = 1u;
        __syncthreads();
        n = m.nlist;
        if (m.some_odd) return topk_radix_memory(m.sh, r);
        if (n >= (uint32_t)K && n <= (uint32_t)cap) break;
        rank = n < (uint32_t)K ? min(2 * rank + 8, SR * TOPK_THREADS) : rank * 5 / 8;
        __syncthreads();
    }
    constexpr int R = TOPK_LIST / TOPK_THREADS;
    float x[R];
    auto any = [&](int u) { return u * TOPK_THREADS < (int)n; };
    auto in = [&](int u) { return u * TOPK_THREADS + tid < (int)n; };
#pragma unroll
    for (int u = 0; u < R; ++u)
        if (any(u)) x[u] = list_x[u * TOPK_THREADS + tid];
    for (int w = tid; w < nwords; w += TOPK_THREADS) words[w] = 0u;
    float tau;
    uint32_t need_eq;
    if (!topk_tau<R>(m, x, any, in, [&](int u) { return list_i[u * TOPK_THREADS + tid]; }, (uint32_t)K, tau, need_eq)) return topk_radix_memory(m.sh, r);
    __syncthreads();
    if (tid == 0) m.ncand = 0u;
    __syncthreads();
    // the keys beyond tau, and the equal ones: all of them, or the need_eq lowest columns
#pragma unroll
    for (int u = 0; u < R; ++u)
        if (any(u) && in(u) && x[u] >= tau) {
            const int col = list_i[u * TOPK_THREADS + tid];
            if (x[u] > tau) atomicOr(&words[col >> 5], 1u << (col & 31));
            else {
                const uint32_t slot = atomicAdd(&m.ncand, 1u);
                if (slot < TOPK_CAND) m.cand_i[slot] = col;
            }
        }
    __syncthreads();
    const uint32_t n_eq = m.ncand;
    if (n_eq > TOPK_CAND) return topk_radix_memory(m.sh, r);
    if (tid < (int)n_eq) {
        const int col = m.cand_i[tid];
        uint32_t before = 0u;
        for (int j = 0; j < (int)n_eq; ++j) before += m.cand_i[j] < col;
        if (before < need_eq) atomicOr(&words[col >> 5], 1u << (col & 31));
    }
    __syncthreads();
    if (r.brow)
        for (int w = tid; w < ldw; w += TOPK_THREADS) r.brow[w] = w < nwords ? words[w] : 0u;
    if (!r.orow) return;
    // consecutive words per thread, in order
    const int per = nwords / TOPK_THREADS;
    uint32_t before = 0u;
    for (int w = 0; w < per; ++w) before += (uint32_t)__popc(words[tid * per + w]);
    const uint32_t own = before;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(before, off, 64);
        if (lane >= off) before += o;
    }
    if (lane == 63) m.sh.wave_tot[wv] = before;
    __syncthreads();
    uint32_t place = before - own;
    for (int w2 = 0; w2 < wv; ++w2) place += m.sh.wave_tot[w2];
    for (int w = 0; w < per; ++w)
        for (uint32_t b = words[tid * per + w]; b; b &= b - 1u) list_i[place++] = (tid * per + w) * 32 + __ffs(b) - 1;
    __syncthreads();
    for (int j = tid; j < K; j += TOPK_THREADS) {
        const int col = list_i[j];
        r.orow[j] = r.s0 + col;
        if (r.srow) r.srow[j] = r.row[col] + 0.f;
    }
}

extern "C" hipError_t dsa_launch_topk(const float *scores, int64_t ld, int row_begin, int row_end,
                                      const int32_t *cu, int N, int K, int32_t *idx, int32_t *n,
                                      uint32_t *bitmap, int ldw, float *sel, hipStream_t stream) {
    const int rows = row_end - row_begin;
    if (rows <= 0) return hipSuccess;
    const int all = 0x7fffffff;
    const int64_t longest = std::min<int64_t>(ld, all);  // (no row reaches past its ld columns)
    const int held = (int)std::min<int64_t>((longest + 3) & ~3, TOPK_LDS_CAP);
    hipLaunchKernelGGL(dsa_topk_rows_kernel<true>, dim3(rows), dim3(TOPK_THREADS), (size_t)held * 4, stream, scores, ld, row_begin, cu, N, K, 0, held,
                       idx, n, bitmap, ldw, sel);
    if (longest <= held) return hipGetLastError();
    int next = held + 1;                                 // rows of at least that many columns are left
    if (K <= TOPK_LONG_K && ld % 4 == 0 && (reinterpret_cast<uintptr_t>(scores) & 15) == 0) {
        const int cap = (std::min(std::max(2 * K + 512, 4096), TOPK_LIST) + TOPK_THREADS - 1) / TOPK_THREADS * TOPK_THREADS;
        const int most = (int)std::min<int64_t>(longest, TOPK_LONG_MAX);
        const size_t lds = sizeof(TopkLong) + (size_t)cap * 8 + (size_t)topk_long_words(most) * 4;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&dsa_topk_long_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(dsa_topk_long_kernel, dim3(rows), dim3(TOPK_THREADS), lds, stream, scores, ld, row_begin, cu, N, K, next, cap, idx, n,
                           bitmap, ldw, sel);
        if (longest == most) return hipGetLastError();
        next = TOPK_LONG_MAX + 1;
    }
    hipLaunchKernelGGL(dsa_topk_rows_kernel<false>, dim3(rows), dim3(TOPK_THREADS), 0, stream, scores, ld, row_begin, cu, N, K, next, all, idx, n,
                       bitmap, ldw, sel);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// The KL divergence of the indexer's distribution over the selected keys (their scores sel[t,j], 0 for j >= n[t], come
// out of the selection kernel's compaction) from a target distribution (the attention mass), with its gradient w.r.t.
// the scores.
// ------------------------------------------------------------------------------------------------

// block-wide reductions over 256 threads (4 waves)
__device__ __forceinline__ float block_max_256(float v, float *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
__device__ __forceinline__ float block_sum_256(float v, float *red) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}
// One workgroup per query row.  loss[t] = sum_j p_j (log p_j - log softmax(I)_j) over j < n[t] (terms with p_j = 0
// are 0), dscore[t,j] = (softmax(I)_j - p_j) * grad_scale, 0 for j >= n[t].
__global__ __launch_bounds__(256) void dsa_indexer_kl_kernel(const float *__restrict__ sel, const float *__restrict__ mass,
                                                              const int32_t *__restrict__ nsel, int K, float grad_scale,
                                                              float *__restrict__ loss, float *__restrict__ dscore) {
    __shared__ float red[4];
    const int t = blockIdx.x, nt = nsel[t];
    const float *irow = sel + (int64_t)t * K, *prow = mass + (int64_t)t * K;
    float m = -INFINITY;
    for (int j = threadIdx.x; j < nt; j += 256) m = fmaxf(m, irow[j]);
    m = block_max_256(m, red);
    float z = 0.f;
    for (int j = threadIdx.x; j < nt; j += 256) z += __expf(irow[j] - m);
    z = block_sum_256(z, red);
    const float lse = m + __logf(z);
    float acc = 0.f;
    for (int j = threadIdx.x; j < K; j += 256) {
        float g = 0.f;
        if (j < nt) {
            const float p = prow[j], logq = irow[j] - lse;
            if (p > 0.f) acc += p * (__logf(p) - logq);
            g = (__expf(logq) - p) * grad_scale;
        }
        if (dscore) dscore[(int64_t)t * K + j] = g;
    }
    acc = block_sum_256(acc, red);
    if (threadIdx.x == 0) loss[t] = nt > 0 ? acc : 0.f;
}

// The same for rows of at most 256 * NV scores (K a multiple of 4, rows 16-byte aligned): one wave per row, the row read
// once with all its 16-byte loads in flight and held in registers, reductions inside the wave - no pass over the row
// waits for another and no barrier (the kernel above reads the scores three times and meets at three barriers).
template <int NV>
__global__ __launch_bounds__(256) void dsa_indexer_kl_rows_kernel(const float *__restrict__ sel, const float *__restrict__ mass,
                                                                   const int32_t *__restrict__ nsel, int T, int K,
                                                                   float grad_scale, float *__restrict__ loss,
                                                                   float *__restrict__ dscore) {
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;                                  // (whole waves; nothing below synchronises the workgroup)
    const int nt = nsel[t], K4 = K >> 2;
    const float4 *irow = reinterpret_cast<const float4 *>(sel + (int64_t)t * K);
    const float4 *prow = reinterpret_cast<const float4 *>(mass + (int64_t)t * K);
    float s[NV][4], p[NV][4];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i4 = lane + 64 * u;
        const float4 a = irow[min(i4, K4 - 1)], b = prow[min(i4, K4 - 1)];
        s[u][0] = a.x; s[u][1] = a.y; s[u][2] = a.z; s[u][3] = a.w;
        p[u][0] = b.x; p[u][1] = b.y; p[u][2] = b.z; p[u][3] = b.w;
    }
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (4 * (lane + 64 * u) + c < nt) m = fmaxf(m, s[u][c]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    float z = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (4 * (lane + 64 * u) + c < nt) z += __expf(s[u][c] - m);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) z += __shfl_xor(z, off, 64);
    const float lse = m + __logf(z);
    float acc = 0.f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i4 = lane + 64 * u;
        float g[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            g[c] = 0.f;
            if (4 * i4 + c < nt) {
                const float logq = s[u][c] - lse;
                if (p[u][c] > 0.f) acc += p[u][c] * (__logf(p[u][c]) - logq);
                g[c] = (__expf(logq) - p[u][c]) * grad_scale;
            }
        }
        if (dscore && i4 < K4) reinterpret_cast<float4 *>(dscore + (int64_t)t * K)[i4] = make_float4(g[0], g[1], g[2], g[3]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) loss[t] = nt > 0 ? acc : 0.f;
}

extern "C" hipError_t dsa_launch_indexer_kl(const float *sel, const float *mass, const int32_t *n, int T, int K,
                                            float grad_scale, float *loss, float *dscore, hipStream_t stream) {
    if (T <= 0) return hipSuccess;
    const bool rows16 = K % 4 == 0 && ((reinterpret_cast<uintptr_t>(sel) | reinterpret_cast<uintptr_t>(mass) |
                                        reinterpret_cast<uintptr_t>(dscore)) & 15) == 0;
    const dim3 grid((unsigned)((T + 3) / 4));
#define KL_ROWS(NV) hipLaunchKernelGGL(dsa_indexer_kl_rows_kernel<NV>, grid, dim3(256), 0, stream, sel, mass, n, T, K, grad_scale, loss, dscore)
    if (rows16 && K <= 256) KL_ROWS(1);
    else if (rows16 && K <= 512) KL_ROWS(2);
    else if (rows16 && K <= 1024) KL_ROWS(4);
    else if (rows16 && K <= 2048) KL_ROWS(8);
    else hipLaunchKernelGGL(dsa_indexer_kl_kernel, dim3(T), dim3(256), 0, stream, sel, mass, n, K, grad_scale, loss, dscore);
#undef KL_ROWS
    return hipGetLastError();
}
