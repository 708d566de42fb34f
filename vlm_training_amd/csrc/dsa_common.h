// Shared device helpers for the gfx950 DSA attention kernels (wave64, MFMA, LDS).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

#define DSA_WAVE 64
// key-side workgroups that run at a time, and the launches whose walks may be cut into pieces: up to three rounds of them (a longer
// launch of whole walks, longest first, ends level)
static inline int dkv_slots(int key_groups) { return 256 * key_groups; }
static inline int64_t dkv_pieces_max_wg(int D) { return D > 128 ? 3 * 256 : 3 * 512; }
// Groups of 32 keys that a wave of the key-side kernel takes: two up to head_dim 128 (each operand read feeds two MFMAs, two workgroups
// per CU), or one, four waves to a workgroup: its walk is twice as fast, and a CU holds one of them.
// With a causal mask walks are cut into pieces or finish in turn, and what counts is the launch's work, workgroups times the mean length of
// a segment in steps (32 rows: 32, 16, .. queries): little of it ends with the pace of single walks, much with the CU's; below
// 96 workgroups single walks count at any length.  Two groups against one, us, head_dim 128: 4 heads per kv head, one segment of 1408 tokens, 96 workgroups (17 000) 89 / 67, of 2432 and 160 (49 000) 135 /
// 143; 2 heads per kv head, 8064 and 128 (64 000) 153 / 190, eight of 1152 and 320 (23 000) 87 / 78, three of 2944 and 288 (53 000) 131 /
// 142.  Over 1050 launches (head_dim 64 to 128, 1 to 8 heads, equal and log-normal segments, with a selection and without) the choice is
// on average 1.3 % slower than the better one; lines on the workgroups alone were 4.2 to 5.
// Without a mask the tiles of a segment walk equally long: one group as long as all of them have a CU to themselves, T / 128 for each kv head
// (one segment, 252: 607 / 457, 268: 627 / 854).
static inline int dkv_key_groups(int D, int T, int N, int Hq, int Hkv, int causal) {
    if (D > 128) return 1;
    if (!causal) return (int64_t)(T / 128) * Hkv <= 256 ? 1 : 2;
    int rows = 1;                                        // of a query: its group's heads, padded to a power of two
    while (rows * Hkv < Hq) rows *= 2;
    const int64_t wg = ((int64_t)T / 128 + N) * Hkv;
    return wg < 96 || (wg <= dkv_pieces_max_wg(D) && wg * T / N * rows <= 40000 * 32) ? 1 : 2;
}
// The split of a selection's rows (row_split_for): the first row of a segment of L tokens that is not the tile kernels'.  pos_split in segments of split_len
// tokens and more, in shorter ones pos_short, but all of a segment that is up to a third longer than that.
__host__ __device__ static inline int tile_rows_end(int L, int pos_split, int split_len, int pos_short) {
    return L >= split_len ? pos_split : L - pos_short > pos_short / 3 ? pos_short : L;
}
// dQ in the key side's launch, where one holds both passes (dsa_tile_bwd.hip)
struct DqBeside { int window; void *dq; };
#define LOG2E_F 1.4426950408889634f
#define LN2_F 0.6931471805599453f

// MFMA operand layouts used throughout (wave64, lane l):
//   16x16x32 bf16:  A[i][k]: i = l%16, k = 8*(l/16)+e (e<8)   B[k][j]: j = l%16, k = 8*(l/16)+e
//                   C[i][j]: j = l%16, i = 4*(l/16)+v (v<4)
//   32x32x16 bf16:  A[i][k]: i = l%32, k = 8*(l/32)+e         B[k][j]: j = l%32, k = 8*(l/32)+e
//                   C[i][j]: j = l%32, i = 8*(v/4) + 4*(l/32) + v%4 (v<16)
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 zero_bf16x8() {
    u32x4 z = {0u, 0u, 0u, 0u};
    return __builtin_bit_cast(bf16x8, z);
}
__device__ __forceinline__ bf16x8 load_bf16x8(const bf16_t *p) {   // 16-byte aligned global/LDS read
    return *reinterpret_cast<const bf16x8 *>(p);
}

// two fp32 -> packed bf16 pair, round-to-nearest-even (one v_cvt_pk_bf16_f32 on gfx950)
// acc + sum_e a[e] * b[e] over 8 bf16 pairs, one fused multiply-add per element in element order.  Every kernel that forms
// delta = rowsum(dO * O) goes through this one chain, so that they agree to the bit.
__device__ __forceinline__ float dot8_chain(bf16x8 a, bf16x8 b, float acc) {
    const u32x4 x = __builtin_bit_cast(u32x4, a), y = __builtin_bit_cast(u32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        acc = __builtin_fmaf(__uint_as_float(x[e] << 16), __uint_as_float(y[e] << 16), acc);
        acc = __builtin_fmaf(__uint_as_float(x[e] & 0xffff0000u), __uint_as_float(y[e] & 0xffff0000u), acc);
    }
    return acc;
}

// delta[h,t] = sum_d dO[t,h,d] * O[t,h,d] of row (t, h) by 16 lanes (`sub` of them): lane i sums the 8-element chunks i, i+16, ...
// in one chain, then a butterfly over the 16 lanes (the tile dQ kernels reproduce this order when they form delta themselves)
__device__ __forceinline__ void delta_row(const bf16_t *__restrict__ dout, const bf16_t *__restrict__ out, int T, int Hq, int D, int64_t row, int sub,
                                          float *__restrict__ delta) {
    float acc = 0.f;
    if (row < (int64_t)T * Hq) {
        for (int c = sub * 8; c < D; c += 128)
            acc = dot8_chain(load_bf16x8(dout + row * D + c), load_bf16x8(out + row * D + c), acc);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (sub == 0 && row < (int64_t)T * Hq) {
        const int t = (int)(row / Hq), h = (int)(row % Hq);
        delta[(int64_t)h * T + t] = acc;
    }
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2bf(float lo, float hi) {
    const f32x2 f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

// segment lookup: index i with cu[i] <= t < cu[i+1] (zero-length segments are stepped over)
__device__ __forceinline__ int find_segment(const int32_t *__restrict__ cu, int N, int t) {
    int lo = 0, hi = N;            // invariant: cu[lo] <= t < cu[hi]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (cu[mid] <= t) lo = mid; else hi = mid;
    }
    return lo;
}

// the same by a whole wave (t wave-uniform, every lane active): the offsets are fetched 64 at a time, one per lane, in one
// memory round trip each instead of one round trip per step of a binary search
__device__ __forceinline__ int find_segment_wave(const int32_t *__restrict__ cu, int N, int t) {
    const int lane = threadIdx.x & 63;
    int below = 0;                 // offsets cu[0 .. N-1] that are <= t; the segment is the last of them
    for (int base = 0; base < N; base += 64) {
        const int c = cu[min(base + lane, N - 1)];
        const int hits = (int)__popcll(__builtin_amdgcn_ballot_w64(base + lane < N && c <= t));
        below += hits;
        if (hits < 64) break;
    }
    return max(below - 1, 0);
}

__device__ __forceinline__ float wave_xor_f(float v, int m) { return __shfl_xor(v, m, 64); }
// maximum / sum over the two lanes 32 apart, on every lane: v_permlane32_swap exchanges the wave's halves in
// the vector ALU (no LDS round trip, so LDS reads in flight are not waited for)
__device__ __forceinline__ float half_max_f(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum_f(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ---- memory straight into LDS (buffer_load ... lds) ------------------------------------------------------------------
// A wave's load puts 64 x 16 bytes at consecutive LDS addresses, lane by lane, without passing through registers.  It is
// inline assembly because the compiler's own intrinsic makes every later LDS read wait for every such load; here the
// kernel waits itself (wait_vmcnt, then a barrier) before anything reads the bytes.  A compiler-made vmcnt wait only ever
// waits longer for the loads it does not know of.
typedef uint32_t buffer_rsrc __attribute__((ext_vector_type(4)));
// a buffer of `bytes` bytes (held to 32 bits) starting at p (wave-uniform): reads past its end give zero
__device__ __forceinline__ buffer_rsrc make_buffer_rsrc(const void *p, int64_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t n = bytes < 0 ? 0u : bytes > 0xffffffffll ? 0xffffffffu : (uint32_t)bytes;
    return buffer_rsrc{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)),
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)n), 0x00020000u};
}
// the same from scalars (a pointer and a size that scalar instructions formed)
__device__ __forceinline__ buffer_rsrc scalar_buffer_rsrc(const void *p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return buffer_rsrc{(uint32_t)a, (uint32_t)(a >> 32), bytes, 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_address(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
// 16 bytes per lane from byte voff of the buffer to LDS byte `lds` (wave-uniform) + 16 * lane.  The scalar offset of the
// instruction stays 0: the bounds check need not include it, so a piece's or a tile's offset goes into voff or into the
// buffer's start.  (The wait states cover a scalar operand that a vector instruction wrote just before, and M0.)
__device__ __forceinline__ void buffer_load_lds16(buffer_rsrc rsrc, int voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 : : "v"(voff), "s"(rsrc), "s"(lds) : "memory", "m0");
}
// the same with 4 bytes per lane, to LDS byte `lds` + 4 * lane
__device__ __forceinline__ void buffer_load_lds4(buffer_rsrc rsrc, int voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tbuffer_load_dword %0, %1, 0 offen lds"
                 : : "v"(voff), "s"(rsrc), "s"(lds) : "memory", "m0");
}
// the same from each lane's own address
__device__ __forceinline__ void global_load_lds4(const void *p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dword %0, off" : : "v"(p), "s"(lds) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
// the barrier alone: LDS operations of this wave may still be in flight
__device__ __forceinline__ void barrier_only() { asm volatile("s_barrier" : : : "memory"); }
