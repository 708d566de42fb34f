// dQ, launches: the kernel is dsa_tile_dq.h
#include "dsa_tile_dq.h"

template <int D, bool HAS_IDX, int NW, int RG, bool CARRIED>
__global__ __launch_bounds__(NW * 64, 1) void dsa_tile_dq_kernel(
    const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k,
    const bf16_t *__restrict__ v, const float *__restrict__ lse, const float *delta,
    const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu, int N, int T, int Hq, int Hkv, int gshift,
    float scale, int pos_split, int split_len, int pos_short, int window, int causal, int d_real, bf16_t *__restrict__ dq, const bf16_t *__restrict__ out_for_delta,
    float *delta_out) {
    dq_block<D, HAS_IDX, NW, RG, CARRIED>(blockIdx.x, gridDim.x, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, gshift, scale, pos_split, split_len, pos_short, window, causal, d_real, dq, out_for_delta, delta_out);
}

template <int D, bool HAS_IDX, int RG, bool CARRIED = false>
static hipError_t launch_dq_i(hipStream_t stream, const void *dout, const void *q, const void *k, const void *v, const float *lse,
                              const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, int gs,
                              int d_real, float scale, int pos_split, int split_len, int pos_short, int window, int causal, void *dq, const void *out_for_delta, float *delta_out) {
    constexpr int NW = 4;
    constexpr size_t lds = dq_lds_bytes<D, NW>(HAS_IDX);
    const auto kernel = &dsa_tile_dq_kernel<D, HAS_IDX, NW, RG, CARRIED>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const dim3 grid((unsigned)(((int64_t)T / ((32 * NW * RG) >> gs) + N + 1) * Hkv));
    hipLaunchKernelGGL(kernel, grid, dim3(64 * NW), lds, stream, (const bf16_t *)dout, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, lse, delta,
                       bitmap, ldw, cu, N, T, Hq, Hkv, gs, scale, pos_split, split_len, pos_short, window, causal, d_real, (bf16_t *)dq, (const bf16_t *)out_for_delta, delta_out);
    return hipGetLastError();
}
// 32 rows per wave instead of 64: each walk is then twice as fast, two workgroups share a CU, and blocks are half as long, which wastes fewer
// rows at the ends of segments; the operand reads they share are worth 5 to 10 %.  wg: workgroups of 256 rows, at most.
// With a causal mask (blocks go heaviest first) the finer blocks win while the launch's work, workgroups times the mean length of a segment,
// is small (measured up to 1280 of them).  64 rows against 32, us, head_dim 128: one segment 3968 tokens 256 workgroups 124 / 102, 6016 and 384 211 / 194, 8064 and 512
// 323 / 344; eight segments of 1920 and 512 90 / 90, of 2432 and 640 147 / 132; 35 of mean 330 and 496 38 % more.
// Without a mask every block of a segment walks equally long, so that what counts is the number of rounds: of 256 workgroups, or of 256
// half as long.  Four segments, head_dim 128: 128 workgroups 36 / 24, 224 65 / 66, 288 155 / 123, 384 205 / 178, 512 306 / 313, 640 525 / 489;
// short segments take 32 rows (of 320 to 512: 5 to 12 % less, log-normal ones more).
// Over 880 causal launches, with a selection and without, and 490 without a mask (head_dim 64 to 128) the choice is on average 0.3 and 0.5 %
// slower than the better one; lines on the workgroups alone were 1.3 to 4 and 7.
static bool dq_one_row_group(int causal, int T, int N, int Hkv, int gs) {
    const int64_t rows = (int64_t)T << gs, wg = (rows / 256 + N) * Hkv;
    if (causal) return wg <= 416 || (wg <= 1280 && wg * T / N <= 2000000);
    if (wg > 1024) return false;
    return T / N < 1500 || (rows / 128 * Hkv + 255) / 256 < 2 * (((2 * (rows / 256) + N) * Hkv + 511) / 512);
}
// d_real: elements of a row, without a selection any multiple of 8 (dense_kernel_dim).  window: rows of a bitmap at positions below it attend
// all of their causal window (0: nothing is known).  carried: see DSA_CARRIED_KS.  out_for_delta != null: the kernel forms
// delta = rowsum(dO * O) of its rows itself and writes it to delta_out
extern "C" hipError_t dsa_launch_tile_dq(const void *dout, const void *q, const void *k, const void *v,
                                         const float *lse, const float *delta, const uint32_t *bitmap, int ldw,
                                         const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real, float scale,
                                         int pos_split, int split_len, int pos_short, int window, int carried, int causal, void *dq, const void *out_for_delta, float *delta_out,
                                         hipStream_t stream) {
    const int gs = group_shift(Hq, Hkv);
    const bool one_group = dq_one_row_group(causal, T, N, Hkv, gs);
#define DQ_ARGS stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, gs, d_real, scale, pos_split, split_len, pos_short, window, causal, dq, out_for_delta, delta_out
#define DQ_CASE(D_, HI) return one_group ? launch_dq_i<D_, HI, 1>(DQ_ARGS) : launch_dq_i<D_, HI, 2>(DQ_ARGS)
    if (carried) return bitmap ? launch_dq_i<256, true, 1, true>(DQ_ARGS) : launch_dq_i<256, false, 1, true>(DQ_ARGS);
    if (bitmap) switch (d_real) {
        case 64: DQ_CASE(64, true);
        case 128: DQ_CASE(128, true);
        case 256: return launch_dq_i<256, true, 1>(DQ_ARGS);
    } else switch (dense_kernel_dim(d_real)) {
        case 64: DQ_CASE(64, false);
        case 80: DQ_CASE(80, false);
        case 96: DQ_CASE(96, false);
        case 128: DQ_CASE(128, false);
        case 256: return launch_dq_i<256, false, 1>(DQ_ARGS);
    }
#undef DQ_ARGS
#undef DQ_CASE
    return hipErrorInvalidValue;
}
