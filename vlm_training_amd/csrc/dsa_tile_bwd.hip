// dK, dV and dQ of one backward in one launch, head_dim 256: the workgroups of dsa_tile_dkv.h first, those of dsa_tile_dq.h behind them.
// Each has four waves of one per SIMD and most of a CU's LDS, so that either takes a CU alone, and the shorter walks of dQ fill what
// the longest ones of the key side leave idle - what two streams did before, for two events, two waits (42 us of the host's time a step)
// and the queues' latency.  Step, us, two streams -> one launch: fp32 2048 tokens 150 -> 114, head_dim 256 at 16 384 tokens 855 -> 848.
#define DKV_AS_FUNCTION
#include "dsa_tile_dkv.h"
#include "dsa_tile_dq.h"

template <bool HAS_IDX, int GSHIFT, bool CARRIED>
__global__ __launch_bounds__(256, 1) void dsa_tile_dkv_kernel_and_dq(
    int key_blocks, const bf16_t *__restrict__ dout, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v,
    const float *__restrict__ lse, const float *__restrict__ delta, const uint32_t *__restrict__ bitmap, int ldw, const int32_t *__restrict__ cu,
    int N, int T, int Hq, int Hkv, float scale, float logit_scale, int causal, const int32_t *__restrict__ order, float *__restrict__ partial,
    bf16_t *__restrict__ dk, bf16_t *__restrict__ dv, int window, bf16_t *__restrict__ dq) {
    if ((int)blockIdx.x < key_blocks)
        dkv_block<256, 1, HAS_IDX, GSHIFT, false, CARRIED>(blockIdx.x, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, logit_scale,
                                                           causal, 256, INT32_MAX, order, partial, dk, dv);
    else
        dq_block<256, HAS_IDX, 4, 1, CARRIED>(blockIdx.x - key_blocks, gridDim.x - key_blocks, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, GSHIFT, scale,
                                              INT32_MAX, 0, INT32_MAX, window, causal, 256, dq, nullptr, nullptr);
}

template <bool HAS_IDX, int GS, bool CARRIED>
static hipError_t launch(unsigned key_blocks, hipStream_t stream, const void *dout, const void *q, const void *k, const void *v, const float *lse,
                         const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int causal,
                         const int32_t *order, float *partial, void *dk, void *dv, int window, void *dq) {
    constexpr size_t key_lds = dkv_lds_bytes<256, 1>(), q_lds = dq_lds_bytes<256, 4>(HAS_IDX), lds = key_lds > q_lds ? key_lds : q_lds;
    const auto kernel = &dsa_tile_dkv_kernel_and_dq<HAS_IDX, GS, CARRIED>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const unsigned blocks = (unsigned)(((int64_t)T / (128 >> GS) + N + 1) * Hkv);
    hipLaunchKernelGGL(kernel, dim3(key_blocks + blocks), dim3(256), lds, stream, (int)key_blocks, (const bf16_t *)dout, (const bf16_t *)q,
                       (const bf16_t *)k, (const bf16_t *)v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, logit_scale(scale), causal, order, partial,
                       (bf16_t *)dk, (bf16_t *)dv, window, (bf16_t *)dq);
    return hipGetLastError();
}
// key_blocks: workgroups of the key side, a multiple of Hkv; q and dO on 16-byte boundaries; every query row is the tile kernels'; delta is there
extern "C" hipError_t dsa_launch_dkv_dq_tiles(unsigned key_blocks, hipStream_t stream, const void *dout, const void *q, const void *k, const void *v,
                                              const float *lse, const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N,
                                              int T, int Hq, int Hkv, float scale, int carried, int causal, const int32_t *order, float *partial,
                                              void *dk, void *dv, int window, void *dq) {
#define LAUNCH(HI, GS, CA) return launch<HI, GS, CA>(key_blocks, stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, scale, causal, order, partial, dk, dv, window, dq)
#define LAUNCH_GS(HI, CA)                     \
    switch (group_shift(Hq, Hkv)) {           \
        case 0: LAUNCH(HI, 0, CA);            \
        case 1: LAUNCH(HI, 1, CA);            \
        case 2: LAUNCH(HI, 2, CA);            \
        case 3: LAUNCH(HI, 3, CA);            \
        default: LAUNCH(HI, 4, CA);           \
    }
    if (carried) { if (bitmap) LAUNCH_GS(true, true) else LAUNCH_GS(false, true) }
    else { if (bitmap) LAUNCH_GS(true, false) else LAUNCH_GS(false, false) }
#undef LAUNCH_GS
#undef LAUNCH
}
