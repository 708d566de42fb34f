// dK and dV, launches: the kernel is dsa_tile_dkv.h
#include "dsa_tile_dkv.h"
#ifndef DKV_UNALIGNED
#define DKV_UNALIGNED 0
#endif

// ---- launch: one instance per head_dim, mask kind and (power-of-two padded) group size ----
struct DkvArgs {
    const void *dout, *q, *k, *v;
    const float *lse, *delta;
    const uint32_t *bitmap;
    int ldw;
    const int32_t *cu;
    int N, T, Hq, Hkv, d_real;
    float scale, logit_scale;
    int causal, skip_len;
    const int32_t *order;
    float *partial;
    void *dk, *dv;
};
template <int D, int KG, bool HAS_IDX, bool CARRIED, int GS>
static hipError_t launch_dkv(unsigned grid, hipStream_t stream, const DkvArgs &a) {
    constexpr size_t lds = dkv_lds_bytes<D, KG>();
    const auto kernel = &dsa_tile_dkv_kernel<D, KG, HAS_IDX, GS, DKV_UNALIGNED, CARRIED>;
    // (LDS above 64 KiB is asked for on every launch: neither a second device nor a second thread can meet a kernel never configured)
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256 / KG), lds, stream, (const bf16_t *)a.dout, (const bf16_t *)a.q, (const bf16_t *)a.k,
                       (const bf16_t *)a.v, a.lse, a.delta, a.bitmap, a.ldw, a.cu, a.N, a.T, a.Hq, a.Hkv, a.scale, a.logit_scale, a.causal, a.d_real, a.skip_len, a.order,
                       a.partial, (bf16_t *)a.dk, (bf16_t *)a.dv);
    return hipGetLastError();
}
template <int D, int KG, bool HAS_IDX, bool CARRIED = false>
static hipError_t launch_dkv_gs(unsigned grid, hipStream_t stream, const DkvArgs &a) {
    switch (group_shift(a.Hq, a.Hkv)) {
        case 0: return launch_dkv<D, KG, HAS_IDX, CARRIED, 0>(grid, stream, a);
        case 1: return launch_dkv<D, KG, HAS_IDX, CARRIED, 1>(grid, stream, a);
        case 2: return launch_dkv<D, KG, HAS_IDX, CARRIED, 2>(grid, stream, a);
        case 3: return launch_dkv<D, KG, HAS_IDX, CARRIED, 3>(grid, stream, a);
        default: return launch_dkv<D, KG, HAS_IDX, CARRIED, 4>(grid, stream, a);
    }
}
template <int D, bool HAS_IDX>
static hipError_t launch_dkv_kg(unsigned grid, hipStream_t stream, const DkvArgs &a) {
#if DKV_UNALIGNED
    // (head_dim 128: with the copies, two groups spill - 4 heads per kv head, 4096 and 2000 tokens without a mask 2190 us, one group 1761, 1000
    // and 300 causal 161 / 98, 4096 720 / 740)
    return launch_dkv_gs<D, D == 128 ? 1 : 2, HAS_IDX>(grid, stream, a);
#else
    if (dkv_key_groups(a.d_real, a.T, a.N, a.Hq, a.Hkv, a.causal) == 1) return launch_dkv_gs<D, 1, HAS_IDX>(grid, stream, a);
    return launch_dkv_gs<D, 2, HAS_IDX>(grid, stream, a);
#endif
}
// grid: workgroups (one per key tile or piece, and kv head).  The file is compiled twice, the second time (DKV_UNALIGNED) for q or dO on no
// 16-byte boundary (no CARRIED form there: all of the rows); k and v lie on one (the entry points see to it).
#define DKV_LAUNCH_ARGS unsigned grid, hipStream_t stream, const void *dout, const void *q, const void *k, const void *v, const float *lse, \
    const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, int d_real, float scale, int carried, int causal, int skip_len,   \
    const int32_t *order, float *partial, void *dk, void *dv
extern "C" hipError_t dsa_launch_dkv_tiles_unaligned(DKV_LAUNCH_ARGS);
#if DKV_UNALIGNED
extern "C" hipError_t dsa_launch_dkv_tiles_unaligned(DKV_LAUNCH_ARGS) {
#else
extern "C" hipError_t dsa_launch_dkv_tiles(DKV_LAUNCH_ARGS) {
    if (((uintptr_t)q | (uintptr_t)dout) & 15)
        return dsa_launch_dkv_tiles_unaligned(grid, stream, dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, carried, causal, skip_len, order, partial, dk, dv);
    if (carried) {
        const DkvArgs c{dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, logit_scale(scale), causal, skip_len, order, partial, dk, dv};
        return bitmap ? launch_dkv_gs<256, 1, true, true>(grid, stream, c) : launch_dkv_gs<256, 1, false, true>(grid, stream, c);
    }
#endif
    const DkvArgs a{dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, d_real, scale, logit_scale(scale), causal, skip_len, order, partial, dk, dv};
    if (bitmap) switch (d_real) {
        case 64: return launch_dkv_kg<64, true>(grid, stream, a);
        case 128: return launch_dkv_kg<128, true>(grid, stream, a);
        case 256: return launch_dkv_gs<256, 1, true>(grid, stream, a);
    } else switch (dense_kernel_dim(d_real)) {
        case 64: return launch_dkv_kg<64, false>(grid, stream, a);
        case 80: return launch_dkv_kg<80, false>(grid, stream, a);
        case 96: return launch_dkv_kg<96, false>(grid, stream, a);
        case 128: return launch_dkv_kg<128, false>(grid, stream, a);
        case 256: return launch_dkv_gs<256, 1, false>(grid, stream, a);
    }
    return hipErrorInvalidValue;
}
