// Pre-attention prologue and post-attention gate of the reference's attention layers, fused:
//   q, k  <-  rope(rms_norm(q_proj), cos, sin)   written straight into the packed (T, H, D) layout the
//             attention operator reads   (models/qwen3_vl/model.py:256-269, models/qwen3_5/model.py:110-129:
//             F.rms_norm per head, transpose, apply_rope, transpose back, .contiguous())
//   out   <-  out * sigmoid(gate)          (models/qwen3_5/model.py:135)
// HBM-bound element-wise work with one reduction per (token, head) row: a row of D bf16 is spread over
// D/8 lanes (16 bytes per lane), so a wave handles 512/D rows per step; the row reduction and the
// rotate_half partner (R/16 lanes away) are cross-lane moves inside those D/8 lanes.  One wave per token
// and step walks the token's query heads or its key heads; cos/sin of the token are loaded once.
// What bounds it is the memory latency a wave sees between its rows: the forward loads four steps' rows together, q and k go to
// workgroups of their own (one weight and one set of sums in registers instead of two: more waves per SIMD), and the partner's
// half comes over as packed bf16 (four lane moves instead of eight).  16 384 tokens, 16 + 2 heads of 256: forward 79 -> 63 us
// (4.8 TB/s), backward 107 -> 105; 8192 tokens, 16 + 8 heads of 128: forward 34 -> 24, backward 42 -> 33.
// Everything here is read once and written once, so it goes past the caches (non-temporal loads and stores): written lines left
// in the Infinity Cache had to be pushed out by the next kernel's reads - 16 384 tokens, 16 heads of 256, norm, rotation and gate
// with backward 372 -> 332 us (5.5 TB/s over all); a layer whose next kernel reads the result (8192 tokens) is not slower for it.
// The backward pass returns the gradients of the projections' outputs and per-workgroup partial sums of
// the two norm weights' gradients (reduced by a second kernel in a fixed order: no atomics).
#include "dsa_common.h"

typedef float f32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x8 bf8_to_f32(u32x4 w) {
    f32x8 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[2 * i] = __uint_as_float(w[i] << 16);
        r[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
    return r;
}
__device__ __forceinline__ u32x4 f32_to_bf8(f32x8 x) {
    return u32x4{pack2bf(x[0], x[1]), pack2bf(x[2], x[3]), pack2bf(x[4], x[5]), pack2bf(x[6], x[7])};
}
// the eight bf16 of another lane
__device__ __forceinline__ u32x4 shfl4(u32x4 x, int lane) {
    return u32x4{(uint32_t)__shfl((int)x[0], lane, 64), (uint32_t)__shfl((int)x[1], lane, 64), (uint32_t)__shfl((int)x[2], lane, 64), (uint32_t)__shfl((int)x[3], lane, 64)};
}
__device__ __forceinline__ float bf16_round(float x) { return __uint_as_float(pack2bf(x, 0.f) << 16); }

// cos/sin of this lane's 8 elements of token t (zero-filled past the rotary width R)
template <bool CS_F32>
__device__ __forceinline__ void load_cs(const void *cs, int64_t t, int R, int d0, f32x8 &out, float fill) {
    if (d0 < R) {
        if (CS_F32) {
            const float *p = reinterpret_cast<const float *>(cs) + t * R + d0;
            const f32x4 a = *reinterpret_cast<const f32x4 *>(p), b = *reinterpret_cast<const f32x4 *>(p + 4);
            out = f32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        } else {
            out = bf8_to_f32(*reinterpret_cast<const u32x4 *>(reinterpret_cast<const bf16_t *>(cs) + t * R + d0));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = fill;
    }
}

// sum over the LPR lanes that share a row (LPR is a power of two <= 32; rows are aligned groups of lanes)
template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
#pragma unroll
    for (int m = 1; m < LPR; m <<= 1) x += __shfl_xor(x, m, 64);
    return x;
}

// a norm weight as the module holds it: fp32 (the trainer's master parameters under autocast) or bf16
__device__ __forceinline__ f32x8 norm_weights(const void *w, int w_bf16, int d0, float offset) {
    f32x8 r;
    if ((uintptr_t)w & 15) {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = w_bf16 ? (float)reinterpret_cast<const bf16_t *>(w)[d0 + i] : reinterpret_cast<const float *>(w)[d0 + i];
    } else if (w_bf16) {
        r = bf8_to_f32(*reinterpret_cast<const u32x4 *>(reinterpret_cast<const bf16_t *>(w) + d0));
    } else {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(w) + d0), b = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(w) + d0 + 4);
        r = f32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] += offset;
    return r;
}

// q's or k's share of the workgroups: blocks 0 .. nbq-1 take q, the rest k
struct RopeSide { int first, blocks, H; bool isq; };
__device__ __forceinline__ RopeSide rope_side(int nbq, int Hq, int Hkv) {
    if ((int)blockIdx.x < nbq) return RopeSide{(int)blockIdx.x, nbq, Hq, true};
    return RopeSide{(int)blockIdx.x - nbq, (int)gridDim.x - nbq, Hkv, false};
}

template <int D, bool CS_F32>
__global__ __launch_bounds__(256) void dsa_qk_norm_rope_fwd_kernel(
    const bf16_t *__restrict__ q_in, int64_t q_tok, int64_t q_head, const bf16_t *__restrict__ k_in, int64_t k_tok,
    int64_t k_head, const void *__restrict__ qw, const void *__restrict__ kw, int w_bf16, float eps, float w_offset,
    const void *__restrict__ cosp, const void *__restrict__ sinp, int R, int T, int Hq, int Hkv, int nbq,
    bf16_t *__restrict__ q_out, bf16_t *__restrict__ k_out, float *__restrict__ q_rstd, float *__restrict__ k_rstd) {
    constexpr int LPR = D / 8, RPW = 64 / LPR, ROWS = 4; // lanes per row, rows per wave and step, steps loaded together
    const RopeSide sd = rope_side(nbq, Hq, Hkv);
    const bf16_t *const in = sd.isq ? q_in : k_in;
    const int64_t tok = sd.isq ? q_tok : k_tok, head = sd.isq ? q_head : k_head;
    bf16_t *const out = sd.isq ? q_out : k_out;
    float *const rstd_out = sd.isq ? q_rstd : k_rstd;
    const void *const wp = sd.isq ? qw : kw;
    const int H = sd.H, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int sub = lane / LPR, d0 = (lane % LPR) * 8;
    const int half_lanes = R / 16;                       // rotate_half partner distance in lanes
    const bool low = d0 < R / 2, rot = d0 < R;
    const int partner = low ? lane + half_lanes : lane - half_lanes;
    const f32x8 w = norm_weights(wp, w_bf16, d0, w_offset);
    for (int64_t t = (int64_t)sd.first * 4 + wv; t < T; t += (int64_t)sd.blocks * 4) {
        f32x8 c, s;
        load_cs<CS_F32>(cosp, t, R, d0, c, 1.f);
        load_cs<CS_F32>(sinp, t, R, d0, s, 0.f);
        const bf16_t *const src = in + t * tok + d0;
        for (int r0 = 0; r0 < H; r0 += ROWS * RPW) {
            u32x4 raw[ROWS];
#pragma unroll
            for (int u = 0; u < ROWS; ++u) raw[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + min(r0 + u * RPW + sub, H - 1) * head));
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                if (u > 0 && r0 + u * RPW >= H) break;   // (wave-uniform)
                const int r = r0 + u * RPW + sub;
                const f32x8 x = bf8_to_f32(raw[u]);
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
                const float rstd = rsqrtf(row_sum<LPR>(ss) * (1.f / D) + eps);
                f32x8 xn, y;
#pragma unroll
                for (int i = 0; i < 8; ++i) xn[i] = x[i] * rstd * w[i];
                const u32x4 nb = f32_to_bf8(xn);                                     // F.rms_norm returns bf16
                // rotate_half: element i < R/2 takes -n[i + R/2], element R/2 <= i < R takes n[i - R/2]
                const f32x8 n = bf8_to_f32(nb), other = bf8_to_f32(shfl4(nb, partner));
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = rot ? n[i] * c[i] + (low ? -other[i] : other[i]) * s[i] : n[i];
                if (r < H) {
                    __builtin_nontemporal_store(f32_to_bf8(y), reinterpret_cast<u32x4 *>(out + (t * H + r) * D + d0));
                    if (d0 == 0) rstd_out[t * H + r] = rstd;
                }
            }
        }
    }
}

// gradients: g = d(loss)/d(rope output).  dn = rope^T g, dx = rstd * (dn*w - xhat * mean(dn*w*xhat)),
// dw += dn * xhat (per workgroup partial sums: part[block][D], q's blocks first)
template <int D, bool CS_F32>
__global__ __launch_bounds__(256) void dsa_qk_norm_rope_bwd_kernel(
    const bf16_t *__restrict__ gq, const bf16_t *__restrict__ gk, const bf16_t *__restrict__ q_in, int64_t q_tok,
    int64_t q_head, const bf16_t *__restrict__ k_in, int64_t k_tok, int64_t k_head, const void *__restrict__ qw,
    const void *__restrict__ kw, int w_bf16, float w_offset, const void *__restrict__ cosp, const void *__restrict__ sinp, int R,
    const float *__restrict__ q_rstd, const float *__restrict__ k_rstd, int T, int Hq, int Hkv, int nbq,
    bf16_t *__restrict__ dq_in, int64_t dq_tok, int64_t dq_head, bf16_t *__restrict__ dk_in, int64_t dk_tok,
    int64_t dk_head, float *__restrict__ part) {
    constexpr int LPR = D / 8, RPW = 64 / LPR;
    __shared__ float red[4][D];
    const RopeSide sd = rope_side(nbq, Hq, Hkv);
    const bf16_t *const in = sd.isq ? q_in : k_in, *const gin = sd.isq ? gq : gk;
    const int64_t tok = sd.isq ? q_tok : k_tok, head = sd.isq ? q_head : k_head;
    bf16_t *const out = sd.isq ? dq_in : dk_in;
    const int64_t out_tok = sd.isq ? dq_tok : dk_tok, out_head = sd.isq ? dq_head : dk_head;
    const float *const rstd_in = sd.isq ? q_rstd : k_rstd;
    const void *const wp = sd.isq ? qw : kw;
    const int H = sd.H, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int sub = lane / LPR, d0 = (lane % LPR) * 8;
    const int half_lanes = R / 16;
    const bool low = d0 < R / 2, rot = d0 < R;
    const int partner = low ? lane + half_lanes : lane - half_lanes;
    const f32x8 w = norm_weights(wp, w_bf16, d0, w_offset);
    f32x8 a;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = 0.f;
    for (int64_t t = (int64_t)sd.first * 4 + wv; t < T; t += (int64_t)sd.blocks * 4) {
        f32x8 c, s;
        load_cs<CS_F32>(cosp, t, R, d0, c, 1.f);
        load_cs<CS_F32>(sinp, t, R, rot ? (low ? d0 + R / 2 : d0 - R / 2) : d0, s, 0.f);         // the partner's
        const bf16_t *const src = in + t * tok + d0, *const gsrc = gin + t * H * D + d0;
        for (int r0 = 0; r0 < H; r0 += RPW) {
            const int r = r0 + sub, rc = min(r, H - 1);
            const bool live = r < H;
            const u32x4 graw = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(gsrc + rc * D));
            const f32x8 x = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + rc * head))), g = bf8_to_f32(graw);
            const float rstd = live ? rstd_in[t * H + rc] : 0.f;
            const f32x8 gp = bf8_to_f32(shfl4(graw, partner));
            f32x8 dn, xh;
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // transpose of rotate_half: dn[i] = g[i] cos[i] + (i < R/2 ? g[i+R/2] sin[i+R/2] : -g[i-R/2] sin[i-R/2])
                const float other = gp[i] * s[i];
                dn[i] = rot ? g[i] * c[i] + (low ? other : -other) : g[i];
                xh[i] = x[i] * rstd;
                dot += dn[i] * w[i] * xh[i];
            }
            const float mean = row_sum<LPR>(dot) * (1.f / D);
            f32x8 dx;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                dx[i] = rstd * (dn[i] * w[i] - xh[i] * mean);
                a[i] += dn[i] * xh[i];                   // dead rows carry zeros (rstd)
            }
            if (live) __builtin_nontemporal_store(f32_to_bf8(dx), reinterpret_cast<u32x4 *>(out + t * out_tok + r * out_head + d0));
        }
    }
    // rows of one wave -> one value per d; then the four waves; fixed order throughout
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int m = LPR; m < 64; m <<= 1) a[i] += __shfl_xor(a[i], m, 64);
    }
    if (sub == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) red[wv][d0 + i] = a[i];
    }
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += 256) part[(int64_t)blockIdx.x * D + d] = red[0][d] + red[1][d] + red[2][d] + red[3][d];
}

// dw[which][d] = sum over the workgroups' partial sums, fp32 or bf16 as the weight is.  A workgroup owns 16 consecutive d of one
// weight, four per thread: thread (x, y) of 4 x 256 adds the partials of blocks y, y+256, ..., then the 256 sub-sums are added
// in y order (sixteen at a time, then the sixteen) - the same order on every run.  Bound by the latency of those loads: 64 d
// per workgroup, one load per thread and step, 12.9 us at head_dim 256 and 2048 blocks; this form 6.
template <bool OUT_BF16>
__global__ __launch_bounds__(1024) void dsa_norm_weight_reduce_kernel(const float *__restrict__ part, int nbq, int nbk, int D,
                                                                      void *__restrict__ dqw, void *__restrict__ dkw) {
    __shared__ f32x4 red[256][4];
    __shared__ f32x4 red2[16][4];
    const int x = threadIdx.x & 3, y = threadIdx.x >> 2;
    const int which = (blockIdx.x * 16) / D, d = (blockIdx.x * 16) % D + 4 * x;
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int b = (which ? nbq : 0) + y; b < (which ? nbq + nbk : nbq); b += 256) a += *reinterpret_cast<const f32x4 *>(part + (int64_t)b * D + d);
    red[y][x] = a;
    __syncthreads();
    if (y < 16) {
        f32x4 t = red[16 * y][x];
#pragma unroll
        for (int i = 1; i < 16; ++i) t += red[16 * y + i][x];
        red2[y][x] = t;
    }
    __syncthreads();
    if (y == 0) {
        f32x4 t = red2[0][x];
#pragma unroll
        for (int i = 1; i < 16; ++i) t += red2[i][x];
        void *out = which ? dkw : dqw;
        if (OUT_BF16) *reinterpret_cast<u32x2 *>((bf16_t *)out + d) = u32x2{pack2bf(t[0], t[1]), pack2bf(t[2], t[3])};
        else *reinterpret_cast<f32x4 *>((float *)out + d) = t;
    }
}

// ---- out * sigmoid(gate) (models/qwen3_5/model.py:135); rows of `width` elements, gate rows strided ----
__global__ __launch_bounds__(256) void dsa_sigmoid_gate_fwd_kernel(const bf16_t *__restrict__ x, const bf16_t *__restrict__ gate,
                                                                   int64_t gate_tok, int64_t gate_head, int D, int H, int64_t rows,
                                                                   bf16_t *__restrict__ y) {
    // one 16-byte chunk per thread and step; chunk c covers elements [8c, 8c+8) of the (rows, H*D) matrix
    const int64_t chunks = rows * H * D / 8;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < chunks; c += (int64_t)gridDim.x * 256) {
        const int64_t e = c * 8, t = e / ((int64_t)H * D);
        const int rem = (int)(e - t * H * D), hh = rem / D, d = rem % D;
        const f32x8 a = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + e)));
        const f32x8 g = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(gate + t * gate_tok + hh * gate_head + d)));
        f32x8 r;
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = a[i] * bf16_round(1.f / (1.f + __expf(-g[i])));   // torch.sigmoid returns bf16
        __builtin_nontemporal_store(f32_to_bf8(r), reinterpret_cast<u32x4 *>(y + e));
    }
}
__global__ __launch_bounds__(256) void dsa_sigmoid_gate_bwd_kernel(const bf16_t *__restrict__ gy, const bf16_t *__restrict__ x,
                                                                   const bf16_t *__restrict__ gate, int64_t gate_tok,
                                                                   int64_t gate_head, int D, int H, int64_t rows,
                                                                   bf16_t *__restrict__ dx, bf16_t *__restrict__ dgate,
                                                                   int64_t dgate_tok, int64_t dgate_head) {
    const int64_t chunks = rows * H * D / 8;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < chunks; c += (int64_t)gridDim.x * 256) {
        const int64_t e = c * 8, t = e / ((int64_t)H * D);
        const int rem = (int)(e - t * H * D), hh = rem / D, d = rem % D;
        const f32x8 gyv = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(gy + e)));
        const f32x8 a = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + e)));
        const f32x8 g = bf8_to_f32(__builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(gate + t * gate_tok + hh * gate_head + d)));
        f32x8 r1, r2;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float sg = 1.f / (1.f + __expf(-g[i]));
            r1[i] = gyv[i] * sg;
            r2[i] = gyv[i] * a[i] * sg * (1.f - sg);
        }
        __builtin_nontemporal_store(f32_to_bf8(r1), reinterpret_cast<u32x4 *>(dx + e));
        __builtin_nontemporal_store(f32_to_bf8(r2), reinterpret_cast<u32x4 *>(dgate + t * dgate_tok + hh * dgate_head + d));
    }
}

// ---- launchers -------------------------------------------------------------------------------------
static inline int prologue_blocks(int T) {
    const int want = (T + 3) / 4;
    return want < 1 ? 1 : (want > 2048 ? 2048 : want);
}
extern "C" int dsa_prologue_bwd_blocks(int T) { return prologue_blocks(T); }
// q's workgroups: every wave the same number of tokens (a wave with one token more than the others is what the launch ends on);
// k's: fewer, as its few heads make a token cheaper - by the steps of a token and about two more to get them going.  The
// backward stays within `most` of each (its partial sums: D floats per workgroup, in a workspace for 2 D per block).
static inline int even_blocks(int T, int most) {
    const int waves = 4 * (most < 1 ? 1 : most), per_wave = (T + waves - 1) / waves;
    return (T + 4 * per_wave - 1) / (4 * per_wave);
}
static inline int prologue_blocks_q(int T, int most) { return even_blocks(T, most); }
static inline int prologue_blocks_k(int T, int most, int Hq, int Hkv, int D) {
    const int rpw = 512 / D, q = (Hq + rpw - 1) / rpw + 2, k = (Hkv + rpw - 1) / rpw + 2;
    const int share = (int)((int64_t)even_blocks(T, most) * k / q);
    return even_blocks(T, share < most ? share : most);
}
#define FWD_BLOCKS 8192                                  // (up to 32 768 tokens: one per wave)
#define PROLOGUE_SWITCH(KERNEL, ...)                                                        \
    switch (D) {                                                                            \
        case 64: if (cs_f32) hipLaunchKernelGGL((KERNEL<64, true>), __VA_ARGS__); else hipLaunchKernelGGL((KERNEL<64, false>), __VA_ARGS__); break;    \
        case 128: if (cs_f32) hipLaunchKernelGGL((KERNEL<128, true>), __VA_ARGS__); else hipLaunchKernelGGL((KERNEL<128, false>), __VA_ARGS__); break; \
        case 256: if (cs_f32) hipLaunchKernelGGL((KERNEL<256, true>), __VA_ARGS__); else hipLaunchKernelGGL((KERNEL<256, false>), __VA_ARGS__); break; \
        default: return hipErrorInvalidValue;                                               \
    }

extern "C" hipError_t dsa_launch_qk_norm_rope_fwd(const void *q_in, int64_t q_tok, int64_t q_head, const void *k_in,
                                                  int64_t k_tok, int64_t k_head, const void *qw, const void *kw, int w_bf16, float eps,
                                                  float w_offset, const void *cosp, const void *sinp, int cs_f32, int R, int T,
                                                  int Hq, int Hkv, int D, void *q_out, void *k_out, float *q_rstd,
                                                  float *k_rstd, hipStream_t stream) {
    if (T == 0) return hipSuccess;
    const int most = T < 4 * FWD_BLOCKS ? (T + 3) / 4 : FWD_BLOCKS, nbq = prologue_blocks_q(T, most), nbk = prologue_blocks_k(T, most, Hq, Hkv, D);
    PROLOGUE_SWITCH(dsa_qk_norm_rope_fwd_kernel, dim3(nbq + nbk), dim3(256), 0, stream, (const bf16_t *)q_in, q_tok,
                    q_head, (const bf16_t *)k_in, k_tok, k_head, qw, kw, w_bf16, eps, w_offset, cosp, sinp, R, T, Hq, Hkv, nbq,
                    (bf16_t *)q_out, (bf16_t *)k_out, q_rstd, k_rstd)
    return hipGetLastError();
}

extern "C" hipError_t dsa_launch_qk_norm_rope_bwd(const void *gq, const void *gk, const void *q_in, int64_t q_tok,
                                                  int64_t q_head, const void *k_in, int64_t k_tok, int64_t k_head,
                                                  const void *qw, const void *kw, int w_bf16, float w_offset, const void *cosp,
                                                  const void *sinp, int cs_f32, int R, const float *q_rstd,
                                                  const float *k_rstd, int T, int Hq, int Hkv, int D, void *dq_in,
                                                  int64_t dq_tok, int64_t dq_head, void *dk_in, int64_t dk_tok,
                                                  int64_t dk_head, void *dqw, void *dkw, int grad_bf16, float *part, hipStream_t stream) {
    const int most = prologue_blocks(T), nbq = T > 0 ? prologue_blocks_q(T, most) : 0, nbk = T > 0 ? prologue_blocks_k(T, most, Hq, Hkv, D) : 0;
    if (T > 0) {
        PROLOGUE_SWITCH(dsa_qk_norm_rope_bwd_kernel, dim3(nbq + nbk), dim3(256), 0, stream, (const bf16_t *)gq, (const bf16_t *)gk,
                        (const bf16_t *)q_in, q_tok, q_head, (const bf16_t *)k_in, k_tok, k_head, qw, kw, w_bf16, w_offset, cosp, sinp,
                        R, q_rstd, k_rstd, T, Hq, Hkv, nbq, (bf16_t *)dq_in, dq_tok, dq_head, (bf16_t *)dk_in, dk_tok, dk_head, part)
    }
    if (grad_bf16) hipLaunchKernelGGL((dsa_norm_weight_reduce_kernel<true>), dim3(2 * D / 16), dim3(1024), 0, stream, part, nbq, nbk, D, dqw, dkw);
    else hipLaunchKernelGGL((dsa_norm_weight_reduce_kernel<false>), dim3(2 * D / 16), dim3(1024), 0, stream, part, nbq, nbk, D, dqw, dkw);
    return hipGetLastError();
}

extern "C" hipError_t dsa_launch_sigmoid_gate_fwd(const void *x, const void *gate, int64_t gate_tok, int64_t gate_head, int D,
                                                  int H, int64_t rows, void *y, hipStream_t stream) {
    const int64_t chunks = rows * H * D / 8;
    if (chunks == 0) return hipSuccess;
    const int nb = (int)((chunks + 255) / 256 > 16384 ? 16384 : (chunks + 255) / 256);
    hipLaunchKernelGGL(dsa_sigmoid_gate_fwd_kernel, dim3(nb), dim3(256), 0, stream, (const bf16_t *)x, (const bf16_t *)gate,
                       gate_tok, gate_head, D, H, rows, (bf16_t *)y);
    return hipGetLastError();
}
extern "C" hipError_t dsa_launch_sigmoid_gate_bwd(const void *gy, const void *x, const void *gate, int64_t gate_tok,
                                                  int64_t gate_head, int D, int H, int64_t rows, void *dx, void *dgate,
                                                  int64_t dgate_tok, int64_t dgate_head, hipStream_t stream) {
    const int64_t chunks = rows * H * D / 8;
    if (chunks == 0) return hipSuccess;
    const int nb = (int)((chunks + 255) / 256 > 16384 ? 16384 : (chunks + 255) / 256);
    hipLaunchKernelGGL(dsa_sigmoid_gate_bwd_kernel, dim3(nb), dim3(256), 0, stream, (const bf16_t *)gy, (const bf16_t *)x,
                       (const bf16_t *)gate, gate_tok, gate_head, D, H, rows, (bf16_t *)dx, (bf16_t *)dgate, dgate_tok,
                       dgate_head);
    return hipGetLastError();
}

// ---- several (T, width) bf16 tensors side by side in one row-major buffer: the gradients of a layer's projections, so that one
// GEMM gives all their weight gradients.  A source row of `width` elements goes to column dst_col in groups of `group` elements
// dst_group apart (the two halves of an interleaved projection).  A thread keeps its 16-byte column over the rows: the search for
// its source is done once, and four rows are in flight.  Bound by memory: 102 MB of gradients (8192 tokens, six projections), 38 us = 5.4 TB/s.
struct PackArgs { const bf16_t *src[8]; int width[8], group[8], dst_col[8], dst_group[8], n; };
__global__ __launch_bounds__(256) void dsa_pack_columns_kernel(PackArgs a, int T, bf16_t *__restrict__ dst, int64_t dst_row) {
    int c = (blockIdx.x * 256 + threadIdx.x) * 8, i = 0;
    while (i < a.n && c >= a.width[i]) c -= a.width[i++];
    if (i == a.n) return;
    const bf16_t *const src = a.src[i] + c;
    const int64_t w = a.width[i];
    bf16_t *const d = dst + a.dst_col[i] + c / a.group[i] * a.dst_group[i] + c % a.group[i];
    constexpr int U = 4;
    for (int t0 = blockIdx.y * U; t0 < T; t0 += gridDim.y * U) {
        u32x4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + min(t0 + u, T - 1) * w));
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t0 + u < T) *reinterpret_cast<u32x4 *>(d + (t0 + u) * dst_row) = x[u];
    }
}
extern "C" hipError_t dsa_launch_pack_columns(int n, const void *const *src, const int32_t *width, const int32_t *group, const int32_t *dst_col,
                                              const int32_t *dst_group, int T, void *dst, int64_t dst_row, hipStream_t stream) {
    PackArgs a;
    int64_t chunks = 0;
    a.n = n;
    for (int i = 0; i < n; ++i) {
        a.src[i] = (const bf16_t *)src[i];
        a.width[i] = width[i];
        a.group[i] = group[i];
        a.dst_col[i] = dst_col[i];
        a.dst_group[i] = dst_group[i];
        chunks += width[i] / 8;
    }
    const int rows = (T + 3) / 4;
    hipLaunchKernelGGL(dsa_pack_columns_kernel, dim3((unsigned)((chunks + 255) / 256), (unsigned)(rows < 2048 ? rows : 2048)), dim3(256), 0, stream, a, T,
                       (bf16_t *)dst, dst_row);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// fp32 operands on the bf16 kernels: x = hi + lo with hi = bf16(x), lo = bf16(x - hi), the parts stacked along
// head_dim into rows of 4*D bf16 so that the products of the stacked operands give back near-fp32 logits:
//   order 0: [hi, lo, hi, 0]  (q, v)        order 1: [hi, hi, lo, 0]  (k, dO)
// and the way back, out[r, :] = y[r, 0:D] + y[r, part*D:(part+1)*D] in fp32.  One thread per 4 elements.
// ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ void split_stack4(const float *__restrict__ x, int64_t i, int D, int order, bf16_t *__restrict__ y) {
    const int64_t r = i / (D / 4);
    const int c = (int)(i % (D / 4)) * 4;
    const f32x4 v = *reinterpret_cast<const f32x4 *>(x + r * D + c);
    const uint32_t h0 = pack2bf(v[0], v[1]), h1 = pack2bf(v[2], v[3]);
    const uint32_t l0 = pack2bf(v[0] - __uint_as_float(h0 << 16), v[1] - __uint_as_float(h0 & 0xffff0000u));
    const uint32_t l1 = pack2bf(v[2] - __uint_as_float(h1 << 16), v[3] - __uint_as_float(h1 & 0xffff0000u));
    bf16_t *o = y + r * 4 * D + c;
    const u32x2 hi = {h0, h1}, lo = {l0, l1}, z = {0u, 0u};
    *reinterpret_cast<u32x2 *>(o) = hi;
    *reinterpret_cast<u32x2 *>(o + D) = order ? hi : lo;
    *reinterpret_cast<u32x2 *>(o + 2 * D) = order ? lo : hi;
    *reinterpret_cast<u32x2 *>(o + 3 * D) = z;
}
__device__ __forceinline__ void split_combine4(const bf16_t *__restrict__ y, int64_t i, int D, int part, float *__restrict__ out) {
    const int64_t r = i / (D / 4);
    const int c = (int)(i % (D / 4)) * 4;
    const u32x2 a = *reinterpret_cast<const u32x2 *>(y + r * 4 * D + c);
    const u32x2 b = *reinterpret_cast<const u32x2 *>(y + r * 4 * D + part * D + c);
    const f32x4 o = {__uint_as_float(a[0] << 16) + __uint_as_float(b[0] << 16),
                     __uint_as_float(a[0] & 0xffff0000u) + __uint_as_float(b[0] & 0xffff0000u),
                     __uint_as_float(a[1] << 16) + __uint_as_float(b[1] << 16),
                     __uint_as_float(a[1] & 0xffff0000u) + __uint_as_float(b[1] & 0xffff0000u)};
    *reinterpret_cast<f32x4 *>(out + r * D + c) = o;
}
__global__ __launch_bounds__(256) void dsa_split_stack_kernel(const float *__restrict__ x, int64_t rows, int D, int order,
                                                               bf16_t *__restrict__ y) {
    const int64_t n4 = rows * (D / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) split_stack4(x, i, D, order, y);
}
__global__ __launch_bounds__(256) void dsa_split_combine_kernel(const bf16_t *__restrict__ y, int64_t rows, int D, int part,
                                                                 float *__restrict__ out) {
    const int64_t n4 = rows * (D / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) split_combine4(y, i, D, part, out);
}
// the three operands of one attention call in one launch: q-shaped (rows_q) first, then the two kv-shaped ones
__global__ __launch_bounds__(256) void dsa_split_stack_qkv_kernel(const float *__restrict__ q, const float *__restrict__ k,
                                                                   const float *__restrict__ v, int64_t rows_q, int64_t rows_kv,
                                                                   int D, bf16_t *__restrict__ yq, bf16_t *__restrict__ yk,
                                                                   bf16_t *__restrict__ yv) {
    const int64_t nq = rows_q * (D / 4), nkv = rows_kv * (D / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nq + 2 * nkv; i += (int64_t)gridDim.x * 256) {
        if (i < nq) split_stack4(q, i, D, 0, yq);
        else if (i < nq + nkv) split_stack4(k, i - nq, D, 1, yk);
        else split_stack4(v, i - nq - nkv, D, 0, yv);
    }
}
__global__ __launch_bounds__(256) void dsa_split_combine_qkv_kernel(const bf16_t *__restrict__ yq, const bf16_t *__restrict__ yk,
                                                                     const bf16_t *__restrict__ yv, int64_t rows_q,
                                                                     int64_t rows_kv, int D, float *__restrict__ dq,
                                                                     float *__restrict__ dk, float *__restrict__ dv) {
    const int64_t nq = rows_q * (D / 4), nkv = rows_kv * (D / 4);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nq + 2 * nkv; i += (int64_t)gridDim.x * 256) {
        if (i < nq) split_combine4(yq, i, D, 2, dq);
        else if (i < nq + nkv) split_combine4(yk, i - nq, D, 1, dk);
        else split_combine4(yv, i - nq - nkv, D, 2, dv);
    }
}
extern "C" hipError_t dsa_launch_split_stack(const float *x, int64_t rows, int D, int order, void *y, hipStream_t stream) {
    const int64_t n4 = rows * (D / 4);
    if (n4 == 0) return hipSuccess;
    const int nb = (int)((n4 + 255) / 256 > 8192 ? 8192 : (n4 + 255) / 256);
    hipLaunchKernelGGL(dsa_split_stack_kernel, dim3(nb), dim3(256), 0, stream, x, rows, D, order, (bf16_t *)y);
    return hipGetLastError();
}
extern "C" hipError_t dsa_launch_split_combine(const void *y, int64_t rows, int D, int part, float *out, hipStream_t stream) {
    const int64_t n4 = rows * (D / 4);
    if (n4 == 0) return hipSuccess;
    const int nb = (int)((n4 + 255) / 256 > 8192 ? 8192 : (n4 + 255) / 256);
    hipLaunchKernelGGL(dsa_split_combine_kernel, dim3(nb), dim3(256), 0, stream, (const bf16_t *)y, rows, D, part, out);
    return hipGetLastError();
}
extern "C" hipError_t dsa_launch_split_stack_qkv(const float *q, const float *k, const float *v, int64_t rows_q, int64_t rows_kv,
                                                 int D, void *yq, void *yk, void *yv, hipStream_t stream) {
    const int64_t n4 = (rows_q + 2 * rows_kv) * (D / 4);
    if (n4 == 0) return hipSuccess;
    const int nb = (int)((n4 + 255) / 256 > 8192 ? 8192 : (n4 + 255) / 256);
    hipLaunchKernelGGL(dsa_split_stack_qkv_kernel, dim3(nb), dim3(256), 0, stream, q, k, v, rows_q, rows_kv, D, (bf16_t *)yq,
                       (bf16_t *)yk, (bf16_t *)yv);
    return hipGetLastError();
}
extern "C" hipError_t dsa_launch_split_combine_qkv(const void *yq, const void *yk, const void *yv, int64_t rows_q, int64_t rows_kv,
                                                   int D, float *dq, float *dk, float *dv, hipStream_t stream) {
    const int64_t n4 = (rows_q + 2 * rows_kv) * (D / 4);
    if (n4 == 0) return hipSuccess;
    const int nb = (int)((n4 + 255) / 256 > 8192 ? 8192 : (n4 + 255) / 256);
    hipLaunchKernelGGL(dsa_split_combine_qkv_kernel, dim3(nb), dim3(256), 0, stream, (const bf16_t *)yq, (const bf16_t *)yk,
                       (const bf16_t *)yv, rows_q, rows_kv, D, dq, dk, dv);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// fp32 -> bf16 (round to nearest even, the hardware conversion) of three arrays in one launch: the indexer's inputs of
// an fp32 caller.  Four elements per thread; the last one to three of an array go one by one.
// ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ void round4_bf16(const float *__restrict__ x, int64_t i4, int64_t n, bf16_t *__restrict__ y) {
    const int64_t i = i4 * 4;
    if (i + 4 <= n) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(x + i);
        const u32x2 o = {pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
        *reinterpret_cast<u32x2 *>(y + i) = o;
    } else {
        for (int64_t j = i; j < n; ++j) y[j] = (bf16_t)x[j];
    }
}
__global__ __launch_bounds__(256) void dsa_round_bf16_x3_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                                 const float *__restrict__ c, int64_t na, int64_t nb, int64_t nc,
                                                                 bf16_t *__restrict__ ya, bf16_t *__restrict__ yb,
                                                                 bf16_t *__restrict__ yc) {
    const int64_t qa = (na + 3) / 4, qb = (nb + 3) / 4, qc = (nc + 3) / 4;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < qa + qb + qc; i += (int64_t)gridDim.x * 256) {
        if (i < qa) round4_bf16(a, i, na, ya);
        else if (i < qa + qb) round4_bf16(b, i - qa, nb, yb);
        else round4_bf16(c, i - qa - qb, nc, yc);
    }
}
extern "C" hipError_t dsa_launch_round_bf16_x3(const float *a, const float *b, const float *c, int64_t na, int64_t nb, int64_t nc,
                                               void *ya, void *yb, void *yc, hipStream_t stream) {
    const int64_t n4 = (na + 3) / 4 + (nb + 3) / 4 + (nc + 3) / 4;
    if (n4 == 0) return hipSuccess;
    const int nb_ = (int)((n4 + 255) / 256 > 8192 ? 8192 : (n4 + 255) / 256);
    hipLaunchKernelGGL(dsa_round_bf16_x3_kernel, dim3(nb_), dim3(256), 0, stream, a, b, c, na, nb, nc, (bf16_t *)ya, (bf16_t *)yb,
                       (bf16_t *)yc);
    return hipGetLastError();
}
