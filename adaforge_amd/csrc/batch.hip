// Batched prefill kernels for gfx950: up to kPassMax prompt tokens through a layer with every
// weight read once for the whole pass (crates/cuda-backend/src/batch.rs, kernels/ada/q4_batch.cu
// in the reference, 32 tokens there).  A layer's pass is a chain of launches: the input image of every
// token's GEMV input (batch_input_kernel, with the residual and RMSNorm prologues), the Q4_0 GEMM over
// all tokens (batch_gemm_kernel up to kBatchMax tokens, wide_gemm_kernel above; partial sums when the
// GEMM splits K across workgroups), and the attention of all tokens (batch_attention_kernel or
// wide_attention_kernel, after a pass that appends every token's K and V).  Above kBatchMax tokens a
// pass is bound by its products, which the wide kernels share out like any large matrix product; up to
// it by the weight stream.  512 tokens through six layers of the 12B shape: 14.3 ms in 16 passes of 32,
// 5.3 ms in one.
//
// Up to kBatchMax tokens each token's GEMM input is written as two fp16 halves per 32-element block: with u the block
// scaled by 2^(14 - e) (e = ilogb of the block's max |x|, so that |u| < 2^15), hi = fp16(u) and
// lo = fp16(u - hi), both rounded to nearest even; hi + lo holds u to about 2^-23 of the block's max.  The GEMM runs on the
// fp16 matrix cores with the tokens in the MFMA's M dimension: v_mfma_f32_16x16x32_f16 with A = the
// hi (then the lo) halves of 16 tokens over one 32-weight block (k) and B = the block's weights
// n - 8 of 16 rows as fp16 (exact: each nibble placed in the mantissa of 1024 + n, then 1032
// subtracted), both MFMAs accumulating into one fp32 tile, so D[t][r] = sum_j u_j(t) (n_rj - 8) with
// every product exact.  Each lane adds d_r 2^(e - 14) D[t][r] to its fp32 partial per block.
#include "device.h"

namespace af {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

namespace {

constexpr uint32_t kGemmThreads = 256;  // four waves splitting the blocks of the workgroup's K range
constexpr uint32_t kGemmTargetGrid = 512;

uint32_t padded_tokens(uint32_t T) { return (T + 15) / 16 * 16; }

// Work split of a GEMM: R row tiles per workgroup, S workgroups along K (partials summed by
// batch_reduce_kernel), so that about kGemmTargetGrid workgroups share the weight stream and each
// wave keeps at least two blocks.
struct GemmPlan {
    uint32_t R, S;
};
// The input image is read by every workgroup of a K range, R row tiles at a time, so R sets its
// reuse: up to 8 tiles (4 of each matrix of a gate/up pair) while at least 32 row groups remain.
GemmPlan gemm_plan(uint32_t rows, uint32_t blocks, bool pair) {
    const uint32_t tiles = (rows + 15) / 16, r_max = pair ? 4 : 8;
    uint32_t R = 1;
    while (R < r_max && tiles >= 64 * R) R *= 2;
    const uint32_t wgs = (tiles + R - 1) / R;
    uint32_t S = std::max<uint32_t>(1, std::min<uint32_t>(32, (kGemmTargetGrid + wgs - 1) / wgs));
    S = std::max<uint32_t>(1, std::min(S, blocks / 8));
    return GemmPlan{R, S};
}

}  // namespace

// ---- input images of a batch --------------------------------------------------------------------
//
// Image of K = 32 nb inputs for Tp tokens: hi [nb][Tp][32] fp16, then lo [nb][Tp][32] fp16, then
// [nb][Tp] floats 2^(e - 14) (0 for an all-zero block and for padding tokens).  A quad of threads
// writes one block, thread p of it elements 4 p .. + 3 and 16 + 4 p .. + 3 (v[0..3], v[4..7]): the
// eight that one lane of the wide GEMM's operand holds (wide_halves).

// x 2^sh as two fp16 halves: hi = f16(u), lo = f16(u - hi), packed in pairs (x0, x1).
__device__ __forceinline__ void split_pair(float x0, float x1, int sh, uint32_t& hi, uint32_t& lo) {
    const float u0 = ldexpf(x0, sh), u1 = ldexpf(x1, sh);
    const _Float16 h0 = (_Float16)u0, h1 = (_Float16)u1;
    const _Float16 l0 = (_Float16)(u0 - (float)h0), l1 = (_Float16)(u1 - (float)h1);
    hi = (uint32_t)__builtin_bit_cast(uint16_t, h0) | (uint32_t)__builtin_bit_cast(uint16_t, h1) << 16;
    lo = (uint32_t)__builtin_bit_cast(uint16_t, l0) | (uint32_t)__builtin_bit_cast(uint16_t, l1) << 16;
}

// The halves and the scale of block b of token t from the 8 elements v of part p (all four lanes of
// the quad take part).
__device__ __forceinline__ void block_halves(const float (&v)[8], uint32_t b, uint32_t p, uint32_t t, uint32_t Tp,
                                             _Float16* hi, _Float16* lo, float* inv) {
    float m, sum;
    quad_stats(v, m, sum);
    const int e = m > 0.0f ? ilogbf(m) : 0;
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) split_pair(v[2 * k], v[2 * k + 1], 14 - e, hw[k], lw[k]);
    const size_t at = ((size_t)b * Tp + t) * 32 + 4 * p;
    *reinterpret_cast<v2u*>(hi + at) = v2u{hw[0], hw[1]};
    *reinterpret_cast<v2u*>(hi + at + 16) = v2u{hw[2], hw[3]};
    *reinterpret_cast<v2u*>(lo + at) = v2u{lw[0], lw[1]};
    *reinterpret_cast<v2u*>(lo + at + 16) = v2u{lw[2], lw[3]};
    if (p == 0) inv[(size_t)b * Tp + t] = m > 0.0f ? ldexpf(1.0f, e - 14) : 0.0f;
}

// Part p of block b of token t into the wide GEMM's image of G 16-token groups, scaled by 2^sh: the
// halves of one operand lane, in the order in which a dword of code bytes unpacks (nibbles_f16).
__device__ __forceinline__ void wide_halves(const float (&v)[8], int sh, uint32_t b, uint32_t p, uint32_t t, uint32_t G,
                                            v4u* img) {
    uint32_t h0, h1, h2, h3, l0, l1, l2, l3;
    split_pair(v[0], v[2], sh, h0, l0);
    split_pair(v[4], v[6], sh, h1, l1);
    split_pair(v[1], v[3], sh, h2, l2);
    split_pair(v[5], v[7], sh, h3, l3);
    v4u* at = img + ((size_t)b * G + t / 16) * 128 + 16 * p + t % 16;
    at[0] = v4u{h0, h1, h2, h3};
    at[64] = v4u{l0, l1, l2, l3};
}

// One workgroup per token t < Tp (tokens T..Tp-1 write zeros).  The input vector of the GEMV that
// follows:
//   BI_PLAIN: x_t (f32(rms(x_t) w_n) with w_n);
//   BI_RESID: v_t = (f32(rms(x_t) w_a) + res_t) * scale (w_a null: (x_t + res_t) * scale), stored to
//             x_out_t (the residual stream), then f32(rms(v_t) w_n);
//   BI_EMBED: v_t = table row ids[pos0 + t] * emb_scale, stored to x_out_t, then f32(rms(v_t) w_n).
// RMSNorm sums of squares and products in double, f32 results (crates/domain/src/rms_norm.rs:24-41).
// Thread j holds octets j, j + 512, ... (NO of them) in registers (an octet: part p of a block, two
// float4), and every global load of the token (x, res and both norm weights) is issued before the
// first reduction, so the kernel waits for memory once.
// PS: x comes from in.parts split-K partial planes (NO == 1 only).
// WIDE: the wide GEMM's image, one scale per token; no padding tokens are written (their rows of the
// product are never stored).  Workgroup b takes token (b % 8) ceil(T / 8) + b / 8, so that the 16
// tokens whose halves share a 256-byte run of the image are mostly written through one XCD's L2.
template <int NO, bool PS, bool WIDE>
__global__ __launch_bounds__(512) void batch_input_kernel(BatchIn in) {
    extern __shared__ __align__(16) float xs[];  // [K], BI_EMBED only
    __shared__ double red[8];
    __shared__ float redf[8];
    const uint32_t tid = threadIdx.x, K = in.K, nb = K / 32, no = K / 8, Tp = gridDim.x;
    const uint32_t t = WIDE ? blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    _Float16* hi = reinterpret_cast<_Float16*>(in.img);
    _Float16* lo = hi + (size_t)nb * Tp * 32;
    float* inv = reinterpret_cast<float*>(lo + (size_t)nb * Tp * 32);
    const uint32_t WG = wide_groups(in.T);
    if constexpr (WIDE) inv = reinterpret_cast<float*>(in.img + (size_t)nb * WG * 2048);
    if (WIDE && t >= in.T) return;
    if (t >= in.T) {
        for (uint32_t o = tid; o < nb * 4; o += blockDim.x) {
            const uint32_t b = o >> 2, p = o & 3;
            const size_t at = ((size_t)b * Tp + t) * 32 + 8 * p;
            *reinterpret_cast<v4u*>(hi + at) = v4u{0u, 0u, 0u, 0u};
            *reinterpret_cast<v4u*>(lo + at) = v4u{0u, 0u, 0u, 0u};
            if (p == 0) inv[(size_t)b * Tp + t] = 0.0f;
        }
        return;
    }
    const bool resid = in.mode == BI_RESID, embed = in.mode == BI_EMBED;
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 x[NO][2], r[NO][2], wa[NO][2], wn[NO][2];
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const uint32_t o = tid + 512 * j, i0 = 8 * (o >> 2) + (o & 3), i1 = i0 + 4;  // its float4
        x[j][0] = x[j][1] = r[j][0] = r[j][1] = wa[j][0] = wa[j][1] = wn[j][0] = wn[j][1] = z4;
        if (o < no) {
            if constexpr (PS) {
                // every plane's loads issued first, then the sums in split order
                const float* p0 = in.part + (size_t)t * in.part_row;
                const size_t plane = (size_t)in.part_tp * in.part_row;
                float4 pv[kDeferParts][2];
#pragma unroll
                for (int k = 0; k < (int)kDeferParts; ++k) {
                    if ((uint32_t)k < in.parts) {
                        pv[k][0] = reinterpret_cast<const float4*>(p0 + k * plane)[i0];
                        pv[k][1] = reinterpret_cast<const float4*>(p0 + k * plane)[i1];
                    }
                }
                x[j][0] = pv[0][0];
                x[j][1] = pv[0][1];
#pragma unroll
                for (int k = 1; k < (int)kDeferParts; ++k) {
                    if ((uint32_t)k < in.parts) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            x[j][h].x += pv[k][h].x;
                            x[j][h].y += pv[k][h].y;
                            x[j][h].z += pv[k][h].z;
                            x[j][h].w += pv[k][h].w;
                        }
                    }
                }
            } else if (!embed) {
                const float4* p = reinterpret_cast<const float4*>(in.x + (size_t)t * in.stride);
                x[j][0] = p[i0];
                x[j][1] = p[i1];
            }
            if (resid) {
                const float4* p = reinterpret_cast<const float4*>(in.res + (size_t)t * in.stride);
                r[j][0] = p[i0];
                r[j][1] = p[i1];
                if (in.w_a) {
                    wa[j][0] = reinterpret_cast<const float4*>(in.w_a)[i0];
                    wa[j][1] = reinterpret_cast<const float4*>(in.w_a)[i1];
                }
            }
            if (in.w_n) {
                wn[j][0] = reinterpret_cast<const float4*>(in.w_n)[i0];
                wn[j][1] = reinterpret_cast<const float4*>(in.w_n)[i1];
            }
        }
    }
    if (embed) {
        embed_row_at(in.table, gp(in.ids)[in.pos0 + t], in.emb_scale, xs, tid, blockDim.x);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const uint32_t o = tid + 512 * j, i0 = 8 * (o >> 2) + (o & 3);
            if (o < no) {
                x[j][0] = reinterpret_cast<const float4*>(xs)[i0];
                x[j][1] = reinterpret_cast<const float4*>(xs)[i0 + 4];
            }
        }
    }
    if (resid) {
        double ra = 1.0;
        if (in.w_a) {
            double sa = 0.0;
#pragma unroll
            for (int j = 0; j < NO; ++j) sa += sq4(x[j][0]) + sq4(x[j][1]);
            ra = inv_rms(block_sum_d(sa, red), K, in.eps_a);
        }
#pragma unroll
        for (int j = 0; j < NO; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                x[j][h] = resid4(in.w_a ? norm4(x[j][h], ra, wa[j][h]) : x[j][h], r[j][h], in.scale);
    }
    if (in.mode != BI_PLAIN) {
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const uint32_t o = tid + 512 * j, i0 = 8 * (o >> 2) + (o & 3);
            if (o >= no) continue;
            float4* xo = reinterpret_cast<float4*>(in.x_out + (size_t)t * in.stride);
            xo[i0] = x[j][0];
            xo[i0 + 4] = x[j][1];
            if (in.snap) {
                float* sp = in.snap + (size_t)t * in.snap_stride + 4 * i0;
                const float* v = reinterpret_cast<const float*>(&x[j][0]);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    sp[k] = v[k];
                    sp[16 + k] = v[4 + k];
                }
            }
        }
    }
    double rn = 1.0;
    if (in.w_n) {
        double ss = 0.0;
#pragma unroll
        for (int j = 0; j < NO; ++j) ss += sq4(x[j][0]) + sq4(x[j][1]);
        rn = inv_rms(block_sum_d(ss, red), K, in.eps_n);
    }
    // the GEMV's input, in place of x; a quad of threads holds one 32-element block (no is a multiple
    // of 4: whole quads take part)
    float v[NO][8];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < NO; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 u = in.w_n ? norm4(x[j][h], rn, wn[j][h]) : x[j][h];
            v[j][4 * h] = u.x;
            v[j][4 * h + 1] = u.y;
            v[j][4 * h + 2] = u.z;
            v[j][4 * h + 3] = u.w;
#pragma unroll
            for (int k = 0; k < 4; ++k) m = fmaxf(m, fabsf(v[j][4 * h + k]));
        }
    int e = 0;
    if constexpr (WIDE) {
        m = block_max_f(m, redf);
        e = m > 0.0f ? ilogbf(m) : 0;
        if (tid == 0) inv[t] = m > 0.0f ? ldexpf(1.0f, e - 14) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const uint32_t o = tid + 512 * j;
        if (o >= no) continue;
        if constexpr (WIDE) wide_halves(v[j], 14 - e, o >> 2, o & 3, t, WG, reinterpret_cast<v4u*>(in.img));
        else block_halves(v[j], o >> 2, o & 3, t, Tp, hi, lo, inv);
    }
}

// BI_PLAIN inputs without a norm: one thread per 8-element octet, grid (Tp, octets / 256).  PS: the
// input is gelu(gate) * up from a gate/up pair's deferred split-K partials.
template <bool PS>
__global__ __launch_bounds__(256) void batch_plain_input_kernel(BatchIn in) {
    const uint32_t t = blockIdx.x, o = blockIdx.y * 256 + threadIdx.x, nb = in.K / 32, Tp = gridDim.x;
    if (o >= nb * 4) return;  // whole quads: nb * 4 is a multiple of 4
    const uint32_t i0 = 8 * (o >> 2) + (o & 3);  // the octet's float4: i0 and i0 + 4
    _Float16* hi = reinterpret_cast<_Float16*>(in.img);
    _Float16* lo = hi + (size_t)nb * Tp * 32;
    float* inv = reinterpret_cast<float*>(lo + (size_t)nb * Tp * 32);
    float v[8];
    if (PS && t < in.T) {
        // every plane's loads first, then each matrix's sums in split order, then gelu(gate) * up
        const float* p0 = in.part + (size_t)t * in.part_row;
        const size_t plane = (size_t)in.part_tp * in.part_row;
        float4 pv[kDeferPairParts][2][2];
#pragma unroll
        for (int k = 0; k < (int)kDeferPairParts; ++k)
            if ((uint32_t)k < in.parts)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int h = 0; h < 2; ++h) pv[k][q][h] = reinterpret_cast<const float4*>(p0 + (2 * k + q) * plane)[i0 + 4 * h];
        float s[2][8];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                s[q][4 * h] = pv[0][q][h].x;
                s[q][4 * h + 1] = pv[0][q][h].y;
                s[q][4 * h + 2] = pv[0][q][h].z;
                s[q][4 * h + 3] = pv[0][q][h].w;
            }
#pragma unroll
        for (int k = 1; k < (int)kDeferPairParts; ++k)
            if ((uint32_t)k < in.parts)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        s[q][4 * h] += pv[k][q][h].x;
                        s[q][4 * h + 1] += pv[k][q][h].y;
                        s[q][4 * h + 2] += pv[k][q][h].z;
                        s[q][4 * h + 3] += pv[k][q][h].w;
                    }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = gelu_mul(s[0][i], s[1][i]);
    } else if (t < in.T) {
        const float4* x = reinterpret_cast<const float4*>(in.x + (size_t)t * in.stride);
        const float4 u0 = x[i0], u1 = x[i0 + 4];
        v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w;
        v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = 0.0f;
    }
    block_halves(v, o >> 2, o & 3, t, Tp, hi, lo, inv);
}

// ---- Q4_0 GEMM over a batch ---------------------------------------------------------------------

namespace {

// A block's input operands for a wave: the hi and lo halves of its G token groups (lane l: token
// 16 g + l % 16, elements 8 (l / 16) .. + 7) and the block scales of tokens 16 g + 4 (l / 16) + e
// (the lane's outputs).  They come from L2 (the image is shared by all
// workgroups) and are loaded one block ahead.
template <int G>
struct InOps {
    v4u hi[G], lo[G];
    v4f sc[G];  // the block scales 2^(e - 14) of the four tokens whose outputs the lane folds
};

// A block's weights for R row tiles of P matrices (lane l: row l % 16, bytes 8 ((l / 16) & 1) .. + 7 of
// the block's 16 code bytes, and the row's fp16 scale).  They stream from HBM and are loaded
// kCodeAhead blocks ahead.
template <int P, int R>
struct WOps {
    uint2 code[R][P];
    uint16_t d[R][P];
};

// weight blocks in flight per wave: 8, or 2 when a block spans 4 or more tiles
template <int P, int R>
constexpr int code_ahead() { return R * P >= 4 ? 2 : 8; }

template <int G>
__device__ __forceinline__ void load_in(InOps<G>& o, const BatchGemm& a, uint32_t b, uint32_t lane) {
    constexpr uint32_t Tp = 16 * G;
    const uint32_t m = lane & 15, kq = lane >> 4;
    const _Float16* hi = reinterpret_cast<const _Float16*>(a.img);
    const _Float16* lo = hi + (size_t)a.w.blocks * Tp * 32;
    const float* inv = reinterpret_cast<const float*>(lo + (size_t)a.w.blocks * Tp * 32);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const size_t at = ((size_t)b * Tp + 16 * g + m) * 32 + 8 * kq;
        o.hi[g] = *gp(reinterpret_cast<const v4u*>(hi + at));
        o.lo[g] = *gp(reinterpret_cast<const v4u*>(lo + at));
        o.sc[g] = *gp(reinterpret_cast<const v4f*>(inv + (size_t)b * Tp + 16 * g + 4 * kq));
    }
}

template <int P, int R>
__device__ __forceinline__ void load_w(WOps<P, R>& o, const BatchGemm& a, uint32_t b, uint32_t rt0, uint32_t last_tile,
                                       uint32_t lane) {
    const uint32_t m = lane & 15, kq = lane >> 4;
    const uint32_t per_tile = a.w.nst * 4;  // block records per row tile (tiled layout, Q4View)
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t rec = (size_t)min(rt0 + r, last_tile) * per_tile + b;
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const Q4View& w = q ? a.w2 : a.w;
            o.code[r][q] = ld_stream(reinterpret_cast<const uint2*>(w.codes + rec * 256 + m * 16 + 8 * (kq & 1)));
            o.d[r][q] = gp(w.scales)[rec * 16 + m];
        }
    }
}

// Four nibbles (one per byte of c) as fp16 (n - 8), in two pairs: n into the mantissa of 1024 + n
// (0x6400 | n), then 1032 subtracted, exactly.
__device__ __forceinline__ void nibbles_f16(uint32_t c, v2h& p0, v2h& p1) {
    const v2h bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    p0 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0u, c, 0x0c010c00u) | 0x64006400u) - bias;
    p1 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0u, c, 0x0c030c02u) | 0x64006400u) - bias;
}

template <int P, int G, int R>
__device__ __forceinline__ void mfma_block(const InOps<G>& x, const WOps<P, R>& w, uint32_t kq,
                                           float (&acc)[R][P][G][4]) {
    const uint32_t sh = kq >= 2 ? 4u : 0u;  // k 0..15: low nibbles, 16..31: high nibbles
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < P; ++q) {
            v2h f0, f1, f2, f3;
            nibbles_f16((w.code[r][q].x >> sh) & 0x0F0F0F0Fu, f0, f1);
            nibbles_f16((w.code[r][q].y >> sh) & 0x0F0F0F0Fu, f2, f3);
            const v8h B = {f0.x, f0.y, f1.x, f1.y, f2.x, f2.y, f3.x, f3.y};
            const float d = h2f(w.d[r][q]);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                v4f D = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x.hi[g]), B, zero, 0, 0, 0);
                D = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x.lo[g]), B, D, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][q][g][e] = fmaf(d * x.sc[g][e], D[e], acc[r][q][g][e]);
            }
        }
}

template <int P>
__device__ __forceinline__ void gemm_epilogue(const BatchGemm& a, uint32_t t, uint32_t row, const float (&v)[P]) {
    float* y = a.y + (size_t)t * a.y_stride + row;
    if constexpr (P == 2) *y = gelu_mul(v[0], v[1]);
    else if (a.add) *y = __fadd_rn(v[0], a.add[(size_t)t * a.y_stride + row]);
    else *y = v[0];
}

}  // namespace

// Grid (ceil(tiles / R), S): workgroup (x, s) takes row tiles R x .. R x + R - 1 (for a gate/up pair,
// those tiles of both matrices) over K range s of S; its four waves split the range's blocks and add
// their partials in LDS in wave order.  Each wave streams its blocks through a two-stage register
// pipeline (the next block's loads in flight while the current block's MFMAs run).  With S = 1 the
// workgroup writes y; otherwise it writes its partials for batch_reduce_kernel.
template <int P, int G, int R>
__global__ __launch_bounds__(256) void batch_gemm_kernel(BatchGemm a) {
    constexpr uint32_t Tp = 16 * G;
    __shared__ float red[4][R][P][Tp][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = wave_id(), kq = lane >> 4;
    const uint32_t tiles = (a.w.rows + 15) / 16, rt0 = blockIdx.x * R, S = gridDim.y, split = blockIdx.y;
    const uint32_t nb = a.w.blocks;
    const uint32_t s0 = nb * split / S, s1 = nb * (split + 1) / S;
    const uint32_t b0 = s0 + (s1 - s0) * wave / 4, b1 = s0 + (s1 - s0) * (wave + 1) / 4;
    float acc[R][P][G][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < P; ++q)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][q][g][e] = 0.0f;
    // weights kCodeAhead blocks ahead in a register ring, inputs one block ahead (ping-pong)
    constexpr int kCodeAhead = code_ahead<P, R>();
    WOps<P, R> wr[kCodeAhead];
    InOps<G> xi[2];
    const uint32_t last_b = nb - 1;
#pragma unroll
    for (int u = 0; u < kCodeAhead; ++u) load_w(wr[u], a, min(b0 + u, last_b), rt0, tiles - 1, lane);
    if (b0 < b1) load_in(xi[0], a, b0, lane);
    for (uint32_t b = b0; b < b1; b += kCodeAhead) {
#pragma unroll
        for (int u = 0; u < kCodeAhead; ++u) {
            const uint32_t bb = b + u;
            if (bb >= b1) break;
            if (bb + 1 < b1) load_in(xi[(u + 1) & 1], a, bb + 1, lane);
            mfma_block(xi[u & 1], wr[u], kq, acc);
            load_w(wr[u], a, min(bb + kCodeAhead, last_b), rt0, tiles - 1, lane);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < P; ++q)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int e = 0; e < 4; ++e) red[wave][r][q][16 * g + 4 * kq + e][lane & 15] = acc[r][q][g][e];
    __syncthreads();
    const size_t prow = (size_t)tiles * 16;
    for (uint32_t i = tid; i < R * Tp * 16; i += kGemmThreads) {
        const uint32_t r = i / (Tp * 16), t = (i / 16) % Tp, n = i & 15;
        const uint32_t tile = rt0 + r, row = tile * 16 + n;
        if (tile >= tiles || t >= a.T) continue;
        float v[P];
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = ((red[0][r][q][t][n] + red[1][r][q][t][n]) + red[2][r][q][t][n]) + red[3][r][q][t][n];
        if (S > 1) {
#pragma unroll
            for (int q = 0; q < P; ++q) a.part[((size_t)(split * P + q) * Tp + t) * prow + row] = v[q];
        } else if (row < a.w.rows) {
            gemm_epilogue<P>(a, t, row, v);
        }
    }
}

// y from the S split-K partials of batch_gemm_kernel, summed in split order; one thread per (t, row).
template <int P>
__global__ __launch_bounds__(256) void batch_reduce_kernel(BatchGemm a, uint32_t S, uint32_t Tp) {
    const uint32_t rows = a.w.rows, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.T * rows) return;
    const uint32_t t = i / rows, row = i % rows;
    const size_t prow = (size_t)(rows + 15) / 16 * 16;
    float v[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        float s = a.part[((size_t)q * Tp + t) * prow + row];
        for (uint32_t k = 1; k < S; ++k) s += a.part[((size_t)(k * P + q) * Tp + t) * prow + row];
        v[q] = s;
    }
    gemm_epilogue<P>(a, t, row, v);
}

// ---- Q4_0 GEMM over a wide pass -------------------------------------------------------------------
//
// y[t][r] = sum_b d_rb sum_j (n_rbj - 8) x_tbj for more than kBatchMax tokens.  A workgroup of four
// waves takes M = 64 WM tokens x 64 WN rows (WM WN = 4; a wave 64 x 64: 4 x 4 MFMA tiles) over K range
// `split`, one 32-weight block (one MFMA depth) per step: the tokens' halves are copied from the
// image, which is laid out as the MFMAs read it, and the weights unpacked once per workgroup, both
// into LDS, double buffered; step s + 1's are written while step s is multiplied, and step s + 2's
// loads are in flight.  The block's d_rb differs from the next one's, so each block's 16 x 16
// products are folded into fp32 sums on their own (one FMA per product and lane: half as many VALU
// cycles as the two MFMAs take; the token's scale waits for the epilogue, so that the fold has no other
// factor).  Sums run over kWideChain blocks, then join a total, so that no chain of fp32 additions is
// longer than K / 32 / kWideChain + kWideChain.
//
// Work items (split, row group, token tile), token tile fastest, go to the XCDs in contiguous
// shares (workgroup b runs on XCD b % 8), so that the workgroups that unpack the same weights share
// an L2.
constexpr uint32_t kWideChain = 8;

// One lane's eight fp16 weights n - 8 of a block from the dword of its code bytes 4 q .. 4 q + 3: the
// nibbles' bits in the mantissa of 1024 + n (or 1024 + 16 n), then 1032 subtracted (or scaled by 1/16
// and 72 subtracted), exactly.  Weights 4 q + {0, 2}, 16 + 4 q + {0, 2}, 4 q + {1, 3}, 16 + 4 q + {1, 3}.
__device__ __forceinline__ v4u unpack_dword(uint32_t c) {
    const v2h bias = {(_Float16)1032.0f, (_Float16)1032.0f}, hb = {(_Float16)-72.0f, (_Float16)-72.0f},
              sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t c8 = c >> 8;
    const v2h a = __builtin_bit_cast(v2h, (c & 0x000F000Fu) | 0x64006400u) - bias;
    const v2h b = __builtin_elementwise_fma(__builtin_bit_cast(v2h, (c & 0x00F000F0u) | 0x64006400u), sixteenth, hb);
    const v2h e = __builtin_bit_cast(v2h, (c8 & 0x000F000Fu) | 0x64006400u) - bias;
    const v2h f = __builtin_elementwise_fma(__builtin_bit_cast(v2h, (c8 & 0x00F000F0u) | 0x64006400u), sixteenth, hb);
    return v4u{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, e),
               __builtin_bit_cast(uint32_t, f)};
}

template <int WM, int P>
__global__ __launch_bounds__(256, 2) void wide_gemm_kernel(BatchGemm a, uint32_t S, uint32_t mtiles, uint32_t ngroups) {
    constexpr int WN = 4 / WM, MG = 4 * WM, NT = 4 * WN;  // 16-token groups and 16-row tiles of the workgroup
    __shared__ v4u As[2][MG * 128];  // [token group][hi, lo][64 lanes]
    __shared__ v4u Bs[2][NT * 64];   // [row tile][64 lanes]
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = wave_id(), r = lane & 15, q = lane >> 4;
    const uint32_t wm = wave / WN, wn = wave % WN;
    const uint32_t total = mtiles * ngroups * S, per = gridDim.x / 8;
    const uint32_t item = blockIdx.x % 8 * per + blockIdx.x / 8;
    if (item >= total) return;
    const uint32_t mt0 = item % mtiles, ng = item / mtiles % ngroups, split = item / mtiles / ngroups;
    const uint32_t nb = a.w.blocks, G = mtiles * MG, tiles = (a.w.rows + 15) / 16;
    const uint32_t b0 = nb * split / S, b1 = nb * (split + 1) / S;
    // row tile i of the workgroup (of wave i / 4): a gate/up pair's waves hold two tiles of each matrix,
    // alternating, so that a lane holds both products of a row
    auto tile_of = [&](uint32_t i) { return P == 2 ? ng * (NT / 2) + i / 4 * 2 + (i % 4) / 2 : ng * NT + i; };
    auto mat_of = [&](uint32_t i) -> const Q4View& { return P == 2 && (i & 1) ? a.w2 : a.w; };

    const v4u* img = reinterpret_cast<const v4u*>(a.img) + (size_t)mt0 * MG * 128 + tid;
    v4u sa[MG / 2];    // step s + 1's halves on their way to LDS
    uint32_t sc[WN];   // and code dwords of the row tiles this wave unpacks (wave WN .. + WN - 1)
    uint16_t dn[4];    // the next step's scales of the lane's rows
    const uint8_t* cp[WN];
    const uint16_t* dp[4];
#pragma unroll
    for (int i = 0; i < WN; ++i) {
        const uint32_t k = wave * WN + i;
        cp[i] = mat_of(k).codes + (size_t)min(tile_of(k), tiles - 1) * a.w.nst * 1024 + r * 16 + q * 4;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t k = wn * 4 + i;
        dp[i] = mat_of(k).scales + (size_t)min(tile_of(k), tiles - 1) * a.w.nst * 64 + r;
    }
    auto load = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < MG / 2; ++i) sa[i] = *gp(img + (size_t)b * G * 128 + 256 * i);
#pragma unroll
        for (int i = 0; i < WN; ++i) sc[i] = *gp(reinterpret_cast<const uint32_t*>(cp[i] + (size_t)b * 256));
    };
    auto load_d = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) dn[i] = gp(dp[i])[(size_t)b * 16];
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < MG / 2; ++i) As[buf][tid + 256 * i] = sa[i];
#pragma unroll
        for (int i = 0; i < WN; ++i) Bs[buf][(wave * WN + i) * 64 + lane] = unpack_dword(sc[i]);
    };
    v4f acc[4][4], tot[4][4];
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = tot[m][n] = zero;

    const uint32_t last = b1 - 1;
    load(b0);
    load_d(b0);
    stage(0);
    load(min(b0 + 1, last));
    __syncthreads();
    for (uint32_t b = b0; b < b1; ++b) {
        const int buf = (b - b0) & 1;
        float d[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) d[n] = h2f(dn[n]);
        v8h ah[4], al[4], bw[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            ah[m] = __builtin_bit_cast(v8h, As[buf][(wm * 4 + m) * 128 + lane]);
            al[m] = __builtin_bit_cast(v8h, As[buf][(wm * 4 + m) * 128 + 64 + lane]);
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) bw[n] = __builtin_bit_cast(v8h, Bs[buf][(wn * 4 + n) * 64 + lane]);
        stage(buf ^ 1);
        load(min(b + 2, last));
        load_d(min(b + 1, last));
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            v4f D[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) D[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[m], bw[n], zero, 0, 0, 0);
#pragma unroll
            for (int m = 0; m < 4; ++m) D[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[m], bw[n], D[m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][n][e] = fmaf(d[n], D[m][e], acc[m][n][e]);
        }
        if (((b - b0) & (kWideChain - 1)) == kWideChain - 1) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    tot[m][n] += acc[m][n];
                    acc[m][n] = zero;
                }
        }
        __syncthreads();
    }

    // lane: rows r of its tiles, tokens 4 q + e of its groups
    const float* inv = reinterpret_cast<const float*>(a.img + (size_t)nb * G * 2048);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const uint32_t t0 = (mt0 * MG + wm * 4 + m) * 16 + 4 * q;
        const v4f s = *gp(reinterpret_cast<const v4f*>(inv + t0));
#pragma unroll
        for (int n = 0; n < 4; n += P) {
            const uint32_t row = tile_of(wn * 4 + n) * 16 + r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t t = t0 + e;
                if (t >= a.T || row >= a.w.rows) continue;
                const float v = (tot[m][n][e] + acc[m][n][e]) * s[e];
                if constexpr (P == 2) {
                    const float u = (tot[m][n + 1][e] + acc[m][n + 1][e]) * s[e];
                    a.y[(size_t)t * a.y_stride + row] = gelu_mul(v, u);
                } else if (S > 1) {
                    a.part[((size_t)split * G * 16 + t) * (tiles * 16) + row] = v;
                } else {
                    a.y[(size_t)t * a.y_stride + row] = v;
                }
            }
        }
    }
}

// ---- attention of a batch ----------------------------------------------------------------------
//
// Grid (nchunks, kv_heads, query tiles): workgroup (c, h, j) takes query tile ~j of KV head h (queries
// i = t group + g of its tokens t and query heads h group + g, 16 per tile; the last tiles, which
// see the most keys, start first) against chunk c of the keys that the tile's tokens see, streamed in
// sub-chunks of KC keys through LDS, with an online softmax; a single chunk writes the output itself.  Both products run
// on the fp16 matrix cores (v_mfma_f32_16x16x32_f16, fp32 accumulation): the cached K and V are
// fp16 already, and the fp32 queries and probabilities enter as fp16 pairs hi + lo (hi = f16(x),
// lo = f16(x - hi)) after scaling by a power of two (queries to below 32 in magnitude, probabilities
// by 2^14), so each operand keeps about 22 significant bits and every product is exact in fp32.

namespace {


__device__ __forceinline__ void split_f16(float x, _Float16& hi, _Float16& lo) {
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);  // exact in fp32: hi is the nearest fp16 to x
}

// Maximum over the four lanes l % 16 equal, left in each (row_total's maximum).
__device__ __forceinline__ float lanes4_max(float v) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

}  // namespace

template <int D, int KC>
__global__ __launch_bounds__(256) void batch_attention_kernel(BatchAttn a) {
    constexpr int KP = D + 8;         // row stride of K and of the query planes (halves)
    constexpr int VP = KC + 8;        // row stride of V^T and of the probability planes (halves)
    constexpr int KT = KC / 16;       // 16-key score tiles
    constexpr int DH = 4 / KT;        // head-width parts per score tile (four waves)
    constexpr int DS = D / 32 / DH;   // MFMA steps per part
    constexpr int NT = D / 64;        // 16-channel output tiles per wave
    __shared__ __align__(16) _Float16 qh[16 * KP], ql[16 * KP];
    __shared__ __align__(16) _Float16 ks[KC * KP];
    __shared__ __align__(16) _Float16 vt[D * VP];
    __shared__ __align__(16) _Float16 ph[16 * VP], pl[16 * VP];
    __shared__ float sc[DH][16][KC];
    __shared__ float qscale[16], mrun[16], lrun[16], alpha[16];
    __shared__ int tok[16], lo_q[16], hi_q[16];

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 15, kq = lane >> 4;
    const uint32_t c = blockIdx.x, h = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;
    const uint32_t q_heads = a.kv_heads * a.group, nq = a.T * a.group;
    if (tid < 16) {
        const uint32_t qi = 16 * qt + tid;
        const bool ok = qi < nq;
        const int p = (int)(a.pos0 + (ok ? qi / a.group : 0));
        tok[tid] = ok ? (int)(qi / a.group) : -1;
        hi_q[tid] = ok ? p : -1;
        lo_q[tid] = a.window ? max(0, p + 1 - (int)a.window) : 0;
        mrun[tid] = -INFINITY;
        lrun[tid] = 0.0f;
    }
    // the tile's queries as scaled fp16 pairs (wave w: rows 4 w .. 4 w + 3)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t r = 4 * wave + i, qi = 16 * qt + r;
        float v[D / 64];
        const bool ok = qi < nq;
        const float* src = a.q + ((size_t)(ok ? qi / a.group : 0) * q_heads + h * a.group + qi % a.group) * D;
        float mx = 0.0f;
#pragma unroll
        for (int j = 0; j < D / 64; ++j) {
            v[j] = ok ? src[lane + 64 * j] : 0.0f;
            mx = fmaxf(mx, fabsf(v[j]));
        }
        mx = wave_max(mx);
        const float s = mx > 0.0f ? ldexpf(1.0f, 4 - ilogbf(mx)) : 1.0f;  // |q s| < 32
#pragma unroll
        for (int j = 0; j < D / 64; ++j) split_f16(v[j] * s, qh[r * KP + lane + 64 * j], ql[r * KP + lane + 64 * j]);
        if (lane == 0) qscale[r] = 1.0f / s;
    }
    // the keys the tile's first token to its last sees, in whole sub-chunks per chunk (a chunk past the
    // end is empty: maximum -inf, sums 0)
    const uint32_t t_lo = 16 * qt / a.group, t_hi = min(a.T - 1, (16 * qt + 15) / a.group);
    const uint32_t klo = a.window ? (uint32_t)max(0, (int)(a.pos0 + t_lo + 1) - (int)a.window) : 0u;
    const uint32_t khi = a.pos0 + t_hi + 1;
    const uint32_t span = ((khi - klo + KC - 1) / KC + a.nchunks - 1) / a.nchunks * KC;
    const uint32_t k_begin = klo + c * span, k_end = min(k_begin + span, khi);
    v4f acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    for (uint32_t k0 = k_begin; k0 < k_end; k0 += KC) {
        __syncthreads();  // the last sub-chunk's K, V^T, probabilities and alpha are read
        const uint32_t kn = min((uint32_t)KC, k_end - k0);
        for (uint32_t i = tid; i < KC * D / 8; i += 256) {  // K rows, 16-byte pieces
            const uint32_t row = i / (D / 8), pc = i % (D / 8);
            v4u val = {0u, 0u, 0u, 0u};
            if (row < kn) val = *gp(reinterpret_cast<const v4u*>(a.kcache + ((size_t)h * a.ring + (k0 + row) % a.ring) * D + 8 * pc));
            *reinterpret_cast<v4u*>(ks + row * KP + 8 * pc) = val;
        }
        for (uint32_t i = tid; i < KC / 2 * (D / 8); i += 256) {  // V rows 2j, 2j + 1 -> V^T
            const uint32_t j = i / (D / 8), pc = i % (D / 8);
            v4u v0 = {0u, 0u, 0u, 0u}, v1 = {0u, 0u, 0u, 0u};
            if (2 * j < kn)
                v0 = *gp(reinterpret_cast<const v4u*>(a.vcache + ((size_t)h * a.ring + (k0 + 2 * j) % a.ring) * D + 8 * pc));
            if (2 * j + 1 < kn)
                v1 = *gp(reinterpret_cast<const v4u*>(a.vcache + ((size_t)h * a.ring + (k0 + 2 * j + 1) % a.ring) * D + 8 * pc));
            const uint32_t w0[4] = {v0.x, v0.y, v0.z, v0.w}, w1[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {  // channel 8 pc + e: (key 2j, key 2j + 1)
                const uint32_t d = (e & 1) ? __builtin_amdgcn_perm(w1[e / 2], w0[e / 2], 0x07060302u)
                                           : __builtin_amdgcn_perm(w1[e / 2], w0[e / 2], 0x05040100u);
                *reinterpret_cast<uint32_t*>(vt + (8 * pc + e) * VP + 2 * j) = d;
            }
        }
        __syncthreads();
        {  // scores: wave w -> key tile w % KT, head-width part w / KT; lane: S[4 kq + i][16 kt + m]
            const uint32_t kt = wave % KT, dp = wave / KT;
            v4f sv = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int d = 0; d < DS; ++d) {
                const uint32_t k = 32 * (dp * DS + d) + 8 * kq;
                const v8h B = *reinterpret_cast<const v8h*>(ks + (16 * kt + m) * KP + k);
                sv = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(qh + m * KP + k), B, sv, 0, 0, 0);
                sv = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(ql + m * KP + k), B, sv, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[dp][4 * kq + i][16 * kt + m] = sv[i];
        }
        __syncthreads();
        // online softmax, wave w: queries 4 w .. 4 w + 3, lane = key
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = 4 * wave + i, key = k0 + lane;
            float s = -INFINITY;
            if (lane < (uint32_t)KC && tok[r] >= 0 && key < k_end && (int)key >= lo_q[r] && (int)key <= hi_q[r]) {
                float v = sc[0][r][lane];
#pragma unroll
                for (int dp = 1; dp < DH; ++dp) v += sc[dp][r][lane];
                s = v * qscale[r] * a.scale;
            }
            const float mo = mrun[r], mn = fmaxf(mo, wave_max(s));
            const float p = s == -INFINITY ? 0.0f : expf(s - mn);
            const float al = mn == -INFINITY ? 1.0f : expf(mo - mn);
            const float sum = wave_sum(p);
            if (lane < (uint32_t)KC) split_f16(p * 16384.0f, ph[r * VP + lane], pl[r * VP + lane]);
            if (lane == 0) {
                mrun[r] = mn;
                lrun[r] = fmaf(lrun[r], al, sum);
                alpha[r] = al;
            }
        }
        __syncthreads();
        {  // values: wave w -> channel tiles w NT + j; lane: O[4 kq + i][16 (w NT + j) + m]
            float al[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) al[i] = alpha[4 * kq + i];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[j][i] *= al[i];
                const uint32_t dim = 16 * (wave * NT + j) + m;
#pragma unroll
                for (int kk = 0; kk < KC / 32; ++kk) {
                    const uint32_t k = 32 * kk + 8 * kq;
                    const v8h B = *reinterpret_cast<const v8h*>(vt + dim * VP + k);
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(ph + m * VP + k), B, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(pl + m * VP + k), B, acc[j], 0, 0, 0);
                }
            }
        }
    }
    __syncthreads();
    if (a.nchunks == 1) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t r = 4 * kq + i, qi = 16 * qt + r;
                if (tok[r] < 0) continue;
                a.out[(size_t)tok[r] * a.out_stride + (size_t)(h * a.group + qi % a.group) * D + 16 * (wave * NT + j) + m] =
                    acc[j][i] * (1.0f / 16384.0f) / lrun[r];
            }
        return;
    }
    // chunk partials: sum p v (the probabilities' 2^14 removed), max, sum p
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t r = 4 * kq + i;
            if (tok[r] < 0) continue;
            const uint32_t qi = 16 * qt + r, row = (uint32_t)tok[r] * q_heads + h * a.group + qi % a.group;
            a.part[((size_t)row * a.nchunks + c) * (D + 2) + 16 * (wave * NT + j) + m] = acc[j][i] * (1.0f / 16384.0f);
        }
    if (tid < 16 && tok[tid] >= 0) {
        const uint32_t qi = 16 * qt + tid, row = (uint32_t)tok[tid] * q_heads + h * a.group + qi % a.group;
        float* pr = a.part + ((size_t)row * a.nchunks + c) * (D + 2);
        pr[D] = mrun[tid];
        pr[D + 1] = lrun[tid];
    }
}

// ---- attention of a wide pass ---------------------------------------------------------------------
//
// As batch_attention_kernel, for passes of more than kBatchMax tokens: grid (nchunks, kv_heads, query
// tiles of 64), a wave holding 16 queries from scores to output, so that the softmax needs no
// exchange between waves.  Products are taken transposed, S^T = K Q^T and O^T = V^T P^T: a lane then
// holds one query's column of both (query lane % 16), its maximum, sum and rescaling factor are its
// own (two lane swaps reduce over the four lanes of a query), and the probabilities are the second
// product's B operand as they stand: a lane's scores of two 16-key tiles are keys 4 q + e and 16 +
// 4 q + e (q = lane / 16), which only fixes the order of the keys in V^T (key j of 32 at 8 (j % 16 /
// 4) + 4 (j / 16) + j % 4).  K and V of the next sub-chunk are loaded into registers while this one's
// products run.
//
// The queries stay in registers (fp16 pairs, D / 4 VGPRs), so K is read from LDS once per wave and
// sub-chunk.  V^T rows have 36 dwords (KC 64) or 20, and a row's 16-byte pieces are XORed with its
// dimension / 16, so that neither the transposing stores (lane = 8 dimensions of a key pair) nor the operand
// reads (lane = dimension) hit a bank more than twice as often as they must.
template <int D, int KC>
__global__ __launch_bounds__(256, D == 256 ? 2 : 1) void wide_attention_kernel(BatchAttn a) {
    constexpr int KP = D + 8;           // K row stride (halves)
    constexpr int VS = KC / 2 + 4;      // V^T row stride (dwords)
    constexpr int KT = KC / 16, DT = D / 16, DS = D / 32;
    constexpr int NK = KC * D / 8 / 256, NV = NK / 2;  // 16-byte K pieces, V key-pair pieces per thread
    __shared__ __align__(16) _Float16 ks[KC * KP];
    __shared__ __align__(16) uint32_t vt[D * VS];

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = wave_id(), m = lane & 15, q = lane >> 4;
    const uint32_t c = blockIdx.x, h = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;
    const uint32_t q_heads = a.kv_heads * a.group, nq = a.T * a.group;
    // this lane's query (the last one again past the end; not stored)
    const uint32_t qi = 64 * qt + 16 * wave + m, qc = min(qi, nq - 1), t = qc / a.group;
    const uint32_t row = t * q_heads + h * a.group + qc % a.group;
    const int hi_q = (int)(a.pos0 + t), lo_q = a.window ? max(0, hi_q + 1 - (int)a.window) : 0;
    // the keys the tile's first token to its last sees, in whole sub-chunks per chunk (a chunk past the
    // end is empty: maximum -inf, sums 0)
    const uint32_t t_lo = 64 * qt / a.group, t_hi = min(a.T - 1, (64 * qt + 63) / a.group);
    const uint32_t klo = a.window ? (uint32_t)max(0, (int)(a.pos0 + t_lo + 1) - (int)a.window) : 0u;
    const uint32_t khi = a.pos0 + t_hi + 1;
    const uint32_t span = ((khi - klo + KC - 1) / KC + a.nchunks - 1) / a.nchunks * KC;
    const uint32_t k_begin = klo + c * span, k_end = min(k_begin + span, khi);

    const uint16_t* kh = a.kcache + (size_t)h * a.ring * D;
    const uint16_t* vh = a.vcache + (size_t)h * a.ring * D;
    v4u kr[NK], vr[2 * NV];
    // rows past the last key repeat it (their scores are masked; their values are cleared in store);
    // a sub-chunk's keys span less than one turn of the ring
    auto slot = [&](uint32_t k0, uint32_t r) {
        const uint32_t s = k0 % a.ring + min(r, min((uint32_t)KC, k_end - k0) - 1);
        return s >= a.ring ? s - a.ring : s;
    };
    auto load_k = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const uint32_t e = tid + 256 * i;
            kr[i] = *gp(reinterpret_cast<const v4u*>(kh + (size_t)slot(k0, e / (D / 8)) * D + 8 * (e % (D / 8))));
        }
    };
    auto load_v = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const uint32_t e = tid + 256 * i, j = 2 * (e / (D / 8)), pc = 8 * (e % (D / 8));
            vr[2 * i] = *gp(reinterpret_cast<const v4u*>(vh + (size_t)slot(k0, j) * D + pc));
            vr[2 * i + 1] = *gp(reinterpret_cast<const v4u*>(vh + (size_t)slot(k0, j + 1) * D + pc));
        }
    };
    auto store = [&](uint32_t k0) {
        const uint32_t kn = min((uint32_t)KC, k_end - k0);
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const uint32_t e = tid + 256 * i;
            *reinterpret_cast<v4u*>(ks + e / (D / 8) * KP + 8 * (e % (D / 8))) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const uint32_t e = tid + 256 * i, j = 2 * (e / (D / 8)), pc = e % (D / 8);
            v4u v0 = vr[2 * i], v1 = vr[2 * i + 1];
            if (j >= kn) v0 = v4u{0u, 0u, 0u, 0u};
            if (j + 1 >= kn) v1 = v4u{0u, 0u, 0u, 0u};
            // keys j, j + 1 at halves 8 (j % 16 / 4) + 4 (j % 32 / 16) + j % 4 of their 32 keys
            const uint32_t at = j / 32 * 16 + (j % 16 / 4) * 4 + j % 32 / 16 * 2 + j % 4 / 2;
            const uint32_t sw = ((at / 4) ^ (pc / 2 % (KC / 8))) * 4 + at % 4;
#pragma unroll
            for (int d = 0; d < 8; ++d)
                vt[(8 * pc + d) * VS + sw] = __builtin_amdgcn_perm(v1[d / 2], v0[d / 2], d & 1 ? 0x07060302u : 0x05040100u);
        }
    };
    if (k_begin < k_end) {
        load_k(k_begin);
        load_v(k_begin);
    }

    // the query as scaled fp16 pairs: lane (query m, q) holds channels 32 s + 8 q .. + 7 of step s
    v8h qh[DS], ql[DS];
    float qscale;
    {
        const float* src = a.q + (size_t)row * D + 8 * q;
        v4f v[DS][2];
        float mx = 0.0f;
#pragma unroll
        for (int s = 0; s < DS; ++s)
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                v[s][k] = *gp(reinterpret_cast<const v4f*>(src + 32 * s + 4 * k));
#pragma unroll
                for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(v[s][k][e]));
            }
        mx = lanes4_max(mx);
        const float s = mx > 0.0f ? ldexpf(1.0f, 4 - ilogbf(mx)) : 1.0f;  // |q s| < 32
#pragma unroll
        for (int i = 0; i < DS; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                _Float16 hi, lo;
                split_f16(v[i][e / 4][e % 4] * s, hi, lo);
                qh[i][e] = hi;
                ql[i][e] = lo;
            }
        qscale = a.scale / s;  // (s is a power of two)
    }
    v4f acc[DT];
#pragma unroll
    for (int j = 0; j < DT; ++j) acc[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    float mrun = -INFINITY, lrun = 0.0f;

    for (uint32_t k0 = k_begin; k0 < k_end; k0 += KC) {
        __syncthreads();  // the last sub-chunk's K and V^T are read
        store(k0);
        __syncthreads();
        if (k0 + KC < k_end) load_k(k0 + KC);
        __builtin_amdgcn_sched_barrier(0);
        // scores: S^T[16 kt + 4 q + e][m]
        v4f sv[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            v4f x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < DS; ++s) {
                const v8h A = *reinterpret_cast<const v8h*>(ks + (16 * kt + m) * KP + 32 * s + 8 * q);
                x = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, qh[s], x, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, ql[s], x, 0, 0, 0);
            }
            sv[kt] = x;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = (int)(k0 + 16 * kt + 4 * q + e);
                const float s = key >= lo_q && key <= hi_q ? sv[kt][e] * qscale : -INFINITY;
                sv[kt][e] = s;
                mx = fmaxf(mx, s);
            }
        const float mn = fmaxf(mrun, lanes4_max(mx));
        const float al = mn == -INFINITY ? 1.0f : expf(mrun - mn);
        float sum = 0.0f;
        v8h ph[KT / 2], pl[KT / 2];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float p = sv[kt][e] == -INFINITY ? 0.0f : expf(sv[kt][e] - mn);
                sum += p;
                _Float16 hi, lo;
                split_f16(p * 16384.0f, hi, lo);
                ph[kt / 2][kt % 2 * 4 + e] = hi;
                pl[kt / 2][kt % 2 * 4 + e] = lo;
            }
        mrun = mn;
        lrun = fmaf(lrun, al, row_total(sum));
        __builtin_amdgcn_sched_barrier(0);
        if (k0 + KC < k_end) load_v(k0 + KC);  // (here: with the scores' registers free)
        __builtin_amdgcn_sched_barrier(0);
        // values: O^T[16 j + 4 q + e][m]
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            v4f o = acc[j] * al;
#pragma unroll
            for (int kk = 0; kk < KT / 2; ++kk) {
                const uint32_t sw = ((4 * kk + q) ^ (j % (KC / 8))) * 4;
                const v8h A = *reinterpret_cast<const v8h*>(vt + (16 * j + m) * VS + sw);
                o = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, ph[kk], o, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, pl[kk], o, 0, 0, 0);
            }
            acc[j] = o;
        }
    }
    if (qi >= nq) return;
    if (a.nchunks == 1) {
        float* out = a.out + (size_t)t * a.out_stride + (size_t)(h * a.group + qc % a.group) * D + 4 * q;
        const float inv = 1.0f / 16384.0f;
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            v4f o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = acc[j][e] * inv / lrun;
            *reinterpret_cast<v4f*>(out + 16 * j) = o;
        }
        return;
    }
    // chunk partials: sum p v (the probabilities' 2^14 removed), max, sum p
    float* pr = a.part + ((size_t)row * a.nchunks + c) * (D + 2);
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; e += 2)
            *reinterpret_cast<float2*>(pr + 16 * j + 4 * q + e) =
                make_float2(acc[j][e] * (1.0f / 16384.0f), acc[j][e + 1] * (1.0f / 16384.0f));
    if (q == 0) *reinterpret_cast<float2*>(pr + D) = make_float2(mrun, lrun);
}

// out[t][qh] = sum_c w_c o_c / sum_c w_c l_c, w_c = exp(m_c - max_c m_c), chunks in order; one
// workgroup per (token, query head), one thread per channel.
template <int D>
__global__ __launch_bounds__(D) void batch_attention_merge_kernel(BatchAttn a) {
    const uint32_t row = blockIdx.x, q_heads = a.kv_heads * a.group, t = row / q_heads, qh = row % q_heads;
    const float* pr = a.part + (size_t)row * a.nchunks * (D + 2);
    float M = -INFINITY;
    for (uint32_t c = 0; c < a.nchunks; ++c) M = fmaxf(M, pr[c * (D + 2) + D]);
    float L = 0.0f, acc = 0.0f;
    for (uint32_t c = 0; c < a.nchunks; ++c) {
        const float mc = pr[c * (D + 2) + D];
        const float w = mc == -INFINITY ? 0.0f : expf(mc - M);
        L = fmaf(w, pr[c * (D + 2) + D + 1], L);
        acc = fmaf(w, pr[c * (D + 2) + threadIdx.x], acc);
    }
    a.out[(size_t)t * a.out_stride + (size_t)qh * D + threadIdx.x] = acc / L;
}

// ---- launchers ----------------------------------------------------------------------------------

// Chunks of a tile's keys: about one per sub-chunk (64 keys, 32 at width 512), at most
// kBatchAttnChunks, in a pass of at most kBatchMax tokens, where the tiles alone would leave most CUs
// idle; a wide pass has tiles enough for a few chunks each (about 512 workgroups, two per CU at width
// 256; its chunk partials fit the same scratch).
hipError_t launch_batch_attention(BatchAttn a, uint32_t head_width, hipStream_t s) {
    if (a.T == 0 || a.T > kPassMax || a.kv_heads == 0 || a.group == 0 || (head_width != 256 && head_width != 512))
        return hipErrorInvalidValue;
    const uint32_t KC = head_width == 256 ? 64 : 32, per = a.T > kBatchMax ? 64 : 16;
    const int64_t lo = a.window ? std::max<int64_t>(0, (int64_t)a.pos0 + 1 - a.window) : 0;
    const uint32_t keys = a.pos0 + a.T - (uint32_t)lo, sub = (keys + KC - 1) / KC;
    const uint32_t tiles = (a.T * a.group + per - 1) / per, base = tiles * a.kv_heads;
    a.nchunks = std::min(sub, kBatchAttnChunks);
    if (a.T > kBatchMax)
        a.nchunks = std::min({a.nchunks, ((head_width == 256 ? 512 : 256) + base - 1) / base, kBatchAttnChunks * kBatchMax / a.T});
    const dim3 grid(a.nchunks, a.kv_heads, tiles);
    if (head_width == 256) {
        if (a.T > kBatchMax) hipLaunchKernelGGL((wide_attention_kernel<256, 32>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((batch_attention_kernel<256, 64>), grid, dim3(256), 0, s, a);
    } else {
        if (a.T > kBatchMax) hipLaunchKernelGGL((wide_attention_kernel<512, 32>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((batch_attention_kernel<512, 32>), grid, dim3(256), 0, s, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.nchunks == 1) return e;
    const dim3 rows(a.T * a.kv_heads * a.group);
    if (head_width == 256) hipLaunchKernelGGL((batch_attention_merge_kernel<256>), rows, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((batch_attention_merge_kernel<512>), rows, dim3(512), 0, s, a);
    return hipGetLastError();
}

uint32_t batch_padded(uint32_t tokens) {
    return tokens > kBatchMax ? 16 * wide_groups(tokens) : padded_tokens(tokens);
}

// K splits of a wide GEMM: about 512 workgroups (two per CU), each with at least kWideChain blocks;
// a gate/up pair is not split (its epilogue needs whole sums; its grid is large anyway).
static uint32_t wide_splits(uint32_t rows, uint32_t blocks, uint32_t tokens, bool pair) {
    if (pair) return 1;
    const uint32_t m = wide_tokens(tokens), items = (rows + 16383 / m) / (16384 / m) * ((tokens + m - 1) / m);
    return std::max<uint32_t>(1, std::min({(512 + items / 2) / items, kDeferParts, blocks / kWideChain}));
}

size_t batch_image_bytes(uint32_t blocks, uint32_t tokens) {
    if (tokens > kBatchMax)  // (every narrower pass's image fits too)
        return std::max(batch_image_bytes(blocks, kBatchMax),
                        ((size_t)blocks * 2048 + 64) * ((tokens + 127) / 128 * 8));
    return (size_t)blocks * padded_tokens(tokens) * (128 + 4);
}

size_t batch_gemm_part_bytes(uint32_t rows, uint32_t blocks, uint32_t tokens, bool gelu_pair) {
    size_t wide = 0;  // the largest over the wide passes up to `tokens`
    for (uint32_t t = 64; t < tokens + 64; t += 64) {
        const uint32_t T = std::min(t, tokens), S = T > kBatchMax ? wide_splits(rows, blocks, T, gelu_pair) : 1;
        if (S > 1) wide = std::max(wide, (size_t)S * 16 * wide_groups(T) * ((rows + 15) / 16 * 16) * 4);
    }
    if (tokens > kBatchMax) return std::max(wide, batch_gemm_part_bytes(rows, blocks, kBatchMax, gelu_pair));
    const GemmPlan p = gemm_plan(rows, blocks, gelu_pair);
    if (p.S == 1) return 0;
    return (size_t)p.S * (gelu_pair ? 2 : 1) * padded_tokens(tokens) * ((rows + 15) / 16 * 16) * 4;
}

// The wide GEMM's input image: one workgroup per token, in every mode.
static hipError_t launch_wide_input(const BatchIn& in, hipStream_t s) {
    const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (in.stride % 4 || !a16(in.x) || !a16(in.res) || !a16(in.x_out) || !a16(in.w_a) || !a16(in.w_n))
        return hipErrorInvalidValue;
    const uint32_t octets = in.K / 8;
    const dim3 g((in.T + 7) / 8 * 8);
    const size_t lds = in.mode == BI_EMBED ? (size_t)in.K * 4 : 0;
    if (in.parts) {
        if (in.mode != BI_RESID || octets > 512 || in.parts > kDeferParts || !a16(in.part) || in.part_row % 4 ||
            in.part_row < in.K)
            return hipErrorInvalidValue;
        hipLaunchKernelGGL((batch_input_kernel<1, true, true>), g, dim3(512), 0, s, in);
    } else if (octets <= 512) {
        hipLaunchKernelGGL((batch_input_kernel<1, false, true>), g, dim3(512), lds, s, in);
    } else if (octets <= 1024) {
        hipLaunchKernelGGL((batch_input_kernel<2, false, true>), g, dim3(512), lds, s, in);
    } else {
        hipLaunchKernelGGL((batch_input_kernel<4, false, true>), g, dim3(512), lds, s, in);
    }
    return hipGetLastError();
}

hipError_t launch_batch_input(const BatchIn& in, hipStream_t s) {
    if (in.T == 0 || in.T > kPassMax || in.K == 0 || in.K > 16384 || in.K % 32) return hipErrorInvalidValue;
    if (in.T > kBatchMax) return launch_wide_input(in, s);
    if (in.mode == BI_PLAIN && !in.w_n) {
        if (in.stride % 4 || reinterpret_cast<uintptr_t>(in.x) % 16) return hipErrorInvalidValue;
        const uint32_t octets = in.K / 8;
        const dim3 g(padded_tokens(in.T), (octets + 255) / 256);
        if (in.parts) {
            if (in.parts > kDeferPairParts || reinterpret_cast<uintptr_t>(in.part) % 16 || in.part_row % 4 ||
                in.part_row < in.K)
                return hipErrorInvalidValue;
            hipLaunchKernelGGL(batch_plain_input_kernel<true>, g, dim3(256), 0, s, in);
        } else {
            hipLaunchKernelGGL(batch_plain_input_kernel<false>, g, dim3(256), 0, s, in);
        }
    } else {
        // float4 access to x, res, x_out and the norm weights
        const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
        if (in.stride % 4 || !a16(in.x) || !a16(in.res) || !a16(in.x_out) || !a16(in.w_a) || !a16(in.w_n))
            return hipErrorInvalidValue;
        const uint32_t octets = in.K / 8;
        const dim3 g(padded_tokens(in.T));
        const size_t lds = in.mode == BI_EMBED ? (size_t)in.K * 4 : 0;
        if (in.parts) {
            if (in.mode != BI_RESID || octets > 512 || in.parts > kDeferParts || !a16(in.part) || in.part_row % 4 ||
                in.part_row < in.K)
                return hipErrorInvalidValue;
            hipLaunchKernelGGL((batch_input_kernel<1, true, false>), g, dim3(512), 0, s, in);
        } else if (octets <= 512) {
            hipLaunchKernelGGL((batch_input_kernel<1, false, false>), g, dim3(512), lds, s, in);
        } else if (octets <= 1024) {
            hipLaunchKernelGGL((batch_input_kernel<2, false, false>), g, dim3(512), lds, s, in);
        } else {
            hipLaunchKernelGGL((batch_input_kernel<4, false, false>), g, dim3(512), lds, s, in);
        }
    }
    return hipGetLastError();
}

template <int P, int G>
static hipError_t gemm_launch(const BatchGemm& a, hipStream_t s, uint32_t* parts) {
    const GemmPlan p = gemm_plan(a.w.rows, a.w.blocks, P == 2);
    const uint32_t tiles = (a.w.rows + 15) / 16;
    const dim3 grid((tiles + p.R - 1) / p.R, p.S);
    if (p.S > 1 && !a.part) return hipErrorInvalidValue;
    switch (p.R) {
        case 1: hipLaunchKernelGGL((batch_gemm_kernel<P, G, 1>), grid, dim3(kGemmThreads), 0, s, a); break;
        case 2: hipLaunchKernelGGL((batch_gemm_kernel<P, G, 2>), grid, dim3(kGemmThreads), 0, s, a); break;
        case 4: hipLaunchKernelGGL((batch_gemm_kernel<P, G, 4>), grid, dim3(kGemmThreads), 0, s, a); break;
        default:
            if constexpr (P == 1) hipLaunchKernelGGL((batch_gemm_kernel<P, G, 8>), grid, dim3(kGemmThreads), 0, s, a);
            break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.S == 1) return e;
    if (a.defer && !a.add && p.S <= (P == 2 ? kDeferPairParts : kDeferParts)) {
        if (parts) *parts = p.S;
        return hipSuccess;
    }
    const uint32_t n = a.T * a.w.rows;
    hipLaunchKernelGGL((batch_reduce_kernel<P>), dim3((n + 255) / 256), dim3(256), 0, s, a, p.S, 16u * G);
    return hipGetLastError();
}

template <int P>
static hipError_t wide_launch(const BatchGemm& a, hipStream_t s, uint32_t* parts) {
    const uint32_t m = wide_tokens(a.T), rows_wg = 16384 / m / P;  // (rows of each matrix)
    const uint32_t mtiles = (a.T + m - 1) / m, ngroups = (a.w.rows + rows_wg - 1) / rows_wg;
    const uint32_t S = wide_splits(a.w.rows, a.w.blocks, a.T, P == 2);
    if (a.add || (S > 1 && !a.part)) return hipErrorInvalidValue;
    const dim3 grid((mtiles * ngroups * S + 7) / 8 * 8);
    if (m == 128) hipLaunchKernelGGL((wide_gemm_kernel<2, P>), grid, dim3(256), 0, s, a, S, mtiles, ngroups);
    else hipLaunchKernelGGL((wide_gemm_kernel<1, P>), grid, dim3(256), 0, s, a, S, mtiles, ngroups);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || S == 1) return e;
    if (a.defer) {
        if (parts) *parts = S;
        return hipSuccess;
    }
    const uint32_t n = a.T * a.w.rows;
    hipLaunchKernelGGL((batch_reduce_kernel<P>), dim3((n + 255) / 256), dim3(256), 0, s, a, S, 16 * wide_groups(a.T));
    return hipGetLastError();
}

hipError_t launch_batch_gemm(const BatchGemm& a, bool gelu_pair, hipStream_t s, uint32_t* parts) {
    if (parts) *parts = 0;
    if (a.T > kBatchMax && a.T <= kPassMax && a.w.rows && a.w.blocks &&
        !(gelu_pair && (a.w2.rows != a.w.rows || a.w2.blocks != a.w.blocks)))
        return gelu_pair ? wide_launch<2>(a, s, parts) : wide_launch<1>(a, s, parts);
    if (a.T == 0 || a.T > kBatchMax || a.w.rows == 0 || a.w.blocks == 0) return hipErrorInvalidValue;
    if (gelu_pair && (a.w2.rows != a.w.rows || a.w2.blocks != a.w.blocks)) return hipErrorInvalidValue;
    const bool two = a.T > 16;
    if (gelu_pair) return two ? gemm_launch<2, 2>(a, s, parts) : gemm_launch<2, 1>(a, s, parts);
    return two ? gemm_launch<1, 2>(a, s, parts) : gemm_launch<1, 1>(a, s, parts);
}

}  // namespace af
