// Batched prefill kernels for gfx950: up to kPassMax prompt tokens through a layer with every
// weight read once for the whole pass (crates/cuda-backend/src/batch.rs, kernels/ada/q4_batch.cu
// in the reference, 32 tokens there).  A layer's pass is a chain of launches: the input image of every
// token's GEMV input (batch_input_kernel, with the residual and RMSNorm prologues), the Q4_0 GEMM over
// all tokens (batch_gemm_kernel up to kBatchMax tokens, wide_gemm_kernel above; partial sums when the
// GEMM splits K across workgroups), and the attention of all tokens (batch_attention_kernel or
// wide_attention_kernel, after a pass that appends every token's K and V).  Above kBatchMax tokens a
// pass is bound by its products, which the wide kernels share out like any large matrix product; up to
// it by the weight stream.  512 tokens through six layers of the 12B shape: 14.3 ms in 16 passes of 32,
// 4.86 ms in one.
//
// The products run on the fp16 matrix cores (v_mfma_f32_16x16x32_f16) with the tokens in the M dimension: A =
// a token's inputs over one 32-weight block (k) as two fp16 halves, B = the block's weights n - 8 of 16 rows as
// fp16 (exact: each nibble placed in the mantissa of 1024 + n, then 1032 subtracted), so that D[t][r] =
// sum_j u_j(t) (n_rj - 8) with every product exact.  The halves are of u, the inputs scaled by 2^(14 - e), e the
// ilogb of the largest |x| of the token (a wide pass) or of the token's range of K (up to kBatchMax tokens):
// |u| < 2^15, hi = fp16(u) and lo = fp16(u - hi), both rounded to nearest even, hold u to 2^-23 of itself, or to
// 2^-25 where that is more; a block far below the largest has a scale of its own (block_spread).  Each lane adds d_r
// D[t][r] to its fp32 sum per block, and the sum is multiplied by 2^(e - 14) once at the end.
#include "device.h"

namespace af {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

namespace {

uint32_t padded_tokens(uint32_t T) { return T <= 8 ? 8 : (T + 15) / 16 * 16; }

}  // namespace

// ---- input images of a batch --------------------------------------------------------------------
//
// Elements are taken in octets: part p of a block is elements 4 p .. 4 p + 3 and 16 + 4 p .. + 3, the
// eight that one lane of an MFMA operand holds.

// x 2^sh as two fp16 halves: hi = f16(u), lo = f16(u - hi), packed in pairs (x0, x1).
__device__ __forceinline__ void split_pair(float x0, float x1, int sh, uint32_t& hi, uint32_t& lo) {
    const float u0 = ldexpf(x0, sh), u1 = ldexpf(x1, sh);
    const _Float16 h0 = (_Float16)u0, h1 = (_Float16)u1;
    const _Float16 l0 = (_Float16)(u0 - (float)h0), l1 = (_Float16)(u1 - (float)h1);
    hi = (uint32_t)__builtin_bit_cast(uint16_t, h0) | (uint32_t)__builtin_bit_cast(uint16_t, h1) << 16;
    lo = (uint32_t)__builtin_bit_cast(uint16_t, l0) | (uint32_t)__builtin_bit_cast(uint16_t, l1) << 16;
}

// The halves of an octet (elements 4 p .. + 3 and 16 + 4 p .. + 3 of a block) scaled by 2^sh: one
// operand lane, in the order in which a dword of code bytes unpacks (unpack_dword).
__device__ __forceinline__ void octet_halves(const float (&v)[8], int sh, v4u& hi, v4u& lo) {
    uint32_t h0, h1, h2, h3, l0, l1, l2, l3;
    split_pair(v[0], v[2], sh, h0, l0);
    split_pair(v[4], v[6], sh, h1, l1);
    split_pair(v[1], v[3], sh, h2, l2);
    split_pair(v[5], v[7], sh, h3, l3);
    hi = v4u{h0, h1, h2, h3};
    lo = v4u{l0, l1, l2, l3};
}

// Exponent e of a token's scale 2^(14 - e): ilogb of its largest |x| (128 for an infinity, whose products are
// not finite at any scale).
__device__ __forceinline__ int token_exponent(float m) { return m > 0.0f ? min(ilogbf(m), 128) : 0; }

// The halves hi + lo hold u to 2^-23 of itself, or to 2^-25.  So with one scale for a whole token (|u| < 2^15) a
// block is held to 2^-23 of its own largest element as long as that is 2^-16 of the token's or more.  A block
// below 2^-kBlockSpread (four bits earlier, for its smaller elements) has its own scale, e + spread instead
// of e, and its products are multiplied by 2^spread: an outlier channel costs no other block its bits.
// 512 positions through six layers of the 12B shape: 3.93 ms, 4.37 where every token has such blocks (3.92
// without the rule).  Returns spread, 0 for every other block; at least -100 (below that a block no longer counts in fp32 sums).
constexpr int kBlockSpread = 12;
__device__ __forceinline__ int block_spread(float m, int e) {
    const int d = m > 0.0f ? ilogbf(m) - e : 0;
    return d < -kBlockSpread ? max(d, -100) : 0;
}

// Largest |v| of a block, in each of its four lanes (parts 0-3).
__device__ __forceinline__ float block_max4(const float (&v)[8]) {
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = fmaxf(m, fabsf(v[k]));
    m = fmaxf(m, dpp<kDppXor1>(m));
    return fmaxf(m, dpp<kDppXor2>(m));
}
__device__ __forceinline__ float block_max4(const v4f (&v)[2]) {
    const float u[8] = {v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
    return block_max4(u);
}

// Part p of block b of token t into the wide GEMM's image of G 16-token groups.
__device__ __forceinline__ void wide_halves(const float (&v)[8], int sh, uint32_t b, uint32_t p, uint32_t t, uint32_t G,
                                            v4u* img) {
    v4u* at = img + ((size_t)b * G + t / 16) * 128 + 16 * p + t % 16;
    octet_halves(v, sh, at[0], at[64]);
}

// One workgroup per token.  The input vector of the GEMM that follows (as floats [T][K], or as the wide
// GEMM's image):
//   BI_PLAIN: x_t (f32(rms(x_t) w_n) with w_n);
//   BI_RESID: v_t = (f32(rms(x_t) w_a) + res_t) * scale (w_a null: (x_t + res_t) * scale), stored to
//             x_out_t (the residual stream), then f32(rms(v_t) w_n);
//   BI_EMBED: v_t = table row ids[pos0 + t] * emb_scale, stored to x_out_t, then f32(rms(v_t) w_n).
// RMSNorm sums of squares and products in double, f32 results (crates/domain/src/rms_norm.rs:24-41).
// Thread j holds octets j, j + 512, ... (NO of them) in registers (an octet: part p of a block, two
// float4), and every global load of the token (x, res and both norm weights) is issued before the
// first reduction, so the kernel waits for memory once.
// PS: x comes from in.parts split-K partial planes (NO == 1 only).
// WIDE: the wide GEMM's image, one scale per token but for small blocks (block_spread); no padding tokens are
// written (their rows of the product are never stored).  Workgroup b takes token (b % 8) ceil(T / 8) + b / 8, so that the 16
// tokens whose halves share a 256-byte run of the image are mostly written through one XCD's L2.
template <int NO, bool PS, bool WIDE>
__global__ __launch_bounds__(512) void batch_input_kernel(BatchIn in) {
    extern __shared__ __align__(16) float xs[];  // [K], BI_EMBED only
    __shared__ double red[8];
    __shared__ float redf[8], reds[8];
    const uint32_t tid = threadIdx.x, K = in.K, nb = K / 32, no = K / 8, WG = wide_groups(in.T);
    const uint32_t t = WIDE ? blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    if (t >= in.T) return;
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
    // the GEMM's input
    float v[NO][8];
#pragma unroll
    for (int j = 0; j < NO; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 u = in.w_n ? norm4(x[j][h], rn, wn[j][h]) : x[j][h];
            v[j][4 * h] = u.x;
            v[j][4 * h + 1] = u.y;
            v[j][4 * h + 2] = u.z;
            v[j][4 * h + 3] = u.w;
        }
    int e = 0;
    float bm[NO];  // the octets' blocks' largest elements
    float *inv = nullptr, *factor = nullptr;
    if constexpr (WIDE) {
        // the token's largest block and its smallest that is not zero, with the same barriers
        float m = 0.0f, least = INFINITY;
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            bm[j] = block_max4(v[j]);
            m = fmaxf(m, bm[j]);
            if (bm[j] > 0.0f) least = fminf(least, bm[j]);
        }
        m = wave_max(m);
        least = -wave_max(-least);
        if ((tid & 63) == 0) {
            redf[tid >> 6] = m;
            reds[tid >> 6] = least;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            m = fmaxf(m, redf[w]);
            least = fminf(least, reds[w]);
        }
        e = token_exponent(m);
        inv = reinterpret_cast<float*>(in.img + (size_t)nb * WG * 2048);
        const bool spread = m > 0.0f && block_spread(least, e) != 0;
        if (spread) factor = inv + 16 * WG + t;
        if (tid == 0) inv[t] = m > 0.0f ? ldexpf(spread ? -1.0f : 1.0f, e - 14) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const uint32_t o = tid + 512 * j;
        if (o >= no) continue;
        if constexpr (WIDE) {
            const int d = block_spread(bm[j], e);
            if (factor && (o & 3) == 0) factor[(size_t)(o >> 2) * 16 * WG] = ldexpf(1.0f, d);
            wide_halves(v[j], 14 - e - d, o >> 2, o & 3, t, WG, reinterpret_cast<v4u*>(in.img));
        } else {
            v4f* y = reinterpret_cast<v4f*>(reinterpret_cast<float*>(in.img) + (size_t)t * K) + 8 * (o >> 2) + (o & 3);
            y[0] = v4f{v[j][0], v[j][1], v[j][2], v[j][3]};
            y[4] = v4f{v[j][4], v[j][5], v[j][6], v[j][7]};
        }
    }
}

// ---- Q4_0 GEMM over a batch ---------------------------------------------------------------------
//
// Up to kBatchMax tokens: bound by the weight stream (66 MB of a gate/up pair in about 10 us), so that
// everything else has to stay out of its way.  A workgroup of 16 waves takes 64 RW rows (RW waves
// of four 16-row tiles) over one of S ranges of K, its KW = 16 / RW waves of the same rows dealing
// the range's 4-block super-tiles among them:
// - Each wave requests its first super-tiles' weights (one 16-byte load per lane and tile), then the
//   workgroup turns its range of the fp32 inputs into fp16 halves in LDS (one or two waves a token),
//   scaled by a power of two per token and range (a small block also by its own, block_spread): no image
//   is read or written in memory, and no launch makes one.
// - The dwords of a lane's 16 code bytes (block lane / 16, row lane % 16) are exchanged between the
//   four lanes of a row in registers (lane swaps), so that dword b holds the lane's k-slots of block
//   b; nine operations then unpack eight weights (unpack_dword), and each product is folded with one
//   FMA per token and row.
// - Up to 8 tokens (PACK) the hi and lo halves are rows 0-7 and 8-15 of one MFMA operand, otherwise of two.
// The waves' sums are added in LDS.  With S > 1 the ranges' sums go to planes in memory, and the last
// workgroup of a row group to finish adds them and writes y, unless the next kernel
// does (defer) or the planes are many (kFuseSplits: batch_reduce_kernel).
//
// Where a token has small blocks, a second form of the loop multiplies by their factors (3840 -> 15360, 32
// tokens: 22.7 us against 20.6; 15360 -> 3840, 5 tokens: 17.2 against 14.5).
//
// 3840 -> 15360, 32 tokens: 20.4 us against 34.3 us for the separate input-image, GEMM and reduce launches
// this replaced (16 operations per eight weights, a per-block input scale, operands from L2 one block
// ahead); 15360 -> 3840, 5 tokens: 14.5 against 26.2 us.

namespace {

constexpr int kThrough = 16;        // buffer access policy sc1: through to (or from) the memory side
constexpr int kWaitVm0 = 0x0F70;    // s_waitcnt vmcnt(0), expcnt and lgkmcnt unconstrained
constexpr uint32_t kGemmLds = 128 * 1024;   // the range's input halves at most
// Ranges whose sums the last workgroup of a row group adds itself: with 32 tokens its 256 rows' planes are
// 32 KB each, and one CU takes longer over more of them than another launch does.
constexpr uint32_t kFuseSplits = 4;

// Work split of a GEMM: workgroups of W waves take 64 RW rows (of both matrices together for a gate/up
// pair, groups of them in all) over one of S ranges of K, so that about one workgroup per CU shares
// the weight stream, a range's input halves fit LDS and each wave has a super-tile.
// - Up to 8 tokens W 8, RW 1: the halves are cheap to make (8 KB per 1,024 columns), so a workgroup per 64 rows
//   makes its own (16 waves, 15360 -> 3840, 5 tokens: 15.6 us against 14.9; 4096 -> 3840: 11.0 against 8.9).
// - Above, the same with 16 tokens per workgroup (two groups tg of them above 16 tokens, which read the weights twice
//   rather than share one workgroup: 1024 -> 1000, 30 tokens: 7.1 us against 9.3), where its workgroups fit the 256
//   CUs in one round; their halves leave no room for a second one on a CU, so past that the grid takes two rounds,
//   and W 16 and RW 2 or 4 (up to 16 tokens, or 32) share the halves among more rows instead.  Over 29 shapes of
//   1,024 to 65,536 rows and 256 to 16,384 columns by 9 to 32 tokens the line lies there: 256 workgroups (8192 rows,
//   3840 columns, 9 tokens) 11.2 us against 11.8 with W 16, 288 (6144, 3840) 16.4 against 11.5, 320 (5120, 4096, 24
//   tokens) 21.6 against 15.1.  The one shape better on the other side is 15360 -> 3840 by 9 to 16 tokens (480; 23.8
//   against 25.7).
struct GemmPlan {
    uint32_t rw, waves, tg, groups, S;
};
GemmPlan gemm_plan(uint32_t rows, uint32_t blocks, uint32_t T, bool pair) {
    const uint32_t tiles = (rows + 15) / 16 * (pair ? 2 : 1), nst = (blocks + 3) / 4;
    const auto form = [&](uint32_t rw, uint32_t waves, uint32_t tg) {
        const uint32_t groups = (tiles + 4 * rw - 1) / (4 * rw) * tg;
        const uint32_t most = kGemmLds / (4096u * (T <= 8 ? 1 : T <= 16 || tg == 2 ? 2 : 4));  // super-tiles of a range
        const uint32_t need = (nst + most - 1) / most, each = waves == 16 ? nst / (waves / rw) : (nst + 7) / 8;
        const uint32_t want = std::max(1u, std::min((256 + groups / 2) / groups, each));
        return GemmPlan{rw, waves, tg, groups, std::max(need, std::min(want, kDeferParts))};
    };
    const GemmPlan p = form(1, 8, T > 16 ? 2 : 1);
    return T <= 8 || p.groups * p.S <= 256 ? p : T <= 16 ? form(2, 16, 1) : form(4, 16, 1);
}

// Super-tiles [s0, s1) of range k of S.
__host__ __device__ inline uint32_t range_begin(uint32_t nst, uint32_t S, uint32_t k) { return (uint32_t)((uint64_t)nst * k / S); }

}  // namespace

// One lane's eight fp16 weights n - 8 of a block from the dword of its code bytes 4 q .. 4 q + 3: the
// nibbles' bits in the mantissa of 1024 + n (or 1024 + 16 n), then 1032 subtracted (or scaled by 1/16
// and 72 subtracted), exactly.  Weights 4 q + {0, 2}, 16 + 4 q + {0, 2}, 4 q + {1, 3}, 16 + 4 q + {1, 3}.
__device__ __forceinline__ v4u unpack_dword(uint32_t c) {
    const v2h bias = {(_Float16)1032.0f, (_Float16)1032.0f}, hb = {(_Float16)-72.0f, (_Float16)-72.0f},
              sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    // (the constants in registers, the mask's scalar: v_and_or_b32 takes no literals)
    uint32_t low = 0x000F000Fu, high = 0x00F000F0u, magic = 0x64006400u;
    asm("" : "+s"(low), "+s"(high), "+v"(magic));
    const uint32_t c8 = c >> 8;
    const v2h a = __builtin_bit_cast(v2h, (c & low) | magic) - bias;
    const v2h b = __builtin_elementwise_fma(__builtin_bit_cast(v2h, (c & high) | magic), sixteenth, hb);
    const v2h e = __builtin_bit_cast(v2h, (c8 & low) | magic) - bias;
    const v2h f = __builtin_elementwise_fma(__builtin_bit_cast(v2h, (c8 & high) | magic), sixteenth, hb);
    return v4u{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, e),
               __builtin_bit_cast(uint32_t, f)};
}

// Lane group g (lanes 16 g .. + 15) holding dwords v[0..3] of its column: afterwards dword b of lane
// group g is dword g of lane group b (the four lanes of a row transpose their 4 x 4 dwords).
__device__ __forceinline__ v4u transpose_lanes(v4u v) {
    const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);  // groups 2, 3 of x with 0, 1 of z
    const auto b = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);  // groups 1, 3 of one with 0, 2 of the other
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return v4u{c[0], c[1], d[0], d[1]};
}
// Lane group g's value g of its column, in every lane: o[b] is lane group b's v.
__device__ __forceinline__ void spread_lanes(uint32_t v, uint32_t (&o)[4]) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
    o[0] = a[0];
    o[1] = a[1];
    o[2] = b[0];
    o[3] = b[1];
}

// u[0] + ... + u[N - 1] (N a power of two), halves first: the rounding errors of log2 N additions in a row, not N - 1.
template <int N>
__device__ __forceinline__ float tree_sum(const float (&u)[N]) {
    if constexpr (N == 1) {
        return u[0];
    } else {
        float h[N / 2];
#pragma unroll
        for (int k = 0; k < N / 2; ++k) h[k] = u[2 * k] + u[2 * k + 1];
        return tree_sum(h);
    }
}

template <int G, bool PACK, int P, int RW, int W>
__global__ __launch_bounds__(64 * W) void batch_gemm_kernel(BatchGemm a, uint32_t S, uint32_t groups, uint32_t tgroups,
                                                            uint32_t fuse) {
    constexpr int KW = W / RW, kTokens = PACK ? 8 : 16 * G;
    constexpr int NF = PACK ? 1 : 2 * G;        // 1 KB operands per block: [token group][hi, lo], or one packed
    constexpr uint32_t TR = 16 * G;             // operand rows (tokens; PACK: hi, then lo of eight tokens)
    constexpr uint32_t NR = 64 * RW;            // rows of the workgroup
    static_assert(W <= kTokens, "a wave per token in the input stage, or several tokens");
    constexpr int TW = kTokens / W;             // tokens per wave there
    constexpr int NO = kGemmLds / (4096 * NF) / 4;  // octet rounds of 64 lanes per token
    // super-tiles requested ahead of the one being multiplied (16 waves have 128 registers each)
    constexpr int kAhead = W == 16 ? 1 : 2;
    extern __shared__ __align__(16) v4u smem[]; // input halves [block][NF][64 lanes], later sums [KW][TR][NR] f32
    __shared__ float inv[32];                   // the tokens' scales 2^(e - 14), negative with small blocks
    __shared__ __align__(16) float factor[1024];  // of those tokens' blocks (block_spread) [block][kTokens]
    static_assert(kGemmLds / (1024 * NF) * kTokens == 1024, "a factor per block of the range and token");
    __shared__ bool last;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = wave_id(), r = lane & 15, q = lane >> 4;
    const uint32_t rw = wave % RW, kw = wave / RW;
    // item (row group, split), split fastest, in contiguous shares per XCD (workgroup b runs on XCD
    // b % 8): the splits of a row group mostly share an XCD
    const uint32_t item = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;
    if (item >= groups * S) return;
    // (row group, token group): with two of the latter, tokens 16 tg .. + 15 are this workgroup's
    const uint32_t gi = item / S, split = item % S, rg = gi / tgroups, tg = gi % tgroups;
    const uint32_t Tp = (PACK ? 8 : TR) * tgroups;  // tokens per plane
    if (tgroups > 1) {
        a.x += (size_t)tg * TR * a.x_stride;
        a.y += (size_t)tg * TR * a.y_stride;
        a.T = min(a.T - tg * TR, TR);
    }
    const uint32_t nst = a.w.nst, nb = a.w.blocks, tiles = (a.w.rows + 15) / 16;
    const uint32_t s0 = range_begin(nst, S, split), s1 = range_begin(nst, S, split + 1);

    // ---- weights: the wave's row tiles 4 rw .. + 3 of the workgroup (a gate/up pair alternates the
    // matrices), super-tiles s0 + kw, + KW, ...
    // (through a buffer of no bytes past the range: the same two loads, without a memory access, so that
    // every wait is an exact count)
    const uint8_t* cp[4];
    const uint16_t* dp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = 4 * (rg * RW + rw) + i, tile = min(P == 2 ? v / 2 : v, tiles - 1);
        const Q4View& w = P == 2 && (i & 1) ? a.w2 : a.w;
        cp[i] = w.codes + (size_t)tile * nst * 1024;
        dp[i] = w.scales + (size_t)tile * nst * 64;
    }
    v4u wc[kAhead][4];
    uint32_t wd[kAhead][4];
    auto request = [&](int u, uint32_t st) {
        const bool in = st < s1;
        const size_t at = in ? st : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(cp[i]) + at * 1024, 0,
                                                                                 in ? 1024 : 0, 0x00020000);
            const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(dp[i]) + at * 64, 0,
                                                                                 in ? 128 : 0, 0x00020000);
            wc[u][i] = __builtin_amdgcn_raw_buffer_load_b128(rc, lane * 16, 0, 2);
            wd[u][i] = __builtin_amdgcn_raw_buffer_load_b16(rd, lane * 2, 0, 2);
        }
    };

    // ---- inputs: token t = wave + W k, octet o = (block o / 4, part o % 4) of the range
    const uint32_t no = (s1 - s0) * 16;  // octets of the range, those past the last block zero
    v4f x[TW][NO][2];
#pragma unroll
    for (int k = 0; k < TW; ++k) {
        const uint32_t t = wave + W * k;
        const float4* xp = reinterpret_cast<const float4*>(a.x + (size_t)min(t, a.T - 1) * a.x_stride);
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            // (past the range too: a load under a branch would be waited for at the branch's end)
            const uint32_t o = 64 * j + lane, b = min(s0 * 4 + (o >> 2), nb - 1), i0 = 8 * b + (o & 3);
            x[k][j][0] = *gp(reinterpret_cast<const v4f*>(xp + i0));
            x[k][j][1] = *gp(reinterpret_cast<const v4f*>(xp + i0 + 4));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) request(u, s0 + kw + KW * u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < TW; ++k) {
        const uint32_t t = wave + W * k;
        if (t >= a.T) continue;  // (its operand rows are not stored)
        float m = 0.0f, least = INFINITY;  // largest element; smallest octet's, of those not zero
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            if ((uint32_t)(64 * j) >= no) break;
            float om = 0.0f;
            const uint32_t o = 64 * j + lane;
            const bool in = o < no && s0 * 4 + (o >> 2) < nb;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[k][j][h][e] = in ? x[k][j][h][e] : 0.0f;
                    om = fmaxf(om, fabsf(x[k][j][h][e]));
                }
            m = fmaxf(m, om);
            least = fminf(least, om > 0.0f ? om : INFINITY);
        }
        m = wave_max(m);
        const int e = token_exponent(m);
        // small blocks: scaled to the token's exponent here, which is exact, and by their factors in the products
        // (looked for where an octet is small, which a block of other elements may hold too)
        bool small = false;
        if (__builtin_expect(__any(m > 0.0f && least < ldexpf(1.0f, e - kBlockSpread)), 0)) {
#pragma unroll
            for (int j = 0; j < NO; ++j) {
                if ((uint32_t)(64 * j) >= no) break;
                const uint32_t o = 64 * j + lane;
                const int d = block_spread(block_max4(x[k][j]), e);  // (a range is whole blocks)
                small |= d != 0;
#pragma unroll
                for (int h = 0; h < 8; ++h) x[k][j][h / 4][h % 4] = ldexpf(x[k][j][h / 4][h % 4], -d);
                if (o < no && o % 4 == 0) factor[o / 4 * kTokens + t] = ldexpf(1.0f, d);
            }
            small = __any(small);
        }
        if (lane == 0) inv[t] = m > 0.0f ? ldexpf(small ? -1.0f : 1.0f, e - 14) : 0.0f;
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const uint32_t o = 64 * j + lane;
            if (o < no) {
                // lane 16 p + row of the operand, its rows permuted by the block and part so that the
                // stores of a token's octets spread over the banks
                const uint32_t b = o >> 2, p = o & 3, s = (b & 3) * 4 + p;
                float v[8];
#pragma unroll
                for (int h = 0; h < 8; ++h) v[h] = x[k][j][h / 4][h % 4];
                v4u hi, lo;
                octet_halves(v, 14 - e, hi, lo);
                v4u* at = smem + (size_t)b * NF * 64 + 16 * p;
                if constexpr (PACK) {
                    at[t ^ s] = hi;
                    at[(t + 8) ^ s] = lo;
                } else {
                    at[(t / 16) * 128 + (t % 16 ^ s)] = hi;
                    at[(t / 16) * 128 + 64 + (t % 16 ^ s)] = lo;
                }
            }
        }
    }
    // the ticket raised to the launch's epoch (below), here, where nothing waits for it: just before its draw
    // 15360 -> 3840, 16 tokens, took 25.7 us instead of 25.1
    if (fuse && tid == 0) __hip_atomic_fetch_max(a.counters + gi, a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();

    // ---- products
    float acc[4][G][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][g][e] = 0.0f;
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    // tokens with block factors (the same in every wave)
    const float scale = lane < (uint32_t)kTokens ? inv[lane] : 0.0f;
    const uint32_t spread = (uint32_t)__ballot(scale < 0.0f && lane < a.T);
    auto multiply = [&](auto with_factors) {
        constexpr bool SPREAD = decltype(with_factors)::value;
        constexpr int A = SPREAD ? 1 : kAhead;  // (with factors one super-tile ahead, for its registers)
        for (uint32_t st0 = s0 + kw; st0 < s1; st0 += KW * A) {
#pragma unroll
            for (int u = 0; u < A; ++u) {
                const uint32_t st = st0 + KW * u;
                if (st >= s1) break;
                v4u c[4];
                uint32_t d[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    c[i] = transpose_lanes(wc[u][i]);
                    spread_lanes(wd[u][i], d[i]);
                }
                request(u, st + KW * A);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const v4u* at = smem + (size_t)((st - s0) * 4 + b) * NF * 64 + 16 * q + (r ^ (b * 4 + q));
                    v8h x16[NF];
#pragma unroll
                    for (int f = 0; f < NF; ++f) x16[f] = __builtin_bit_cast(v8h, at[64 * f]);
                    v4f fs[G];
                    if constexpr (SPREAD) {
#pragma unroll
                        for (int g = 0; g < G; ++g) {
                            const uint32_t t4 = PACK ? 4 * (q & 1) : 16 * g + 4 * q;
                            fs[g] = *reinterpret_cast<const v4f*>(factor + ((st - s0) * 4 + b) * kTokens + t4);
#pragma unroll
                            for (int e = 0; e < 4; ++e) fs[g][e] = spread >> (t4 + e) & 1 ? fs[g][e] : 1.0f;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const v8h w = __builtin_bit_cast(v8h, unpack_dword(c[i][b]));
                        const float ds = h2f((uint16_t)d[i][b]);
#pragma unroll
                        for (int g = 0; g < G; ++g) {
                            v4f D = __builtin_amdgcn_mfma_f32_16x16x32_f16(x16[PACK ? 0 : 2 * g], w, zero, 0, 0, 0);
                            if constexpr (!PACK) D = __builtin_amdgcn_mfma_f32_16x16x32_f16(x16[2 * g + 1], w, D, 0, 0, 0);
                            if constexpr (SPREAD) D *= fs[g];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][g][e] = fmaf(ds, D[e], acc[i][g][e]);
                        }
                    }
                }
            }
        }
    };
    if (__builtin_expect(spread != 0, 0)) multiply(std::true_type{});
    else multiply(std::false_type{});
    __syncthreads();  // every wave has read its operands

    // ---- the waves' sums: [kw][operand row][row]
    float* red = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                red[(kw * TR + 16 * g + 4 * q + e) * NR + 64 * rw + 16 * i + r] = acc[i][g][e];
    __syncthreads();
    // thread: row n of the workgroup (P == 2: the gate's row, tiles 2 j and 2 j + 1 paired), tokens t0, + TS, ...
    constexpr uint32_t NY = NR / P, TS = 64 * W / NY, NT = kTokens / TS > 0 ? kTokens / TS : 1;
    const uint32_t n = tid % NY, t0 = tid / NY;
    const uint32_t row = rg * NY + n, prow = tiles * 16;
    const uint32_t col = P == 2 ? n / 16 * 32 + n % 16 : n;
    float v[NT][P];
#pragma unroll
    for (uint32_t j = 0; j < NT; ++j) {
        const uint32_t t = t0 + TS * j;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            float s = 0.0f;
            if (t < a.T) {
                float u[KW];
#pragma unroll
                for (int k = 0; k < KW; ++k) {
                    const float* at = red + (size_t)k * TR * NR + t * NR + col + 16 * p;
                    u[k] = PACK ? at[0] + at[8 * NR] : at[0];
                }
                s = tree_sum(u) * fabsf(inv[t]);
            }
            v[j][p] = s;
        }
    }
    auto put = [&](uint32_t t, const float (&s)[P]) {
        float* y = a.y + (size_t)t * a.y_stride + row;
        if constexpr (P == 2) *y = gelu_mul(s[0], s[1]);
        else *y = s[0];
    };
    if (S == 1) {
#pragma unroll
        for (uint32_t j = 0; j < NT; ++j)
            if (t0 + TS * j < a.T && row < a.w.rows) put(t0 + TS * j, v[j]);
        return;
    }
    // planes [split][P][Tp][prow]
    auto plane = [&](uint32_t k, int p, uint32_t t) { return ((size_t)(k * P + p) * Tp + tg * TR + t) * prow + row; };
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(a.part, 0, 0x7FFFFFFF, 0x00020000);
#pragma unroll
    for (uint32_t j = 0; j < NT; ++j) {
        const uint32_t t = t0 + TS * j;
        if (t < a.T && row < prow)
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (fuse) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[j][p]), prs, (uint32_t)plane(split, p, t) * 4, 0, kThrough);
                else a.part[plane(split, p, t)] = v[j][p];
            }
    }
    if (!fuse) return;
    // the last workgroup of the row group adds the planes: stored through to the memory side and
    // waited for before the ticket, read from there (the XCDs' L2s are not coherent with each other).
    // Tickets count from the launch's epoch: two launches that overlap on the same counters (which
    // callers are told not to make) spoil each other's sums and may leave a count behind, but a
    // later launch's epoch is above it.
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    if (tid == 0) {
        const uint64_t ticket = __hip_atomic_fetch_add(a.counters + gi, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = ticket == a.epoch + S - 1;
        if (last) __hip_atomic_store(a.counters + gi, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
    // every load of a few tokens at once, unconditional (past the planes or rows: out of the buffer, zeros)
    constexpr uint32_t FS = G == 2 ? kFuseSplits : kDeferParts, JB = NT < 4 ? NT : 4;
#pragma unroll
    for (uint32_t j0 = 0; j0 < NT; j0 += JB) {
        float u[JB][P][FS];
#pragma unroll
        for (uint32_t j = 0; j < JB; ++j)
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (uint32_t k = 0; k < FS; ++k) {
                    const uint32_t t = t0 + TS * (j0 + j);
                    const uint32_t off = k < S && t < a.T && row < prow ? (uint32_t)plane(k, p, t) * 4 : 0x80000000u;
                    u[j][p][k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(prs, off, 0, kThrough));
                }
#pragma unroll
        for (uint32_t j = 0; j < JB; ++j) {
            const uint32_t t = t0 + TS * (j0 + j);
            float s[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                s[p] = tree_sum(u[j][p]);
            }
            if (t < a.T && row < a.w.rows) put(t, s);
        }
    }
}

// y from S split-K partial planes; one thread per (t, row).
template <int P>
__global__ __launch_bounds__(256) void batch_reduce_kernel(BatchGemm a, uint32_t S, uint32_t Tp) {
    const uint32_t rows = a.w.rows, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.T * rows) return;
    const uint32_t t = i / rows, row = i % rows;
    const size_t prow = (size_t)(rows + 15) / 16 * 16;
    float v[P];
#pragma unroll
    for (int q = 0; q < P; ++q) {
        float s = 0.0f;  // four planes at a time
        for (uint32_t k = 0; k < S; k += 4) {
            float u[4];
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) u[i] = k + i < S ? a.part[((size_t)((k + i) * P + q) * Tp + t) * prow + row] : 0.0f;
            s += tree_sum(u);
        }
        v[q] = s;
    }
    float* y = a.y + (size_t)t * a.y_stride + row;
    if constexpr (P == 2) *y = gelu_mul(v[0], v[1]);
    else *y = v[0];
}

// ---- Q4_0 GEMM over a wide pass -------------------------------------------------------------------
//
// y[t][r] = sum_b d_rb sum_j (n_rbj - 8) x_tbj for more than kBatchMax tokens.  A workgroup takes M = 64 WM
// tokens x 64 WN rows over K range `split`, WM x WN waves of 64 x 64 (4 x 4 MFMA tiles) for each of WK
// 32-weight blocks (one MFMA depth) per step: the tokens' halves are copied from the image, which
// is laid out as the MFMAs read it, by LDS DMA two steps ahead (one where WK is 4), and the weights unpacked once per
// workgroup into LDS while the step before is multiplied.  The WK waves of a tile add their sums in LDS at the
// end.  The block's d_rb differs from the next one's, so each block's 16 x 16 products are folded into fp32 sums on
// their own (one FMA per product and lane: half as many VALU cycles as the two MFMAs take; the token's scale waits
// for the epilogue, so that the fold has no other factor, unless a token of the tile has small blocks with scales
// of their own: then a second form of the loop multiplies by the blocks' factors).  Sums run over kWideChain blocks,
// then join a total, so that no chain of fp32 additions is longer than K / 32 / kWideChain + kWideChain.
//
// Work items (split, row group, token tile), token tile fastest, go to the XCDs in contiguous
// shares (workgroup b runs on XCD b % 8), so that the workgroups that unpack the same weights share
// an L2.
constexpr uint32_t kWideChain = 8;
typedef __attribute__((address_space(3))) void* lds_ptr;

template <int WM, int WN, int WK, int P>
__global__ __launch_bounds__(64 * WM * WN * WK, 2 / WK ? 2 / WK : 1) void wide_gemm_kernel(BatchGemm a, uint32_t S,
                                                                                             uint32_t mtiles,
                                                                                             uint32_t ngroups) {
    constexpr int MG = 4 * WM, NT = 4 * WN;       // 16-token groups and 16-row tiles of the workgroup
    constexpr int W = WM * WN * WK, TH = 64 * W;  // waves, threads
    constexpr int SA = 8 / WN, SB = 4 / WM;       // 16-byte pieces of the image and code dwords per thread and step
    constexpr int kA = MG * 128 * WK, kB = NT * 64 * WK;  // v4u per stage
    constexpr int NA = WK == 4 ? 2 : 3;           // image stages (three of the 64-token form would fill the LDS)
    constexpr int kAll = NA * kA + 2 * kB;
    static_assert(WK == 1 || W * 1024 <= kAll, "the waves' sums fit the stages");
    // NA image stages [block of the step][token group][hi, lo][64 lanes], two weight stages [block][row
    // tile][64 lanes]
    __shared__ v4u smem[kAll];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = wave_id(), r = lane & 15, q = lane >> 4;
    const uint32_t wk = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    const uint32_t total = mtiles * ngroups * S, per = gridDim.x / 8;
    const uint32_t item = blockIdx.x % 8 * per + blockIdx.x / 8;
    if (item >= total) return;
    const uint32_t mt0 = item % mtiles, ng = item / mtiles % ngroups, split = item / mtiles / ngroups;
    const uint32_t nb = a.w.blocks, G = mtiles * MG, tiles = (a.w.rows + 15) / 16;
    const uint32_t b0 = nb * split / S, b1 = nb * (split + 1) / S, last = b1 - 1;
    // row tile i of the workgroup (of wave i / 4): a gate/up pair's waves hold two tiles of each matrix,
    // alternating, so that a lane holds both products of a row
    auto tile_of = [&](uint32_t i) { return P == 2 ? ng * (NT / 2) + i / 4 * 2 + (i % 4) / 2 : ng * NT + i; };
    auto mat_of = [&](uint32_t i) -> const Q4View& { return P == 2 && (i & 1) ? a.w2 : a.w; };

    // this thread's share of a step: image pieces tid + TH i of its WK blocks (kA / WK per block), and the code
    // dwords of row tiles wave SB + i (of block (wave SB + i) / NT)
    uint32_t sc[SB];
    uint16_t dn[4];  // the next step's scales of the lane's rows
    // (every request is a buffer's base, the thread's constant offset and the block's scalar one: 64-bit
    // addresses per request took a third of the loop's VALU cycles)
    __amdgpu_buffer_rsrc_t rc[SB], rd[4];
#pragma unroll
    for (int i = 0; i < SB; ++i) {
        const uint32_t k = (wave * SB + i) % NT;
        const uint8_t* p = mat_of(k).codes + (size_t)min(tile_of(k), tiles - 1) * a.w.nst * 1024;
        rc[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, a.w.nst * 1024, 0x00020000);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t k = wn * 4 + i;
        const uint16_t* p = mat_of(k).scales + (size_t)min(tile_of(k), tiles - 1) * a.w.nst * 64;
        rd[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, a.w.nst * 128, 0x00020000);
    }
    const __amdgpu_buffer_rsrc_t ri =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(reinterpret_cast<const int8_t*>(a.img)), 0, nb * G * 2048, 0x00020000);
    // (blocks past the range repeat its last one; their scales are zeroed)
    auto copy = [&](uint32_t b, int st) {  // the image's pieces straight into stage st
#pragma unroll
        for (int i = 0; i < SA; ++i) {
            // (piece tid + TH i lies in block TH i / (MG 128) for every thread)
            static_assert((MG * 128) % TH == 0, "a block is whole rounds of the threads");
            const uint32_t blk = min(b + TH * i / (MG * 128), last);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ri, (lds_ptr)(smem + st * kA + wave * 64 + TH * i), 16, tid * 16,
                                                     (blk * G + mt0 * MG) * 2048 + TH * i % (MG * 128) * 16, 0, 0);
        }
    };
    auto load = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < SB; ++i)
            sc[i] = __builtin_amdgcn_raw_buffer_load_b32(rc[i], r * 16 + q * 4, min(b + (wave * SB + i) / NT, last) * 256, 0);
    };
    auto load_d = [&](uint32_t b) {
#pragma unroll
        for (int i = 0; i < 4; ++i) dn[i] = __builtin_amdgcn_raw_buffer_load_b16(rd[i], r * 2, min(b + wk, last) * 32, 0);
    };
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_ptr)smem;
    auto unpack = [&](int st) {  // (a store that the compiler sees would also wait for every copy in flight)
        const uint32_t at = lds + 16 * (NA * kA + st * kB + wave * SB * 64 + lane);
#pragma unroll
        for (int i = 0; i < SB; ++i) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(at), "v"(unpack_dword(sc[i])), "n"(1024 * i) : "memory");
    };
    v4f acc[4][4], tot[4][4];
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = tot[m][n] = zero;

    const float* inv = reinterpret_cast<const float*>(a.img + (size_t)nb * G * 2048);
    float scales[MG / 4];  // of the tile's tokens, 64 at a time
#pragma unroll
    for (int i = 0; i < MG / 4; ++i) scales[i] = gp(inv)[mt0 * MG * 16 + 64 * i + lane];
    load(b0);
    load_d(b0);
    unpack(0);
    load(b0 + WK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < NA - 1; ++st) copy(b0 + st * WK, st);
    __builtin_amdgcn_sched_barrier(0);
    bool small = false;
#pragma unroll
    for (int i = 0; i < MG / 4; ++i) small |= scales[i] < 0.0f && mt0 * MG * 16 + 64 * i + lane < a.T;
    auto multiply = [&](auto spread) {
        constexpr bool SPREAD = decltype(spread)::value;
        // SPREAD: this lane's tokens with factors, bit 4 m + e
        uint32_t own = 0;
        const float* factor = inv + 16 * G + (mt0 * MG + wm * 4) * 16 + 4 * q;
        if constexpr (SPREAD) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const v4f s = *gp(reinterpret_cast<const v4f*>(inv + (mt0 * MG + wm * 4 + m) * 16 + 4 * q));
#pragma unroll
                for (int e = 0; e < 4; ++e) own |= s[e] < 0.0f ? 1u << (4 * m + e) : 0u;
            }
        }
        uint32_t step = 0, sa = 0;  // step % NA
        for (uint32_t b = b0; b < b1; b += WK, ++step) {
            // This step's copies are in (with three stages, all but the SA newest requests: the copies for the
            // next step are the last ones of an iteration) and its weights written, in every wave; every wave
            // has read the stages that are written below.
            if constexpr (NA == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(SA) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            // The operands are read and waited for in one block: the compiler would wait for every copy in
            // flight before an LDS read that it sees.
            v4u ahu[4], alu[4], bwu[4];
            const uint32_t pa = lds + 16 * (sa * kA + wk * MG * 128 + wm * 512 + lane),
                           pb = lds + 16 * (NA * kA + (step & 1) * kB + wk * NT * 64 + wn * 256 + lane);
            asm volatile(
                "ds_read_b128 %8, %13\n\t"
                "ds_read_b128 %0, %12\n\t"
                "ds_read_b128 %1, %12 offset:2048\n\t"
                "ds_read_b128 %2, %12 offset:4096\n\t"
                "ds_read_b128 %3, %12 offset:6144\n\t"
                "ds_read_b128 %4, %12 offset:1024\n\t"
                "ds_read_b128 %5, %12 offset:3072\n\t"
                "ds_read_b128 %6, %12 offset:5120\n\t"
                "ds_read_b128 %7, %12 offset:7168\n\t"
                "ds_read_b128 %9, %13 offset:1024\n\t"
                "ds_read_b128 %10, %13 offset:2048\n\t"
                "ds_read_b128 %11, %13 offset:3072\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(ahu[0]), "=&v"(ahu[1]), "=&v"(ahu[2]), "=&v"(ahu[3]), "=&v"(alu[0]), "=&v"(alu[1]), "=&v"(alu[2]),
                  "=&v"(alu[3]), "=&v"(bwu[0]), "=&v"(bwu[1]), "=&v"(bwu[2]), "=&v"(bwu[3])
                : "v"(pa), "v"(pb)
                : "memory");
            v8h ah[4], al[4], bw[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                ah[m] = __builtin_bit_cast(v8h, ahu[m]);
                al[m] = __builtin_bit_cast(v8h, alu[m]);
                bw[m] = __builtin_bit_cast(v8h, bwu[m]);
            }
            float d[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                d[n] = WK == 1 || b + wk < b1 ? h2f(dn[n]) : 0.0f;
                asm("" : "+v"(d[n]));  // (converted once: as a mixed-precision operand of 64 FMAs it takes 1.5 % longer)
            }
            v4f f[4];
            if constexpr (SPREAD) {
#pragma unroll
                for (int m = 0; m < 4; ++m) f[m] = *gp(reinterpret_cast<const v4f*>(factor + (size_t)min(b + wk, last) * 16 * G + 16 * m));
            }
            unpack((step & 1) ^ 1);
            load(b + 2 * WK);
            load_d(b + WK);
            __builtin_amdgcn_sched_barrier(0);
            copy(b + (NA - 1) * WK, sa ? sa - 1 : NA - 1);
            __builtin_amdgcn_sched_barrier(0);
            sa = sa == NA - 1 ? 0 : sa + 1;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                v4f D[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) D[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[m], bw[n], zero, 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 4; ++m) D[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[m], bw[n], D[m], 0, 0, 0);
                if constexpr (SPREAD) {
#pragma unroll
                    for (int m = 0; m < 4; ++m)
#pragma unroll
                        for (int e = 0; e < 4; ++e) D[m][e] *= own >> (4 * m + e) & 1 ? f[m][e] : 1.0f;
                }
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][n][e] = fmaf(d[n], D[m][e], acc[m][n][e]);
            }
            if ((step & (kWideChain - 1)) == kWideChain - 1) {
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        tot[m][n] += acc[m][n];
                        acc[m][n] = zero;
                    }
            }
        }
    };
    if (__builtin_expect(__any(small), 0)) multiply(std::true_type{});
    else multiply(std::false_type{});
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no copy outlives its LDS
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) tot[m][n] += acc[m][n];

    // lane: rows r of its tiles, tokens 4 q + e of its groups.  The WK waves of a tile exchange their sums
    // through LDS, each adding and writing 4 / WK of the token groups.
    if constexpr (WK > 1) {
        __syncthreads();  // (every wave's last operands are read and its copies in)
        v4f* X = reinterpret_cast<v4f*>(smem);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) X[(wave * 16 + m * 4 + n) * 64 + lane] = tot[m][n];
        __syncthreads();
    }
#pragma unroll
    for (int mi = 0; mi < 4 / WK; ++mi) {
        const uint32_t m = wk * (4 / WK) + mi;
        v4f t4[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            if constexpr (WK == 1) {
                t4[n] = tot[mi][n];
            } else {
                const v4f* X = reinterpret_cast<const v4f*>(smem);
                t4[n] = X[((wave % (WM * WN)) * 16 + m * 4 + n) * 64 + lane];
#pragma unroll
                for (int k = 1; k < WK; ++k) t4[n] += X[((wave % (WM * WN) + k * WM * WN) * 16 + m * 4 + n) * 64 + lane];
            }
        }
        const uint32_t t0 = (mt0 * MG + wm * 4 + m) * 16 + 4 * q;
        v4f s = *gp(reinterpret_cast<const v4f*>(inv + t0));
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = fabsf(s[e]);
#pragma unroll
        for (int n = 0; n < 4; n += P) {
            const uint32_t row = tile_of(wn * 4 + n) * 16 + r;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t t = t0 + e;
                if (t >= a.T || row >= a.w.rows) continue;
                const float v = t4[n][e] * s[e];
                if constexpr (P == 2) {
                    a.y[(size_t)t * a.y_stride + row] = gelu_mul(v, t4[n + 1][e] * s[e]);
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

// Queries i0, i0 + step, ... (16 / step of them) of KV head h against the keys that each sees in [k_begin, k_end),
// in fp32 (plain_attention): where a wave's sums are not finite, an infinite cached value of a key that one
// query sees may have met the zero probability of another.
template <int D>
__device__ __forceinline__ void plain_queries(const BatchAttn& a, const uint16_t* kh, const uint16_t* vh, uint32_t h, uint32_t i0,
                                              uint32_t step, uint32_t c, uint32_t k_begin, uint32_t k_end) {
    const uint32_t lane = threadIdx.x & 63, q_heads = a.kv_heads * a.group;
#pragma unroll 1
    for (uint32_t qi = i0; qi < min(i0 + 16, a.T * a.group); qi += step) {
        const uint32_t t = qi / a.group, qh = h * a.group + qi % a.group, end = a.pos0 + t + 1;
        const float* src = a.q + ((size_t)t * q_heads + qh) * D + 4 * lane;
        float x[D / 64], o[D / 64], m, l;
#pragma unroll
        for (int e = 0; e < D / 64; ++e) x[e] = src[e / 4 * 256 + e % 4];
        const uint32_t lo = a.window && end > a.window ? end - a.window : 0u;
        plain_attention<D>(
            x, a.scale, max(lo, k_begin), min(end, k_end), [&](uint32_t key) { return kh + (size_t)(key % a.ring) * D; },
            [&](uint32_t key) { return vh + (size_t)(key % a.ring) * D; }, o, m, l);
        float* p = a.nchunks == 1 ? a.out + (size_t)t * a.out_stride + (size_t)qh * D
                                  : a.part + (((size_t)t * q_heads + qh) * a.nchunks + c) * (D + 2);
#pragma unroll
        for (int e = 0; e < D / 64; ++e) p[4 * lane + e / 4 * 256 + e % 4] = a.nchunks == 1 ? o[e] / l : o[e];
        if (a.nchunks > 1 && lane == 0) {
            p[D] = m;
            p[D + 1] = l;
        }
    }
}

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
        const float s = query_scale(mx);  // |q s| < 32
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
    float odd = 0.0f;  // NaN if a sum is not finite
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) odd = fmaf(acc[j][i], 0.0f, odd);
    if (__syncthreads_or(odd != 0.0f)) {
        plain_queries<D>(a, a.kcache + (size_t)h * a.ring * D, a.vcache + (size_t)h * a.ring * D, h, 16 * qt + wave, 4, c,
                         k_begin, k_end);
        return;
    }
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
        const float s = query_scale(mx);  // |q s| < 32
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
            // (the small products in a sum of their own: fewer additions round at the score's size.  A layer's error
            // against 64 bits over 512 positions 3.8e-7, with one sum 4.3e-7)
            v4f x = {0.0f, 0.0f, 0.0f, 0.0f}, xl = x;
#pragma unroll
            for (int s = 0; s < DS; ++s) {
                const v8h A = *reinterpret_cast<const v8h*>(ks + (16 * kt + m) * KP + 32 * s + 8 * q);
                x = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, qh[s], x, 0, 0, 0);
                xl = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, ql[s], xl, 0, 0, 0);
            }
            sv[kt] = x + xl;
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
    float odd = lrun * 0.0f;  // NaN if a sum is not finite
#pragma unroll
    for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) odd = fmaf(acc[j][e], 0.0f, odd);
    if (__any(odd != 0.0f)) {
        plain_queries<D>(a, kh, vh, h, 64 * qt + 16 * wave, 1, c, k_begin, k_end);
        return;
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

// Work split of a wide GEMM: 64 or 128 tokens x 128 rows per workgroup, wk waves sharing K inside it, S
// splits of K over workgroups (their sums added by the next kernel), S rounded down so that one round of
// workgroups holds them all (270 workgroups on 256 places took 82 us, 240 took 47).
// - 64 tokens: eight waves, four along K: a CU's 240 places hold a 15360-row gate/up pair once, and four waves
//   in one place leave it waiting (3840 -> 2 x 15360: 50 us against 113 with four waves of 64 x 256).
// - 128 tokens: eight waves, two along K, one workgroup per CU; or four waves, none along K, two workgroups
//   per CU, which hide each other's barriers but need twice the splits: the cheaper by wide_cost.
// A gate/up pair is not split (its epilogue needs whole sums).
struct WidePlan {
    uint32_t wk, mtiles, groups, S;
};
// Time in us of a 128-token form's `items` x S workgroups on 256 CUs, each S-th of K's blocks long, from rates
// measured over 96 cases (1,024 to 15,360 rows and columns, 96 to 512 tokens), partial sums included: a step of a
// CU's two workgroups of four waves 1.0 (one block each), of one alone 0.78, of one of eight waves 1.25 (two
// blocks); 11 more to start and end the former; planes written and read back at 5 TB/s.  The cheaper of
// the two by it was the faster but in 5 of the 96 (by 2-8 %): 4096 -> 3840, 512 tokens 52.2 us with eight waves (two
// splits) against 54.2 (four), 15360 -> 3840 148.6 against 137.4; 128 tokens 28.5 against 33.0 and 48.4 against 49.8; 512
// tokens, 3840 -> 8192 76.1 (no split) against 83.2, the 15360-row pair 300.9 against 253.7.
static double wide_cost(uint32_t wk, uint32_t items, uint32_t S, uint32_t rows, uint32_t blocks, uint32_t tokens) {
    const uint32_t steps = (blocks + S * wk - 1) / (S * wk), per = (items * S + 255) / 256;
    const double planes = S > 1 ? (double)S * tokens * rows * 4 / 5e6 : 0.0;
    return planes + (wk == 2 ? steps * 1.25 * per : steps * (per / 2 + 0.78 * (per % 2)) + 11.0);
}
static WidePlan wide_plan(uint32_t rows, uint32_t blocks, uint32_t tokens, bool pair) {
    constexpr uint32_t kCus = 256;
    const uint32_t m = wide_tokens(tokens), mtiles = (tokens + m - 1) / m, vrows = pair ? (rows + 31) / 32 * 64 : rows;
    const uint32_t groups = (vrows + 127) / 128, items = mtiles * groups;
    const auto splits = [&](uint32_t wk, uint32_t places) {
        return pair ? 1u : std::max<uint32_t>(1, std::min({places / items, kDeferParts, blocks / (kWideChain * wk)}));
    };
    if (m == 64) return WidePlan{4, mtiles, groups, splits(4, kCus)};
    const uint32_t S1 = splits(1, 2 * kCus), S2 = splits(2, kCus);
    // (of whole tiles: every pass of as many takes the same plan, for which batch_gemm_part_bytes sizes the planes)
    const uint32_t whole = mtiles * m;
    const bool two = wide_cost(2, items, S2, rows, blocks, whole) < wide_cost(1, items, S1, rows, blocks, whole);
    return WidePlan{two ? 2u : 1u, mtiles, groups, two ? S2 : S1};
}

size_t batch_image_bytes(uint32_t blocks, uint32_t tokens) {
    const size_t floats = (size_t)blocks * 128 * std::min(tokens, kBatchMax);
    return tokens > kBatchMax ? std::max(floats, ((size_t)blocks * (2048 + 64) + 64) * ((tokens + 127) / 128 * 8)) : floats;
}

size_t batch_gemm_part_need(uint32_t rows, uint32_t blocks, uint32_t tokens, bool gelu_pair) {
    const bool wide = tokens > kBatchMax;
    const uint32_t S = wide ? wide_plan(rows, blocks, tokens, gelu_pair).S : gemm_plan(rows, blocks, tokens, gelu_pair).S;
    const size_t planes = S * (wide || !gelu_pair ? 1u : 2u), prow = (rows + 15) / 16 * 16;  // (a wide pair is not split)
    return S > 1 ? planes * batch_padded(tokens) * prow * 4 : 0;
}

size_t batch_gemm_part_bytes(uint32_t rows, uint32_t blocks, uint32_t tokens, bool gelu_pair) {
    size_t most = 0;  // the largest over the passes of up to `tokens` tokens: one of each plan
    for (uint32_t t : {8u, 16u, 32u, 64u})
        if (t <= 32 || tokens > kBatchMax)
            most = std::max(most, batch_gemm_part_need(rows, blocks, std::min(t, tokens), gelu_pair));
    for (uint32_t t = 128; t < tokens + 128 && tokens > 64; t += 128)
        most = std::max(most, batch_gemm_part_need(rows, blocks, std::min(t, tokens), gelu_pair));
    return most;
}

size_t batch_gemm_counters(uint32_t rows, bool gelu_pair) {
    return 2 * gemm_plan(rows, 1, 1, gelu_pair).groups;  // (the fewest rows per group, two token groups)
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
    if (in.mode == BI_PLAIN) return hipErrorInvalidValue;  // (the GEMM reads x itself)
    {
        // float4 access to x, res, x_out and the norm weights
        const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
        if (in.stride % 4 || !a16(in.x) || !a16(in.res) || !a16(in.x_out) || !a16(in.w_a) || !a16(in.w_n))
            return hipErrorInvalidValue;
        const uint32_t octets = in.K / 8;
        const dim3 g(in.T);
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

template <int P, int G, bool PACK>
static hipError_t gemm_launch(const BatchGemm& a, hipStream_t s, uint32_t* parts) {
    const GemmPlan p = gemm_plan(a.w.rows, a.w.blocks, a.T, P == 2);
    constexpr uint32_t TR = 16 * G;
    const uint32_t Tp = (PACK ? 8 : TR) * p.tg;
    const bool defer = a.defer && P == 1 && p.S > 1;
    const uint64_t planes = (uint64_t)p.S * P * Tp * ((a.w.rows + 15) / 16 * 16) * 4;
    const bool fuse = p.S > 1 && !defer && a.counters && p.S <= (G == 2 ? kFuseSplits : kDeferParts) && planes < 0x7FFFFFFFu;
    if (p.S > 1 && (!a.part || a.part_bytes < planes)) return hipErrorInvalidValue;
    const uint32_t range = (a.w.nst + p.S - 1) / p.S;  // super-tiles, at most
    const size_t lds = std::max<size_t>((size_t)range * 4096 * (PACK ? 1 : 2 * G), 256 * p.waves * TR);  // (operands, later the waves' sums)
    const dim3 grid((p.groups * p.S + 7) / 8 * 8);
    if constexpr (G == 1) {
        if (p.waves == 8)
            hipLaunchKernelGGL((batch_gemm_kernel<1, PACK, P, 1, 8>), grid, dim3(512), lds, s, a, p.S, p.groups, p.tg, fuse ? 1u : 0u);
    }
    if constexpr (!PACK) {
        if (p.waves == 16)
            hipLaunchKernelGGL((batch_gemm_kernel<G, false, P, 2 * G, 16>), grid, dim3(1024), lds, s, a, p.S, p.groups, p.tg, fuse ? 1u : 0u);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.S == 1 || fuse) return e;
    if (defer) {
        if (parts) *parts = p.S;
        return hipSuccess;
    }
    const uint32_t n = a.T * a.w.rows;
    hipLaunchKernelGGL((batch_reduce_kernel<P>), dim3((n + 255) / 256), dim3(256), 0, s, a, p.S, Tp);
    return hipGetLastError();
}

template <int P>
static hipError_t wide_launch(const BatchGemm& a, hipStream_t s, uint32_t* parts) {
    const WidePlan p = wide_plan(a.w.rows, a.w.blocks, a.T, P == 2);
    const uint32_t S = p.S;
    if (S > 1 && (!a.part || a.part_bytes < batch_gemm_part_need(a.w.rows, a.w.blocks, a.T, P == 2))) return hipErrorInvalidValue;
    const dim3 grid((p.mtiles * p.groups * S + 7) / 8 * 8);
    if (p.wk == 4) hipLaunchKernelGGL((wide_gemm_kernel<1, 2, 4, P>), grid, dim3(512), 0, s, a, S, p.mtiles, p.groups);
    else if (p.wk == 2) hipLaunchKernelGGL((wide_gemm_kernel<2, 2, 2, P>), grid, dim3(512), 0, s, a, S, p.mtiles, p.groups);
    else hipLaunchKernelGGL((wide_gemm_kernel<2, 2, 1, P>), grid, dim3(256), 0, s, a, S, p.mtiles, p.groups);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || S == 1) return e;  // (S is 1 for a pair)
    if constexpr (P == 1) {
        if (!a.defer) {
            const uint32_t n = a.T * a.w.rows;
            hipLaunchKernelGGL((batch_reduce_kernel<1>), dim3((n + 255) / 256), dim3(256), 0, s, a, S, 16 * wide_groups(a.T));
            return hipGetLastError();
        }
        if (parts) *parts = S;
    }
    return hipSuccess;
}

hipError_t launch_batch_gemm(const BatchGemm& a, bool gelu_pair, hipStream_t s, uint32_t* parts) {
    if (parts) *parts = 0;
    if (a.T > kBatchMax && a.T <= kPassMax && a.w.rows && a.w.blocks &&
        !(gelu_pair && (a.w2.rows != a.w.rows || a.w2.blocks != a.w.blocks)))
        return gelu_pair ? wide_launch<2>(a, s, parts) : wide_launch<1>(a, s, parts);
    if (a.T == 0 || a.T > kBatchMax || a.w.rows == 0 || a.w.blocks == 0) return hipErrorInvalidValue;
    if (gelu_pair && (a.w2.rows != a.w.rows || a.w2.blocks != a.w.blocks)) return hipErrorInvalidValue;
    // float4 loads of the inputs
    if (!a.x || a.x_stride % 4 || reinterpret_cast<uintptr_t>(a.x) % 16) return hipErrorInvalidValue;
    if (a.T <= 8) return gelu_pair ? gemm_launch<2, 1, true>(a, s, parts) : gemm_launch<1, 1, true>(a, s, parts);
    if (a.T <= 16 || gemm_plan(a.w.rows, a.w.blocks, a.T, gelu_pair).tg == 2)
        return gelu_pair ? gemm_launch<2, 1, false>(a, s, parts) : gemm_launch<1, 1, false>(a, s, parts);
    return gelu_pair ? gemm_launch<2, 2, false>(a, s, parts) : gemm_launch<1, 2, false>(a, s, parts);
}

}  // namespace af
