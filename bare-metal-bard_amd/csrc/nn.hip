// Transformer building blocks of the GPT trainer for gfx950 -- the
// counterpart of bare-metal-bard's src/nn.cu (API: src/nn.h).
//
// Everything here is HBM-bound: arithmetic intensity below one flop per byte.
// The design rules are therefore about bytes, not flops:
//   * each tensor is read and written once, with 128-bit accesses (gfx950
//     global loads and stores need only 4-byte alignment, so rows of any
//     width use them, with 32-bit accesses at the ends of rows of odd width;
//     the embedding forward, the position-embedding gradient, the bias kernels
//     and rows too wide for the registers move odd widths by 32 bits only);
//   * a row-wise reduction (layernorm, softmax) gives a row to one wave64 (or,
//     for the 50k-wide vocabulary rows, one 1024-lane workgroup) that keeps the
//     whole row in registers between its passes, so the row is fetched once;
//   * reductions across rows (the layernorm weight/bias gradients, the bias
//     gradient, the gradient norm) never use floating-point atomics: blocks
//     write partial sums to a library-owned scratch buffer and a second kernel
//     adds them in a fixed order. The grid shapes depend only on the problem
//     shape, so every result is the same bit pattern on every call.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "nn_fused.hpp"
#include "workspace.hpp"
#include "../../include/nn.h"

using bmb::ceil_div;

namespace {

constexpr int NT = 256;
constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ float4 ldu4(const float *p) {
    float4 v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}
__device__ __forceinline__ void stu4(float *p, float4 v) { __builtin_memcpy(p, &v, sizeof(v)); }
// The same past the caches, for outputs that do not fit the 256 MB last-level
// cache beside the input of the same size and would only push out what the next
// kernel reads. Softmax and cross-entropy backward one after the other, rows of
// 50304, streamed and cached, in us: 64 MB of output 56 and 50, 128 MB 100 and
// 90, 192 MB 148 and 154, 256 MB 194 and 204, 512 MB 365 and 381, 1.6 GB 1112
// and 1183; the same sign at widths of 300-60000, but for some rows of the
// softmax (xent_launch).
constexpr size_t STREAM_BYTES = 160u << 20;
__device__ __forceinline__ void stu4_nt(float *p, float4 v) {
    typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
    __builtin_nontemporal_store(f4{v.x, v.y, v.z, v.w}, reinterpret_cast<f4 *>(p));
}
__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Grid size for a flat launch of `n` work items of NT lanes each.
inline unsigned grid_for(long long items) {
    return (unsigned)((items + NT - 1) / NT);
}

// Columns c..c+3 of a row of C: whole, or (RAG) those of them that exist, the
// others as `fill`.
template <bool RAG>
__device__ __forceinline__ float4 ld_cols(const float *row, int c, int C, float fill) {
    if (!RAG || (c >= 0 && c + 3 < C)) return ldu4(row + c);
    float4 v = make_float4(fill, fill, fill, fill);
    if (c + 0 >= 0 && c + 0 < C) v.x = row[c + 0];
    if (c + 1 >= 0 && c + 1 < C) v.y = row[c + 1];
    if (c + 2 >= 0 && c + 2 < C) v.z = row[c + 2];
    if (c + 3 >= 0 && c + 3 < C) v.w = row[c + 3];
    return v;
}
template <bool RAG>
__device__ __forceinline__ void st_cols(float *row, int c, int C, float4 v) {
    if (!RAG || (c >= 0 && c + 3 < C)) {
        stu4(row + c, v);
        return;
    }
    if (c + 0 >= 0 && c + 0 < C) row[c + 0] = v.x;
    if (c + 1 >= 0 && c + 1 < C) row[c + 1] = v.y;
    if (c + 2 >= 0 && c + 2 < C) row[c + 2] = v.z;
    if (c + 3 >= 0 && c + 3 < C) row[c + 3] = v.w;
}
// The same for rows as wide as an int reaches (c + 3 may pass it; c >= -3),
// compared as unsigned. (Of several ways to write the bound this one costs the
// ragged cross-entropy backward nothing, others 8%; here, in place of the
// above, it cost the token-embedding gradient 10% at 8192 positions x 65.)
template <bool RAG>
__device__ __forceinline__ float4 ld_cols_wide(const float *row, int c, int C) {
    const unsigned u = c, w = C;
    if (!RAG || (c >= 0 && u + 3 < w)) return ldu4(row + c);
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (u + 0 < w) v.x = row[c + 0];
    if (u + 1 < w) v.y = row[c + 1];
    if (u + 2 < w) v.z = row[c + 2];
    if (u + 3 < w) v.w = row[c + 3];
    return v;
}
__device__ __forceinline__ void st_cols_wide(float *row, int c, int C, float4 v) {
    const unsigned u = c, w = C;
    if (u + 0 < w) row[c + 0] = v.x;
    if (u + 1 < w) row[c + 1] = v.y;
    if (u + 2 < w) row[c + 2] = v.z;
    if (u + 3 < w) row[c + 3] = v.w;
}

// ------------------------------------------------------------ row/column maps
// Row-structured elementwise kernels split each row of width C into float4
// chunks (the last one may be partial): work item i is row i / C4, columns
// 4*(i % C4) .. +3, with C4 = ceil(C/4). VEC: C % 4 == 0, so every chunk is
// whole and rows are 4-byte aligned for the 128-bit accesses.

// out[r, c] = wte[tok[r], c] + wpe[r % T, c]   (src/nn.cu:23-36)
template <bool VEC>
__global__ __launch_bounds__(NT) void encoder_fwd_k(float *out, const int *tokens,
                                                     const float *wte, const float *wpe,
                                                     int T, int C, int C4, long long items) {
    const long long i = (long long)blockIdx.x * NT + threadIdx.x;
    if (i >= items) return;
    const int r = (int)(i / C4), c = (int)(i % C4) * 4;
    const int t = r % T;
    const float *e = wte + (size_t)tokens[r] * C + c;
    const float *p = wpe + (size_t)t * C + c;
    float *o = out + (size_t)r * C + c;
    if (VEC) {
        const float4 a = ldu4(e), b = ldu4(p);
        stu4(o, make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w));
    } else {
        for (int k = 0; k < 4 && c + k < C; ++k) o[k] = e[k] + p[k];
    }
}

// dwpe[t, c] += sum_b dout[b, t, c], b ascending.
template <bool VEC>
__global__ __launch_bounds__(NT) void encoder_bwd_wpe_k(float *dwpe, const float *dout, int B,
                                                         int T, int C, int C4, long long items) {
    const long long i = (long long)blockIdx.x * NT + threadIdx.x;
    if (i >= items) return;
    const int t = (int)(i / C4), c = (int)(i % C4) * 4;
    const size_t bstride = (size_t)T * C;
    const float *src = dout + (size_t)t * C + c;
    float *dst = dwpe + (size_t)t * C + c;
    if (VEC) {
        float4 s = zero4();
        for (int b = 0; b < B; ++b) {
            const float4 v = ldu4(src + b * bstride);
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        float4 d = ldu4(dst);
        d.x += s.x; d.y += s.y; d.z += s.z; d.w += s.w;
        stu4(dst, d);
    } else {
        for (int k = 0; k < 4 && c + k < C; ++k) {
            float s = 0.0f;
            for (int b = 0; b < B; ++b) s += src[b * bstride + k];
            dst[k] += s;
        }
    }
}

// dwte[tok, :] += sum over positions j with tokens[j] == tok, j ascending.
// One wave per position i (and strip of 256 NCH columns). A position that is
// not the first occurrence of its token leaves; the first one gathers every
// occurrence in order and owns the update of that wte row, so no two waves
// touch the same row. What bounds it is the pass over the ids: a chain of
// dependent loads where few tokens own many positions, and instructions where
// most positions are a token's only one. So it takes 256 Q ids at a time
// with 128-bit loads, and only where it finds the token lists the positions in
// LDS, in ascending order, and loads their rows eight at a time. (64 ids and
// one row per step took 53 us at 4096 positions of 65 tokens x 384, 81 us at
// 8192 of 50257 x 768 and 7.3 ms where all 8192 are one token; now 21, 52 and
// 1200 us.) Q is 4, or 1 up to WTE_FEW positions, where most of a step of 1024
// is past the end (us, Q = 1 against 4: 128 positions x 128 5.5 and 6.3, 512 x
// 768 7.1 and 7.7; 1024 x 128 10.6 and 9.8). Rows of odd width take strips as
// wide as the others (8192 x 767 of 50257: 71 us in strips of 768, 105 of 256).
constexpr int WTE_FEW = 512;

// ids[k] = the lane's ids tokens[j0 + 256 k + 4 lane + 0..3], `other` from
// position `end` on.
template <int Q>
__device__ __forceinline__ void load_ids(int4 (&ids)[Q], const int *tokens, int j0, int end,
                                         int other, int lane) {
    const int *p = tokens + j0 + 4 * lane;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        if (j0 + 256 * Q <= end) {
            __builtin_memcpy(&ids[k], p + 256 * k, sizeof(int4));
        } else {
            const int left = end - (j0 + 4 * lane + 256 * k);
            ids[k].x = left > 0 ? p[256 * k] : other;
            ids[k].y = left > 1 ? p[256 * k + 1] : other;
            ids[k].z = left > 2 ? p[256 * k + 2] : other;
            ids[k].w = left > 3 ? p[256 * k + 3] : other;
        }
    }
}
template <int Q>
__device__ __forceinline__ bool any_is(const int4 (&ids)[Q], int tok) {
    bool hit = false;
#pragma unroll
    for (int k = 0; k < Q; ++k)
        hit |= ids[k].x == tok || ids[k].y == tok || ids[k].z == tok || ids[k].w == tok;
    return __ballot(hit) != 0;
}

template <int NCH, bool VEC, int Q>
__global__ __launch_bounds__(NT) void encoder_bwd_wte_k(float *dwte, const float *dout,
                                                         const int *tokens, int N, int C) {
    __shared__ int found[NT / 64][256 * Q];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * (NT / 64) + wave;
    if (i >= N) return;
    const int tok = __builtin_amdgcn_readfirstlane(tokens[i]);
    int4 ids[Q];
    for (int j0 = 0; j0 < i; j0 += 256 * Q) {
        load_ids(ids, tokens, j0, i, ~tok, lane);
        if (any_is(ids, tok)) return;
    }
    const int c0 = blockIdx.y * 256 * NCH + lane * 4;
    int *list = found[wave];
    float4 s[NCH];
#pragma unroll
    for (int h = 0; h < NCH; ++h) s[h] = zero4();
    for (int j0 = i; j0 < N; j0 += 256 * Q) {
        load_ids(ids, tokens, j0, N, ~tok, lane);
        if (!any_is(ids, tok)) continue;
        int n = 0;
        const unsigned long long below = (1ULL << lane) - 1;
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const int id[4] = {ids[k].x, ids[k].y, ids[k].z, ids[k].w};
            int at = n;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned long long m = __ballot(id[e] == tok);
                at += __popcll(m & below);
                n += __popcll(m);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (id[e] == tok) list[at++] = j0 + 256 * k + 4 * lane + e;
        }
        // The list is this wave's own, and its LDS accesses are in order.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int q = 0; q < n; q += 8) {
            float4 v[8][NCH];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float *src = dout + (size_t)list[min(q + k, n - 1)] * C;
#pragma unroll
                for (int h = 0; h < NCH; ++h)
                    if (c0 + 256 * h < C) v[k][h] = ld_cols<!VEC>(src, c0 + 256 * h, C, 0.0f);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (q + k < n)
#pragma unroll
                    for (int h = 0; h < NCH; ++h) {
                        s[h].x += v[k][h].x; s[h].y += v[k][h].y;
                        s[h].z += v[k][h].z; s[h].w += v[k][h].w;
                    }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    float *dst = dwte + (size_t)tok * C;
#pragma unroll
    for (int h = 0; h < NCH; ++h) {
        const int c = c0 + 256 * h;
        if (c >= C) continue;
        float4 d = ld_cols<!VEC>(dst, c, C, 0.0f);
        d.x += s[h].x; d.y += s[h].y; d.z += s[h].z; d.w += s[h].w;
        st_cols<!VEC>(dst, c, C, d);
    }
}

// ------------------------------------------------------------------ layernorm
// One wave per row, the row held in NCH float4 registers per lane
// (C <= 256*NCH; RAG: C % 4 != 0, the row's last chunk is partial). Mean
// first, then the variance about it (src/nn.cu:54-82): biased, eps 1e-5. RES:
// the row is first formed as res_a + res_b and stored to res_out
// (residual_forward fused in front: the same one rounding per element, then
// the same layernorm of the stored sum).
template <int NCH, bool RES, bool RAG>
__global__ __launch_bounds__(NT) void ln_fwd_k(float *out, float *mean, float *rstd,
                                                const float *inp, const float *weight,
                                                const float *bias, int N, int C,
                                                float *res_out, const float *res_b) {
    const int row = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= N) return;
    const float *x = inp + (size_t)row * C;
    float4 v[NCH];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = (k * 64 + lane) * 4;
        v[k] = c < C ? ld_cols<RAG>(x, c, C, 0.0f) : zero4();
        if (RES && c < C) {
            const float4 y = ld_cols<RAG>(res_b + (size_t)row * C, c, C, 0.0f);
            v[k] = make_float4(v[k].x + y.x, v[k].y + y.y, v[k].z + y.z, v[k].w + y.w);
            st_cols<RAG>(res_out + (size_t)row * C, c, C, v[k]);
        }
        s += (v[k].x + v[k].y) + (v[k].z + v[k].w);
    }
    const float mu = wave_sum(s) / (float)C;
    float q = 0.0f;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = (k * 64 + lane) * 4;
        if (c < C) {
            const float a = v[k].x - mu;
            const float b = !RAG || c + 1 < C ? v[k].y - mu : 0.0f;
            const float d = !RAG || c + 2 < C ? v[k].z - mu : 0.0f;
            const float e = !RAG || c + 3 < C ? v[k].w - mu : 0.0f;
            q += (a * a + b * b) + (d * d + e * e);
        }
    }
    const float var = wave_sum(q) / (float)C;
    const float rs = rsqrtf(var + 1e-5f);
    if (lane == 0) {
        mean[row] = mu;
        rstd[row] = rs;
    }
    float *y = out + (size_t)row * C;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = (k * 64 + lane) * 4;
        if (c < C) {
            const float4 w = ld_cols<RAG>(weight, c, C, 0.0f);
            const float4 b = ld_cols<RAG>(bias, c, C, 0.0f);
            float4 o;
            o.x = ((v[k].x - mu) * rs) * w.x + b.x;
            o.y = ((v[k].y - mu) * rs) * w.y + b.y;
            o.z = ((v[k].z - mu) * rs) * w.z + b.z;
            o.w = ((v[k].w - mu) * rs) * w.w + b.w;
            st_cols<RAG>(y, c, C, o);
        }
    }
}

// Any C: one wave per row, three passes over the row.
__global__ __launch_bounds__(NT) void ln_fwd_generic_k(float *out, float *mean, float *rstd,
                                                        const float *inp, const float *weight,
                                                        const float *bias, int N, int C) {
    const int row = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= N) return;
    const float *x = inp + (size_t)row * C;
    float s = 0.0f;
    for (int c = lane; c < C; c += 64) s += x[c];
    const float mu = wave_sum(s) / (float)C;
    float q = 0.0f;
    for (int c = lane; c < C; c += 64) {
        const float d = x[c] - mu;
        q += d * d;
    }
    const float rs = rsqrtf(wave_sum(q) / (float)C + 1e-5f);
    if (lane == 0) {
        mean[row] = mu;
        rstd[row] = rs;
    }
    float *y = out + (size_t)row * C;
    for (int c = lane; c < C; c += 64) y[c] = ((x[c] - mu) * rs) * weight[c] + bias[c];
}

// Layernorm backward, fused (C <= 256*NCH; RAG: C % 4 != 0). A workgroup of
// LN_WAVES waves owns rows [blk*rpb, (blk+1)*rpb); each wave takes every
// LN_WAVES-th of them. Per row (src/nn.cu:85-111):
//   dinp += rstd * (dxhat - mean(dxhat) - xhat * mean(dxhat * xhat)),
//   dxhat = dout * w, xhat = (x - mean) * rstd.
// The weight and bias gradients of the workgroup's rows are summed in
// registers, combined across its waves through LDS in wave order, and written
// as partial[blk][0:C] (dweight) and partial[blk][C:2C] (dbias). SUM: also the
// column sums of the updated dinp, as partial[blk][2C:3C] (the gradient of a
// bias whose layer's output dinp is the gradient of; its own pass over dinp
// cost 5-10 us).
constexpr int LN_WAVES = 8;

template <int NCH, bool RAG, bool SUM>
__global__ __launch_bounds__(LN_WAVES * 64) void ln_bwd_k(
    float *dinp, float *partial, const float *dout, const float *inp, const float *weight,
    const float *mean, const float *rstd, int N, int C, int rpb) {
    constexpr int OUT = SUM ? 3 : 2;
    extern __shared__ float red[];  // [LN_WAVES][OUT * C]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float4 w[NCH], dw[NCH], db[NCH], ds[SUM ? NCH : 1];
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = (k * 64 + lane) * 4;
        w[k] = c < C ? ld_cols<RAG>(weight, c, C, 0.0f) : zero4();
        dw[k] = zero4();
        db[k] = zero4();
        if (SUM) ds[k] = zero4();
    }
    const int r0 = blockIdx.x * rpb;
    const int r1 = min(N, r0 + rpb);
    for (int r = r0 + wave; r < r1; r += LN_WAVES) {
        const float mu = mean[r], rs = rstd[r];
        const float *x = inp + (size_t)r * C;
        const float *dy = dout + (size_t)r * C;
        float4 xh[NCH], g[NCH];
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
            const int c = (k * 64 + lane) * 4;
            float4 xv = zero4();
            g[k] = zero4();
            if (c < C) {
                xv = ld_cols<RAG>(x, c, C, mu);  // (xhat 0 past the row's end)
                g[k] = ld_cols<RAG>(dy, c, C, 0.0f);
            }
            xh[k] = make_float4((xv.x - mu) * rs, (xv.y - mu) * rs, (xv.z - mu) * rs,
                                (xv.w - mu) * rs);
            const float4 d = make_float4(g[k].x * w[k].x, g[k].y * w[k].y, g[k].z * w[k].z,
                                         g[k].w * w[k].w);
            s1 += (d.x + d.y) + (d.z + d.w);
            s2 += (d.x * xh[k].x + d.y * xh[k].y) + (d.z * xh[k].z + d.w * xh[k].w);
        }
        const float m1 = wave_sum(s1) / (float)C;
        const float m2 = wave_sum(s2) / (float)C;
        float *dx = dinp + (size_t)r * C;
#pragma unroll
        for (int k = 0; k < NCH; ++k) {
            const int c = (k * 64 + lane) * 4;
            if (c < C) {
                float4 o = ld_cols<RAG>(dx, c, C, 0.0f);
                o.x += rs * (g[k].x * w[k].x - m1 - xh[k].x * m2);
                o.y += rs * (g[k].y * w[k].y - m1 - xh[k].y * m2);
                o.z += rs * (g[k].z * w[k].z - m1 - xh[k].z * m2);
                o.w += rs * (g[k].w * w[k].w - m1 - xh[k].w * m2);
                st_cols<RAG>(dx, c, C, o);
                if (SUM) {
                    ds[k].x += o.x; ds[k].y += o.y; ds[k].z += o.z; ds[k].w += o.w;
                }
                dw[k].x += g[k].x * xh[k].x; dw[k].y += g[k].y * xh[k].y;
                dw[k].z += g[k].z * xh[k].z; dw[k].w += g[k].w * xh[k].w;
                db[k].x += g[k].x; db[k].y += g[k].y; db[k].z += g[k].z; db[k].w += g[k].w;
            }
        }
    }
    float *mine = red + wave * OUT * C;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = (k * 64 + lane) * 4;
        if (c < C) {
            if (RAG) {
                st_cols<true>(mine, c, C, dw[k]);
                st_cols<true>(mine + C, c, C, db[k]);
                if (SUM) st_cols<true>(mine + 2 * C, c, C, ds[k]);
            } else {
                bmb::st4(mine + c, dw[k]);
                bmb::st4(mine + C + c, db[k]);
                if (SUM) bmb::st4(mine + 2 * C + c, ds[k]);
            }
        }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < OUT * C; j += LN_WAVES * 64) {
        float s = red[j];
#pragma unroll
        for (int q = 1; q < LN_WAVES; ++q) s += red[q * OUT * C + j];
        partial[(size_t)blockIdx.x * OUT * C + j] = s;
    }
}

// Any C: dinp only, one wave per row, scalar passes. The weight and bias
// gradients come from colsum_k<true> below.
__global__ __launch_bounds__(NT) void ln_bwd_dx_generic_k(float *dinp, const float *dout,
                                                           const float *inp, const float *weight,
                                                           const float *mean, const float *rstd,
                                                           int N, int C) {
    const int r = blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= N) return;
    const float mu = mean[r], rs = rstd[r];
    const float *x = inp + (size_t)r * C;
    const float *dy = dout + (size_t)r * C;
    float s1 = 0.0f, s2 = 0.0f;
    for (int c = lane; c < C; c += 64) {
        const float xh = (x[c] - mu) * rs, d = dy[c] * weight[c];
        s1 += d;
        s2 += d * xh;
    }
    const float m1 = wave_sum(s1) / (float)C, m2 = wave_sum(s2) / (float)C;
    float *dx = dinp + (size_t)r * C;
    for (int c = lane; c < C; c += 64) {
        const float xh = (x[c] - mu) * rs, d = dy[c] * weight[c];
        dx[c] += rs * (d - m1 - xh * m2);
    }
}

// Column sums over row chunks: block (strip, chunk) sums rows
// [chunk*rpc, (chunk+1)*rpc) of columns [strip*NT, strip*NT + NT), one column
// per lane, rows in ascending order.
//   LN == false: partial[chunk][c] = sum dout[r, c]                 (width C)
//   LN == true:  partial[chunk][c] = sum dout * xhat, [C + c] = sum dout (2C)
template <bool LN>
__global__ __launch_bounds__(NT) void colsum_k(float *partial, const float *dout,
                                                const float *inp, const float *mean,
                                                const float *rstd, int N, int C, int rpc) {
    const int c = blockIdx.x * NT + threadIdx.x;
    const int r0 = blockIdx.y * rpc;
    const int r1 = min(N, r0 + rpc);
    if (c >= C) return;
    float s0 = 0.0f, s1 = 0.0f;
    for (int r = r0; r < r1; ++r) {
        const float g = dout[(size_t)r * C + c];
        if (LN) s0 += g * ((inp[(size_t)r * C + c] - mean[r]) * rstd[r]);
        s1 += g;
    }
    const int width = LN ? 2 * C : C;
    float *p = partial + (size_t)blockIdx.y * width;
    if (LN) {
        p[c] = s0;
        p[C + c] = s1;
    } else {
        p[c] = s1;
    }
}

// The bias case of colsum_k with 128-bit loads (C % 4 == 0, dout 16-byte
// aligned): each lane owns 4 adjacent columns and adds its rows in the same
// order, so every column's partial sum is the same fp32 value as colsum_k's.
// Four times fewer load instructions; the row loop is unrolled so that
// several rows' loads are in flight at once.
__global__ __launch_bounds__(NT) void colsum4_k(float *partial, const float *dout, int N, int C,
                                                 int rpc) {
    const int C4 = C / 4;
    const int c4 = blockIdx.x * NT + threadIdx.x;
    const int r0 = blockIdx.y * rpc;
    const int r1 = min(N, r0 + rpc);
    if (c4 >= C4) return;
    const float4 *p = reinterpret_cast<const float4 *>(dout) + c4;
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
    for (int r = r0; r < r1; ++r) {
        const float4 g = p[(size_t)r * C4];
        s.x += g.x;
        s.y += g.y;
        s.z += g.z;
        s.w += g.w;
    }
    reinterpret_cast<float4 *>(partial + (size_t)blockIdx.y * C)[c4] = s;
}

// Each job's column sums over its G partial rows, added onto its destinations
// (ColsumJob). A workgroup covers FIN_COLS columns of one job with
// NT / FIN_COLS slices of lanes: slice q sums g = q, q + slices, ... in order,
// then the slice sums are added in slice order. Few columns per workgroup
// and many slices keep each lane's chain of dependent adds short (the
// partials are a few hundred rows and sit in L2; this kernel is latency-
// bound, 4.8-5.2 us for one job, so a caller with several runs them at once).
// J: the most jobs the launch holds; one job has a kernel of its own, without
// the search for the workgroup's job. (The destinations are read ahead of the
// sums and the search is without branches: as a chain of scalar loads ending in
// a vector load of the destination's address, the finish took 0.3 us longer.)
constexpr int FIN_COLS = 8;
template <int J>
struct ColsumJobs {
    bmb::ColsumJob job[J];
    int first[J + 1];  // job q: workgroups [first[q], first[q + 1])
};
template <int J>
__global__ __launch_bounds__(NT) void colsum_finish_k(ColsumJobs<J> jobs) {
    constexpr int SL = NT / FIN_COLS;
    __shared__ float sl[SL][FIN_COLS];
    int q = 0;
#pragma unroll
    for (int k = 1; k < J; ++k) q += (int)blockIdx.x >= jobs.first[k];
    const bmb::ColsumJob j = jobs.job[q];
    const int width = j.n[0] + j.n[1] + j.n[2], G = j.G;
    float *d0 = j.dst[0], *d1 = j.dst[1], *d2 = j.dst[2];
    const int col = threadIdx.x % FIN_COLS, slice = threadIdx.x / FIN_COLS;
    const int c = ((int)blockIdx.x - jobs.first[q]) * FIN_COLS + col;
    float s = 0.0f;
    if (c < width)
        for (int g = slice; g < G; g += SL) s += j.partial[(size_t)g * width + c];
    sl[slice][col] = s;
    __syncthreads();
    if (slice == 0 && c < width) {
        float t = sl[0][col];
        for (int k = 1; k < SL; ++k) t += sl[k][col];
        if (c < j.n[0])
            d0[c] += t;
        else if (c < j.n[0] + j.n[1])
            d1[c - j.n[0]] += t;
        else
            d2[c - j.n[0] - j.n[1]] += t;
    }
}

// ------------------------------------------------------------ elementwise ops
__device__ __forceinline__ float gelu1(float x) { return bmb::gelu(x); }
__device__ __forceinline__ float dgelu1(float x, float g) { return bmb::gelu_grad(x, g); }

// Flat elementwise map: work item i covers elements 4i .. 4i+3 (the last one
// may be partial); a grid-stride loop keeps the launch under the 2^32
// work-item limit of one dispatch for any n. OP is a functor with vec(base)
// and one(index).
constexpr long long MAP_MAX_BLOCKS = 1 << 20;

template <class OP>
__global__ __launch_bounds__(NT) void map_k(OP op, long long n) {
    const long long items = (n + 3) / 4;
    for (long long i = (long long)blockIdx.x * NT + threadIdx.x; i < items;
         i += (long long)gridDim.x * NT) {
        const long long base = i * 4;
        if (base + 3 < n)
            op.vec(base);
        else
            for (long long j = base; j < n; ++j) op.one(j);
    }
}

struct GeluFwd {
    float *out;
    const float *inp;
    __device__ void vec(long long i) const {
        const float4 x = ldu4(inp + i);
        stu4(out + i, make_float4(gelu1(x.x), gelu1(x.y), gelu1(x.z), gelu1(x.w)));
    }
    __device__ void one(long long i) const { out[i] = gelu1(inp[i]); }
};
struct GeluBwd {
    float *dinp;
    const float *inp, *dout;
    __device__ void vec(long long i) const {
        const float4 x = ldu4(inp + i), g = ldu4(dout + i);
        stu4(dinp + i, make_float4(dgelu1(x.x, g.x), dgelu1(x.y, g.y), dgelu1(x.z, g.z),
                                   dgelu1(x.w, g.w)));
    }
    __device__ void one(long long i) const { dinp[i] = dgelu1(inp[i], dout[i]); }
};
struct Residual {
    float *out;
    const float *a, *b;
    __device__ void vec(long long i) const {
        const float4 x = ldu4(a + i), y = ldu4(b + i);
        stu4(out + i, make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w));
    }
    __device__ void one(long long i) const { out[i] = a[i] + b[i]; }
};
struct AddInplace {
    float *dst;
    const float *src;
    __device__ void vec(long long i) const {
        const float4 x = ldu4(dst + i), y = ldu4(src + i);
        stu4(dst + i, make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w));
    }
    __device__ void one(long long i) const { dst[i] += src[i]; }
};
struct Zero {
    float *p;
    __device__ void vec(long long i) const { stu4(p + i, zero4()); }
    __device__ void one(long long i) const { p[i] = 0.0f; }
};

// AdamW (src/nn.cu:240-255, 336-343) with the reference's fp32 operation order. FP
// contraction is off here so that each product and sum rounds separately, as
// written; the result is then a function of the inputs alone.
__device__ __forceinline__ void adam1(float &p, float &m, float &v, float grad, float lr,
                                      float beta1, float beta2, float eps, float wd, float bc1,
                                      float bc2, float gscale) {
#pragma clang fp contract(off)
    const float g = grad * gscale;
    const float mi = beta1 * m + (1.0f - beta1) * g;
    const float vi = beta2 * v + (1.0f - beta2) * g * g;
    m = mi;
    v = vi;
    const float mhat = mi / bc1;
    const float vhat = vi / bc2;
    p = p - lr * (mhat / (sqrtf(vhat) + eps) + wd * p);
}

struct AdamW {
    float *params;
    const float *grads;
    float *m, *v;
    float lr, beta1, beta2, eps, wd, bc1, bc2, gscale;
    __device__ void one(long long i) const {
        float p = params[i], mi = m[i], vi = v[i];
        adam1(p, mi, vi, grads[i], lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
        params[i] = p;
        m[i] = mi;
        v[i] = vi;
    }
    __device__ void vec(long long i) const {
        float4 p = ldu4(params + i), mi = ldu4(m + i), vi = ldu4(v + i);
        const float4 g = ldu4(grads + i);
        adam1(p.x, mi.x, vi.x, g.x, lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
        adam1(p.y, mi.y, vi.y, g.y, lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
        adam1(p.z, mi.z, vi.z, g.z, lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
        adam1(p.w, mi.w, vi.w, g.w, lr, beta1, beta2, eps, wd, bc1, bc2, gscale);
        stu4(params + i, p);
        stu4(m + i, mi);
        stu4(v + i, vi);
    }
};

template <class OP>
void run_map(const OP &op, long long n) {
    if (n <= 0) return;
    const long long blocks = std::min(MAP_MAX_BLOCKS, ((n + 3) / 4 + NT - 1) / NT);
    bmb::launch(map_k<OP>, dim3((unsigned)blocks), dim3(NT), 0, nullptr, op, n);
}

// out[r, c] += bias[c]
template <bool VEC>
__global__ __launch_bounds__(NT) void bias_fwd_k(float *out, const float *bias, int C, int C4,
                                                  long long items) {
    const long long i = (long long)blockIdx.x * NT + threadIdx.x;
    if (i >= items) return;
    const int r = (int)(i / C4), c = (int)(i % C4) * 4;
    float *o = out + (size_t)r * C + c;
    if (VEC) {
        float4 v = ldu4(o);
        const float4 b = ldu4(bias + c);
        v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
        stu4(o, v);
    } else {
        for (int k = 0; k < 4 && c + k < C; ++k) o[k] += bias[c + k];
    }
}

// dlogits[r, i] = (probs[r, i] - [i == target]) * scale for i < V, 0 beyond.
// One chunk of four columns per lane (four chunks: 618 instead of 532 us at
// 8192 x 50304). RAG: Vp % 4 != 0; a row's chunks then start at the columns
// that are 16-byte aligned in it, so all but its first and last are still moved
// by aligned 128-bit accesses. nt: streaming stores (STREAM_BYTES).
// per: FLAT, a row's chunks, which lane i of the launch divides into row and
// chunk; otherwise a row's workgroups (the row is uniform).
template <bool RAG, bool FLAT>
__global__ __launch_bounds__(NT) void xent_bwd_k(float *dlogits, const float *probs,
                                                  const int *targets, int N, int V, int Vp,
                                                  unsigned per, float scale, bool nt) {
    unsigned r, k;  // row, chunk of it
    if (FLAT) {
        const unsigned i = blockIdx.x * NT + threadIdx.x;
        r = i / per;
        k = i - r * per;
        if (r >= (unsigned)N) return;
    } else {
        r = blockIdx.x / per;
        k = blockIdx.x % per * NT + threadIdx.x;
    }
    const int tgt = targets[r];
    const float *p = probs + (size_t)r * Vp;
    float *d = dlogits + (size_t)r * Vp;
    const int first = RAG ? -(int)(((size_t)r * Vp) & 3) : 0;
    const unsigned c3 = k * 4 + (first + 3);  // c + 3, as unsigned
    if (c3 >= Vp + 3u) return;
    const int c = (int)(c3 - 3);
    const float4 v = ld_cols_wide<RAG>(p, c, Vp);
    const unsigned hit = (unsigned)tgt - (unsigned)c;  // the target's place in the chunk
    float4 o;
    o.x = c < V - 0 ? (v.x - (hit == 0 ? 1.0f : 0.0f)) * scale : 0.0f;
    o.y = c < V - 1 ? (v.y - (hit == 1 ? 1.0f : 0.0f)) * scale : 0.0f;
    o.z = c < V - 2 ? (v.z - (hit == 2 ? 1.0f : 0.0f)) * scale : 0.0f;
    o.w = c < V - 3 ? (v.w - (hit == 3 ? 1.0f : 0.0f)) * scale : 0.0f;
    if (RAG && (c < 0 || (unsigned)c + 3 >= (unsigned)Vp))
        st_cols_wide(d, c, Vp, o);
    else if (nt)
        stu4_nt(d + c, o);
    else
        stu4(d + c, o);
}

// ------------------------------------------------------- softmax + cross-entropy
// One workgroup of NTHR lanes per row, the row's first V logits held in NCH
// float4 registers per lane (V <= 4*NTHR*NCH; RAG: Vp % 4 != 0, chunks placed
// as in xent_bwd_k and V <= 4*NTHR*NCH - 3; 2048 x 50257 485 -> 222 us against
// the three-pass kernel below): max, then
// exp(x - max) and its sum, then the normalised probabilities -- one read of
// the logits and one write of the probabilities (src/nn.cu:197-221).
// exp(x - m) is exp2((x - m) * log2 e) on v_exp_f32.
template <int NTHR>
__device__ __forceinline__ float block_reduce(float v, float *sh, bool is_max) {
    constexpr int NW = NTHR / 64;
    v = is_max ? wave_max(v) : wave_sum(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();  // sh may still be read by a previous reduction
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    float r = sh[0];
#pragma unroll
    for (int k = 1; k < NW; ++k) r = is_max ? fmaxf(r, sh[k]) : r + sh[k];
    return r;
}

__device__ __forceinline__ float xent_loss(float p) { return -logf(fmaxf(p, 1e-30f)); }

// Columns c..c+3 of a row of C >= 4. RAG: without a branch per element (those
// made the 16-chunk kernel spill 72 registers): a chunk that runs past the
// row's end is loaded as the row's last four columns and shifted into place
// (what follows the last column is unspecified); one that starts before the
// row reads the end of the row before (c >= 0 in row 0).
template <bool RAG>
__device__ __forceinline__ float4 ld_row_end(const float *row, int c, int C) {
    if (!RAG) return ldu4(row + c);
    const int at = min(c, C - 4), n = c - at;
    const float4 v = ldu4(row + at);
    return make_float4(n == 0 ? v.x : n == 1 ? v.y : n == 2 ? v.z : v.w,
                       n == 0 ? v.y : n == 1 ? v.z : v.w, n == 0 ? v.z : v.w, v.w);
}

template <int NTHR, int NCH, bool RAG, bool STREAM>
__global__ __launch_bounds__(NTHR) void softmax_xent_k(float *probs, float *losses,
                                                        const float *logits, const int *targets,
                                                        int V, int Vp) {
    __shared__ float sh[NTHR / 64];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float *x = logits + (size_t)row * Vp;
    float *p = probs + (size_t)row * Vp;
    const int first = RAG ? -(int)(((size_t)row * Vp) & 3) : 0;
    float4 v[NCH];
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = first + (k * NTHR + tid) * 4;
        v[k] = c < V ? ld_row_end<RAG>(x, c, Vp)
                     : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        if (RAG && c + 0 < 0) v[k].x = -INFINITY;
        if (RAG && c + 1 < 0) v[k].y = -INFINITY;
        if (RAG && c + 2 < 0) v[k].z = -INFINITY;
        if (c + 1 >= V) v[k].y = -INFINITY;
        if (c + 2 >= V) v[k].z = -INFINITY;
        if (c + 3 >= V) v[k].w = -INFINITY;
        m = fmaxf(m, fmaxf(fmaxf(v[k].x, v[k].y), fmaxf(v[k].z, v[k].w)));
    }
    m = block_reduce<NTHR>(m, sh, true);
    const float ml = m * LOG2E;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        v[k].x = __builtin_amdgcn_exp2f(v[k].x * LOG2E - ml);
        v[k].y = __builtin_amdgcn_exp2f(v[k].y * LOG2E - ml);
        v[k].z = __builtin_amdgcn_exp2f(v[k].z * LOG2E - ml);
        v[k].w = __builtin_amdgcn_exp2f(v[k].w * LOG2E - ml);
        s += (v[k].x + v[k].y) + (v[k].z + v[k].w);
    }
    s = block_reduce<NTHR>(s, sh, false);
    const float inv = 1.0f / s;
    const int tgt = targets[row];
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int c = first + (k * NTHR + tid) * 4;
        const float4 o = make_float4(v[k].x * inv, v[k].y * inv, v[k].z * inv, v[k].w * inv);
        // (Columns in [V, Vp) come out as exp2(-inf) = 0.)
        if (RAG ? c >= 0 && c + 3 < Vp : c < Vp) STREAM ? stu4_nt(p + c, o) : stu4(p + c, o);
        if (tgt >= c && tgt < c + 4 && tgt >= 0 && tgt < V) {
            const int j = tgt - c;
            const float pt = j == 0 ? o.x : j == 1 ? o.y : j == 2 ? o.z : o.w;
            losses[row] = xent_loss(pt);
        }
    }
    // (Unsigned: c passes the largest int behind a Vp near it.)
    for (unsigned c = first + (NCH * NTHR + tid) * 4; c < (unsigned)Vp; c += NTHR * 4)
        if (!RAG || (int)c < Vp - 3) stu4(p + c, zero4());
    // A row with a NaN or an infinity (uniform, rare): 0 * inv made its padding
    // NaN; each lane clears what it wrote there. (Zeroed before the store, every
    // row paid for it: 0.8 us of 10 at 64 x 50304.)
    if (!(inv < INFINITY))
        for (int c = first + tid * 4; c < min(Vp, NCH * NTHR * 4); c += NTHR * 4)
            for (int j = max(c, V); j < min(c + 4, Vp); ++j) p[j] = 0.0f;
    if (RAG) {
        // The columns of the row's partial chunks (up to three at each end),
        // one lane each, from the logits again (with the same arithmetic).
        const int end = Vp - (((unsigned)Vp - first) & 3), head = first < 0 ? first + 4 : 0;
        const int at = tid < 4 ? 0 : max(end, head), e = tid & 3;
        if (tid < 8 && e < (tid < 4 ? head : Vp - at))
            p[at + e] = at + e < V ? __builtin_amdgcn_exp2f(x[at + e] * LOG2E - ml) * inv : 0.0f;
    }
    if (tid == 0) {
        if (tgt >= V && tgt < Vp) losses[row] = xent_loss(0.0f);
        if (tgt < 0 || tgt >= Vp) losses[row] = NAN;
    }
}

// Any V, Vp: three passes over the row with scalar accesses.
__global__ __launch_bounds__(NT) void softmax_xent_generic_k(float *probs, float *losses,
                                                              const float *logits,
                                                              const int *targets, int V, int Vp) {
    __shared__ float sh[NT / 64];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float *x = logits + (size_t)row * Vp;
    float *p = probs + (size_t)row * Vp;
    float m = -INFINITY;
    for (int i = tid; i < V; i += NT) m = fmaxf(m, x[i]);
    m = block_reduce<NT>(m, sh, true);
    const float ml = m * LOG2E;
    float s = 0.0f;
    for (int i = tid; i < V; i += NT) {
        const float e = __builtin_amdgcn_exp2f(x[i] * LOG2E - ml);
        p[i] = e;
        s += e;
    }
    s = block_reduce<NT>(s, sh, false);
    const float inv = 1.0f / s;
    // Each lane rescales exactly the entries it wrote, so no barrier is needed.
    for (int i = tid; i < V; i += NT) p[i] *= inv;
    for (int i = V + tid; i < Vp; i += NT) p[i] = 0.0f;
    const int tgt = targets[row];
    if (tgt >= 0 && tgt < V && (tgt % NT) == tid) losses[row] = xent_loss(p[tgt]);
    if (tid == 0) {
        if (tgt >= V && tgt < Vp) losses[row] = xent_loss(0.0f);
        if (tgt < 0 || tgt >= Vp) losses[row] = NAN;
    }
}

// ------------------------------------------------------------- scalar results
// sum of squares in fp64: NORM_BLOCKS partials, then one workgroup adds them.
constexpr int NORM_BLOCKS = 1024;

__global__ __launch_bounds__(NT) void sumsq_k(double *partial, const float *g, long long n) {
    __shared__ double sh[NT / 64];
    double acc = 0.0;
    const long long n4 = n / 4;
    for (long long i = (long long)blockIdx.x * NT + threadIdx.x; i < n4;
         i += (long long)gridDim.x * NT) {
        const float4 v = ldu4(g + 4 * i);
        acc += (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z + (double)v.w * v.w;
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
        const double v = g[4 * n4 + threadIdx.x];
        acc += v * v;
    }
    acc = wave_sum_d(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// out = sqrt(sum partial) (SQRT) or sum(partial) / n, one workgroup.
template <bool SQRT>
__global__ __launch_bounds__(NT) void finish_scalar_k(float *out, const double *partial,
                                                       int count, long long n) {
    __shared__ double sh[NT / 64];
    double acc = 0.0;
    for (int i = threadIdx.x; i < count; i += NT) acc += partial[i];
    acc = wave_sum_d(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double s = (sh[0] + sh[1]) + (sh[2] + sh[3]);
        *out = SQRT ? (float)sqrt(s) : (float)(s / (double)n);
    }
}

// Sum of n floats in fp64 into partial[blockIdx.x] (grid-stride, scalar).
__global__ __launch_bounds__(NT) void sum_k(double *partial, const float *x, long long n) {
    __shared__ double sh[NT / 64];
    double acc = 0.0;
    for (long long i = (long long)blockIdx.x * NT + threadIdx.x; i < n;
         i += (long long)gridDim.x * NT)
        acc += x[i];
    acc = wave_sum_d(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// ------------------------------------------------------------------ host side
// The partial sums of a reduction live in a buffer leased for the call
// (workspace.hpp). A void op that cannot get one stops the process, as the
// reference's CUDA_CHECK does on any CUDA error (src/gpt.cu:18-26): returning
// would leave its gradients unwritten with nothing to tell the caller.
[[noreturn]] void scratch_failure(const char *what) {
    fprintf(stderr, "bmb: %s: cannot allocate the reduction scratch buffer\n", what);
    exit(1);
}

// Number of float4 chunks per lane for the register-resident row kernels.
int row_chunks(int C) {
    const int n = ceil_div(C, 256);
    return n <= 4 ? n : n <= 8 ? 8 : 0;
}

// Column-sum launch for dout (N, C): G row chunks of rpc rows, chosen from the
// shape alone so that strips * G is about 1024 workgroups.
void colsum_shape(int N, int C, int &rpc, int &G) {
    const int strips = ceil_div(C, NT);
    int g = std::max(1, std::min(ceil_div(N, 16), ceil_div(1024, strips)));
    rpc = ceil_div(N, g);
    G = ceil_div(N, rpc);
}

template <int J>
void colsum_launch(const bmb::ColsumJob *jobs, int count) {
    ColsumJobs<J> a{};
    for (int q = 0; q < J; ++q) {
        if (q < count) a.job[q] = jobs[q];
        const int width = a.job[q].n[0] + a.job[q].n[1] + a.job[q].n[2];
        a.first[q + 1] = a.first[q] + (q < count ? ceil_div(width, FIN_COLS) : 0);
    }
    bmb::launch(colsum_finish_k<J>, dim3(a.first[J]), dim3(NT), 0, nullptr, a);
}

template <int NCH, bool RES>
void ln_fwd_launch(float *out, float *mean, float *rstd, const float *inp, const float *w,
                   const float *b, int N, int C, float *res_out = nullptr,
                   const float *res_b = nullptr) {
    bmb::launch(C % 4 == 0 ? ln_fwd_k<NCH, RES, false> : ln_fwd_k<NCH, RES, true>,
                dim3(ceil_div(N, NT / 64)), dim3(NT), 0, nullptr, out, mean, rstd, inp, w, b, N, C,
                res_out, res_b);
}

// The register-resident forward, if a row fits; false if not.
template <bool RES>
bool ln_fwd_rows(float *out, float *mean, float *rstd, const float *inp, const float *w,
                 const float *b, int N, int C, float *res_out = nullptr,
                 const float *res_b = nullptr) {
    switch (row_chunks(C)) {
        case 1: ln_fwd_launch<1, RES>(out, mean, rstd, inp, w, b, N, C, res_out, res_b); break;
        case 2: ln_fwd_launch<2, RES>(out, mean, rstd, inp, w, b, N, C, res_out, res_b); break;
        case 3: ln_fwd_launch<3, RES>(out, mean, rstd, inp, w, b, N, C, res_out, res_b); break;
        case 4: ln_fwd_launch<4, RES>(out, mean, rstd, inp, w, b, N, C, res_out, res_b); break;
        case 8: ln_fwd_launch<8, RES>(out, mean, rstd, inp, w, b, N, C, res_out, res_b); break;
        default: return false;
    }
    return true;
}

// Row groups of the fused layernorm backward: G workgroups of rpb rows, about
// 256 of them, whole waves of rows.
void ln_bwd_shape(int N, int &rpb, int &G) {
    const int G0 = std::max(1, std::min(256, ceil_div(N, LN_WAVES)));
    rpb = ceil_div(ceil_div(N, G0), LN_WAVES) * LN_WAVES;
    G = ceil_div(N, rpb);
}

template <int NCH, bool SUM>
void ln_bwd_launch(float *dinp, float *partial, const float *dout, const float *inp,
                   const float *w, const float *mean, const float *rstd, int N, int C, int rpb,
                   int G) {
    const size_t smem = (size_t)LN_WAVES * (SUM ? 3 : 2) * C * sizeof(float);
    auto *kern = C % 4 == 0 ? ln_bwd_k<NCH, false, SUM> : ln_bwd_k<NCH, true, SUM>;
    bmb::allow_smem(kern, smem);
    bmb::launch(kern, dim3(G), dim3(LN_WAVES * 64), smem, nullptr, dinp, partial, dout, inp, w,
                mean, rstd, N, C, rpb);
}

template <bool SUM>
void ln_bwd_rows(float *dinp, float *partial, const float *dout, const float *inp, const float *w,
                 const float *mean, const float *rstd, int N, int C, int rpb, int G) {
    switch (row_chunks(C)) {
        case 1: ln_bwd_launch<1, SUM>(dinp, partial, dout, inp, w, mean, rstd, N, C, rpb, G); break;
        case 2: ln_bwd_launch<2, SUM>(dinp, partial, dout, inp, w, mean, rstd, N, C, rpb, G); break;
        case 3: ln_bwd_launch<3, SUM>(dinp, partial, dout, inp, w, mean, rstd, N, C, rpb, G); break;
        case 4: ln_bwd_launch<4, SUM>(dinp, partial, dout, inp, w, mean, rstd, N, C, rpb, G); break;
        default: ln_bwd_launch<8, SUM>(dinp, partial, dout, inp, w, mean, rstd, N, C, rpb, G); break;
    }
}

// One workgroup of nt lanes per row, N rows in as many launches as that takes:
// a dispatch holds fewer than 2^32 lanes. go(r, n): rows [r, r + n).
template <class F>
void rows_in_launches(int N, int nt, F &&go) {
    const int most = (int)(((1LL << 32) - 1) / nt);
    for (int r = 0; r < N; r += std::min(most, N - r)) go(r, std::min(most, N - r));
}

template <int NTHR, int NCH>
void xent_launch(float *probs, float *losses, const float *logits, const int *targets, int N,
                 int V, int Vp) {
    // Rows that leave a quarter or more of the 1024 x 8 chunks empty are faster
    // cached from 1.5 times the cache on (1 GB of 20000 columns 380 us against 406,
    // of 17000 409 against 453; 28000: 392 against 376; 192 MB of 20000: 86 against 75).
    const size_t bytes = (size_t)N * Vp * sizeof(float);
    const bool sparse = NTHR == 1024 && NCH == 8 && V <= 24576 && bytes >= 384u << 20;
    const bool stream = bytes >= STREAM_BYTES && !sparse;
    auto *kern = Vp % 4 == 0 ? (stream ? softmax_xent_k<NTHR, NCH, false, true>
                                       : softmax_xent_k<NTHR, NCH, false, false>)
                             : (stream ? softmax_xent_k<NTHR, NCH, true, true>
                                       : softmax_xent_k<NTHR, NCH, true, false>);
    rows_in_launches(N, NTHR, [&](int r, int n) {
        const size_t off = (size_t)r * Vp;
        bmb::launch(kern, dim3(n), dim3(NTHR), 0, nullptr, probs + off, losses + r, logits + off,
                    targets + r, V, Vp);
    });
}

float scalar_result(const float *dptr) {
    float h = NAN;
    const hipError_t e = hipMemcpy(&h, dptr, sizeof(float), hipMemcpyDeviceToHost);
    bmb::note_launch_status(e);
    return e == hipSuccess ? h : NAN;
}

}  // namespace

void bmb::residual_layernorm_forward(float *res_out, float *ln_out, float *mean, float *rstd,
                                     const float *a, const float *b, const float *weight,
                                     const float *bias, int N, int C) {
    if (N <= 0 || C <= 0) return;
    if (ln_fwd_rows<true>(ln_out, mean, rstd, a, weight, bias, N, C, res_out, b)) return;
    residual_forward(res_out, a, b, N * C);
    layernorm_forward(ln_out, mean, rstd, res_out, weight, bias, N, C);
}

void bmb::colsum_finish_jobs(const ColsumJob *jobs, int count) {
    if (count <= 0) return;
    if (count == 1)
        colsum_launch<1>(jobs, count);
    else
        colsum_launch<COLSUM_JOBS>(jobs, count);
}

size_t bmb::bias_partial_floats(int N, int C) {
    int rpc, G;
    colsum_shape(N, C, rpc, G);
    return (size_t)G * C;
}

bmb::ColsumJob bmb::bias_backward_partial(float *dbias, const float *dout, int N, int C,
                                          float *partial) {
    int rpc, G;
    colsum_shape(N, C, rpc, G);
    if (C % 4 == 0 && ((uintptr_t)dout & 15u) == 0)
        launch(colsum4_k, dim3(ceil_div(C / 4, NT), G), dim3(NT), 0, nullptr, partial, dout, N, C,
               rpc);
    else
        launch(colsum_k<false>, dim3(ceil_div(C, NT), G), dim3(NT), 0, nullptr, partial, dout,
               nullptr, nullptr, nullptr, N, C, rpc);
    return ColsumJob{partial, {dbias, nullptr, nullptr}, {C, 0, 0}, G};
}

size_t bmb::layernorm_partial_floats(int N, int C) {
    int rpb, G;
    ln_bwd_shape(N, rpb, G);
    return (size_t)G * 3 * C;
}

bool bmb::layernorm_backward_partial(float *dinp, float *dweight, float *dbias, float *dsum,
                                     const float *dout, const float *inp, const float *weight,
                                     const float *mean, const float *rstd, int N, int C,
                                     float *partial, ColsumJob &job) {
    // (The waves' sums of three columns arrays fit a CU's 160 KB of LDS.)
    if (row_chunks(C) == 0 || (size_t)LN_WAVES * 3 * C * sizeof(float) > 160 * 1024) {
        layernorm_backward(dinp, dweight, dbias, dout, inp, weight, mean, rstd, N, C);
        if (dsum != nullptr) bias_backward(dsum, dinp, N, C);
        return false;
    }
    int rpb, G;
    ln_bwd_shape(N, rpb, G);
    if (dsum != nullptr)
        ln_bwd_rows<true>(dinp, partial, dout, inp, weight, mean, rstd, N, C, rpb, G);
    else
        ln_bwd_rows<false>(dinp, partial, dout, inp, weight, mean, rstd, N, C, rpb, G);
    job = ColsumJob{partial, {dweight, dbias, dsum}, {C, C, dsum != nullptr ? C : 0}, G};
    return true;
}

extern "C" {

void encoder_forward(float *out, const int *tokens, const float *wte, const float *wpe, int B,
                     int T, int C) {
    if (B <= 0 || T <= 0 || C <= 0) return;
    const int C4 = ceil_div(C, 4);
    const long long items = (long long)B * T * C4;
    if (C % 4 == 0)
        bmb::launch(encoder_fwd_k<true>, dim3(grid_for(items)), dim3(NT), 0, nullptr, out,
                    tokens, wte, wpe, T, C, C4, items);
    else
        bmb::launch(encoder_fwd_k<false>, dim3(grid_for(items)), dim3(NT), 0, nullptr, out,
                    tokens, wte, wpe, T, C, C4, items);
}

void encoder_backward(float *dwte, float *dwpe, const float *dout, const int *tokens, int B,
                      int T, int C) {
    if (B <= 0 || T <= 0 || C <= 0) return;
    const int C4 = ceil_div(C, 4);
    const long long items = (long long)T * C4;
    if (C % 4 == 0)
        bmb::launch(encoder_bwd_wpe_k<true>, dim3(grid_for(items)), dim3(NT), 0, nullptr, dwpe,
                    dout, B, T, C, C4, items);
    else
        bmb::launch(encoder_bwd_wpe_k<false>, dim3(grid_for(items)), dim3(NT), 0, nullptr,
                    dwpe, dout, B, T, C, C4, items);
    const int N = B * T;
    const bool vec = C % 4 == 0, few = N <= WTE_FEW;
    auto wte = [&](auto nch) {
        constexpr int NC = decltype(nch)::value;
        bmb::launch(vec ? few ? encoder_bwd_wte_k<NC, true, 1> : encoder_bwd_wte_k<NC, true, 4>
                        : few ? encoder_bwd_wte_k<NC, false, 1> : encoder_bwd_wte_k<NC, false, 4>,
                    dim3(ceil_div(N, NT / 64), ceil_div(C, 256 * NC)), dim3(NT), 0, nullptr, dwte,
                    dout, tokens, N, C);
    };
    if (C <= 256) wte(std::integral_constant<int, 1>{});
    else if (C <= 512) wte(std::integral_constant<int, 2>{});
    else wte(std::integral_constant<int, 3>{});
}

void layernorm_forward(float *out, float *mean, float *rstd, const float *inp,
                       const float *weight, const float *bias, int N, int C) {
    if (N <= 0 || C <= 0) return;
    if (!ln_fwd_rows<false>(out, mean, rstd, inp, weight, bias, N, C))
        bmb::launch(ln_fwd_generic_k, dim3(ceil_div(N, NT / 64)), dim3(NT), 0, nullptr, out, mean,
                    rstd, inp, weight, bias, N, C);
}

void layernorm_backward(float *dinp, float *dweight, float *dbias, const float *dout,
                        const float *inp, const float *weight, const float *mean,
                        const float *rstd, int N, int C) {
    if (N <= 0 || C <= 0) return;
    if (row_chunks(C) > 0) {
        int rpb, G;
        ln_bwd_shape(N, rpb, G);
        bmb::ScratchLease ws(bmb::SCRATCH_NN, (size_t)G * 2 * C * sizeof(float));
        if (!ws) scratch_failure("layernorm_backward");
        float *partial = static_cast<float *>(ws.get());
        ln_bwd_rows<false>(dinp, partial, dout, inp, weight, mean, rstd, N, C, rpb, G);
        const bmb::ColsumJob job{partial, {dweight, dbias, nullptr}, {C, C, 0}, G};
        bmb::colsum_finish_jobs(&job, 1);
        return;
    }
    int rpc, G;
    colsum_shape(N, C, rpc, G);
    bmb::ScratchLease ws(bmb::SCRATCH_NN, (size_t)G * 2 * C * sizeof(float));
    if (!ws) scratch_failure("layernorm_backward");
    float *partial = static_cast<float *>(ws.get());
    bmb::launch(ln_bwd_dx_generic_k, dim3(ceil_div(N, NT / 64)), dim3(NT), 0, nullptr, dinp,
                dout, inp, weight, mean, rstd, N, C);
    bmb::launch(colsum_k<true>, dim3(ceil_div(C, NT), G), dim3(NT), 0, nullptr, partial, dout,
                inp, mean, rstd, N, C, rpc);
    const bmb::ColsumJob job{partial, {dweight, dbias, nullptr}, {C, C, 0}, G};
    bmb::colsum_finish_jobs(&job, 1);
}

void gelu_forward(float *out, const float *inp, int n) { run_map(GeluFwd{out, inp}, n); }

void gelu_backward(float *dinp, const float *inp, const float *dout, int n) {
    run_map(GeluBwd{dinp, inp, dout}, n);
}

void residual_forward(float *out, const float *a, const float *b, int n) {
    run_map(Residual{out, a, b}, n);
}

void add_inplace(float *dst, const float *src, int n) { run_map(AddInplace{dst, src}, n); }

void bias_forward(float *out, const float *bias, int N, int C) {
    if (N <= 0 || C <= 0) return;
    const int C4 = ceil_div(C, 4);
    const long long items = (long long)N * C4;
    if (C % 4 == 0)
        bmb::launch(bias_fwd_k<true>, dim3(grid_for(items)), dim3(NT), 0, nullptr, out, bias, C,
                    C4, items);
    else
        bmb::launch(bias_fwd_k<false>, dim3(grid_for(items)), dim3(NT), 0, nullptr, out, bias,
                    C, C4, items);
}

void bias_backward(float *dbias, const float *dout, int N, int C) {
    if (N <= 0 || C <= 0) return;
    bmb::ScratchLease ws(bmb::SCRATCH_NN, bmb::bias_partial_floats(N, C) * sizeof(float));
    if (!ws) scratch_failure("bias_backward");
    const bmb::ColsumJob job =
        bmb::bias_backward_partial(dbias, dout, N, C, static_cast<float *>(ws.get()));
    bmb::colsum_finish_jobs(&job, 1);
}

void softmax_crossentropy_forward(float *probs, float *losses, const float *logits,
                                  const int *targets, int N, int V, int Vp) {
    if (N <= 0 || V <= 0 || Vp < V) return;
    const int span = Vp % 4 == 0 ? V : V + 3;  // a ragged row's chunks start up to 3 early
    if (Vp >= 4) {
        if (span <= 1024) return xent_launch<256, 1>(probs, losses, logits, targets, N, V, Vp);
        if (span <= 4096) return xent_launch<256, 4>(probs, losses, logits, targets, N, V, Vp);
        if (span <= 16384) return xent_launch<1024, 4>(probs, losses, logits, targets, N, V, Vp);
        if (span <= 32768) return xent_launch<1024, 8>(probs, losses, logits, targets, N, V, Vp);
        if (span <= 65536) return xent_launch<1024, 16>(probs, losses, logits, targets, N, V, Vp);
    }
    rows_in_launches(N, NT, [&](int r, int n) {
        const size_t off = (size_t)r * Vp;
        bmb::launch(softmax_xent_generic_k, dim3(n), dim3(NT), 0, nullptr, probs + off, losses + r,
                    logits + off, targets + r, V, Vp);
    });
}

void crossentropy_softmax_backward(float *dlogits, const float *probs, const int *targets,
                                   int N, int V, int Vp, float dloss_scale) {
    if (N <= 0 || Vp <= 0) return;
    // A row's chunks: Vp / 4, or, starting up to 3 columns early, as many as Vp + 3 take.
    const bool rag = Vp % 4 != 0, nt = (size_t)N * Vp * sizeof(float) >= STREAM_BYTES;
    const int chunks = rag ? (int)((Vp + 6u) / 4) : Vp / 4, nb = ceil_div(chunks, NT);
    // Whole workgroups per row spare the ragged kernel the division (16384 x 5001:
    // 109 against 112 us, 2048 x 50257: 138 against 143), but idle the last one's
    // rest: 16384 x 2501 (626 of 768 lanes) still takes 51 against 54 us, x 257 (65
    // of 256) 9.5 against 6.3. Aligned rows, whose chunks cost less, are flat at
    // every width (16384 x 128: 3.3 against 5.9 us, x 12300: 254 against 280; at
    // worst 8192 x 50304: 528 against 522).
    const bool flat = !rag || (long long)chunks * 5 < 4LL * nb * NT;
    const int per = flat ? chunks : nb;
    // Rows per launch: a dispatch holds fewer than 2^32 lanes.
    const long long lanes = flat ? chunks : (long long)nb * NT;
    const int rows = (int)std::min((long long)N, ((1LL << 32) - NT) / lanes);
    for (int r = 0; r < N; r += std::min(rows, N - r)) {
        const size_t off = (size_t)r * Vp;
        const int n = std::min(rows, N - r);
        bmb::launch(rag ? flat ? xent_bwd_k<true, true> : xent_bwd_k<true, false>
                        : xent_bwd_k<false, true>,
                    dim3(grid_for(n * lanes)), dim3(NT), 0, nullptr, dlogits + off, probs + off,
                    targets + r, n, V, Vp, (unsigned)per, dloss_scale, nt);
    }
}

void adamw_update(float *params, float *grads, float *m, float *v, int n, float lr, float beta1,
                  float beta2, float eps, float weight_decay, int step, float grad_scale) {
    const float bc1 = 1.0f - powf(beta1, (float)step);
    const float bc2 = 1.0f - powf(beta2, (float)step);
    run_map(AdamW{params, grads, m, v, lr, beta1, beta2, eps, weight_decay, bc1, bc2, grad_scale},
            n);
}

float grad_global_norm(const float *grads, int n) {
    if (n <= 0) return 0.0f;
    bmb::ScratchLease ws(bmb::SCRATCH_NN, NORM_BLOCKS * sizeof(double) + 256);
    if (!ws) {
        fprintf(stderr, "bmb: grad_global_norm: cannot allocate the reduction scratch buffer\n");
        bmb::note_launch_status(hipErrorOutOfMemory);
        return NAN;
    }
    double *partial = static_cast<double *>(ws.get());
    float *out = reinterpret_cast<float *>(partial + NORM_BLOCKS);
    const int blocks = (int)std::max(1LL, std::min<long long>(NORM_BLOCKS, (n / 4 + NT - 1) / NT));
    bmb::launch(sumsq_k, dim3(blocks), dim3(NT), 0, nullptr, partial, grads, (long long)n);
    bmb::launch(finish_scalar_k<true>, dim3(1), dim3(NT), 0, nullptr, out,
                (const double *)partial, blocks, (long long)n);
    return scalar_result(out);
}

void zero_buffer(float *p, size_t n) { run_map(Zero{p}, (long long)n); }

float reduce_mean(const float *d_values, int n) {
    if (n <= 0) return NAN;
    bmb::ScratchLease ws(bmb::SCRATCH_NN, NORM_BLOCKS * sizeof(double) + 256);
    if (!ws) {
        fprintf(stderr, "bmb: reduce_mean: cannot allocate the reduction scratch buffer\n");
        bmb::note_launch_status(hipErrorOutOfMemory);
        return NAN;
    }
    double *partial = static_cast<double *>(ws.get());
    float *out = reinterpret_cast<float *>(partial + NORM_BLOCKS);
    const int blocks = (int)std::max(1LL, std::min<long long>(NORM_BLOCKS, ((long long)n + NT - 1) / NT));
    bmb::launch(sum_k, dim3(blocks), dim3(NT), 0, nullptr, partial, d_values, (long long)n);
    bmb::launch(finish_scalar_k<false>, dim3(1), dim3(NT), 0, nullptr, out,
                (const double *)partial, blocks, (long long)n);
    return scalar_result(out);
}

}  // extern "C"
