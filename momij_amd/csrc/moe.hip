// moe.hip -- RMSNorm into the qx activation format, router logits, top-k routing with
// expert bucketing, and the score-weighted expert combine.
//
// RMSNorm    maple_rms_norm (SeedlessMetal.swift:2496-2526): out = half(x * rsqrt(mean x^2 +
//            eps) * w), fp32.  Written plain (router input) and in qx order (2-bit product
//            input) with per-64-block {sum x, sum base*x}.
// Router     maple_batched_gemv (2574-2595): logits[m][e] = sum_k W[e][k] x[m][k], fp32.
// Route      maple_route_top8 (2720-2791): softmax with exp, top-k by logit (lowest index
//            on ties), scores = gate / sum of the k gates.  Then the (row, slot) pairs are
//            grouped by expert so every routed expert is streamed once for all its rows.
// Combine    maple_score_reduce / maple_score_resid (2452-2493):
//            y = [x +] half(sum_j half(down_j) * score_j), j in slot order.
#include <initializer_list>

#include "mj_device.h"
#include "mj_internal.h"
#include "moe_topk.h"

// One 256-thread block per row; H % 2048 == 0, H <= 8192.
__device__ __forceinline__ void rmsnorm_qx_row(const uint16_t* __restrict__ x,
                                               const uint16_t* __restrict__ w, float eps,
                                               uint16_t* out_plain, uint16_t* xperm,
                                               float2* xsum, int H) {
    const int row = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const uint16_t* xr = x + (size_t)row * H;
    const int nch = H / 2048;
    u4v xv[4];
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c >= nch) break;
        xv[c] = *(const u4v*)(xr + 2048 * c + 8 * t);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = h2f(xv[c][j] & 0xFFFFu), b = h2f(xv[c][j] >> 16);
            ss += a * a;
            ss += b * b;
        }
    }
    ss = wave_sum(ss);
    __shared__ float red[4];
    if (lane == 0) red[t >> 6] = ss;
    __syncthreads();
    const float tot = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = 1.0f / sqrtf(tot / (float)H + eps);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c >= nch) break;
        const int k0 = 2048 * c + 8 * t;
        const u4v wv = *(const u4v*)(w + k0);
        u4v o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = h2f(xv[c][j] & 0xFFFFu) * inv * h2f(wv[j] & 0xFFFFu);
            const float b = h2f(xv[c][j] >> 16) * inv * h2f(wv[j] >> 16);
            o[j] = (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16);
        }
        if (out_plain) *(u4v*)(out_plain + (size_t)row * H + k0) = o;
        if (xperm) emit_qx(o, lane, xperm + (size_t)row * H, xsum + (size_t)row * (H / 64), k0);
    }
}

__global__ __launch_bounds__(256) void k_rmsnorm_qx(const uint16_t* __restrict__ x,
                                                    const uint16_t* __restrict__ w, float eps,
                                                    uint16_t* out_plain, uint16_t* xperm,
                                                    float2* xsum, int H, const int* abort) {
    if (aborted(abort)) return;
    rmsnorm_qx_row(x, w, eps, out_plain, xperm, xsum, H);
}

// The front of one attention block call: the input norm of its rows, their RoPE angles, and the
// pass descriptor, which comes as a kernel argument.  One launch, with nothing to upload: two
// copies, the wait for them, the norm and the table as launches of their own took 30 us of a
// 9-row block's 56.
__global__ __launch_bounds__(256) void k_attn_front(AttnFront f, const uint16_t* __restrict__ x,
                                                    const uint16_t* __restrict__ w, float eps,
                                                    uint16_t* xperm, float2* xsum, int H,
                                                    StepDesc* sd, float2* cs, const int* abort) {
    const int r = blockIdx.x, t = threadIdx.x;
    static_assert(sizeof(StepDesc) % 8 == 0, "copied in 8-byte words");
    if (r == 0)
        for (int i = t; i < (int)(sizeof(StepDesc) / 8); i += 256)
            ((uint64_t*)sd)[i] = ((const uint64_t*)&f.sd)[i];
    if (t < f.half) {
        const float th = (float)(f.sd.L + f.sd.depth[r]) * f.inv_freq[t];
        cs[r * MJ_ROPE_F + t] = make_float2(cosf(th), sinf(th));
    }
    if (aborted(abort)) return;
    rmsnorm_qx_row(x, w, eps, nullptr, xperm, xsum, H);
}

hipError_t launch_attn_front(const AttnFront& f, const uint16_t* x, const uint16_t* w, float eps,
                             uint16_t* xperm, float2* xsum, int rows, int H, StepDesc* sd,
                             float2* cs, const int* abort, hipStream_t st) {
    if (rows < 1 || rows > MJ_ROWS || f.half > MJ_ROPE_F) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_attn_front, dim3(rows), dim3(256), 0, st, f, x, w, eps, xperm, xsum, H, sd,
                       cs, abort);
    return hipGetLastError();
}

hipError_t launch_rmsnorm_qx(const uint16_t* x, const uint16_t* w, float eps, uint16_t* out_plain,
                             uint16_t* xperm, float2* xsum, int rows, int H, const int* abort,
                             hipStream_t st) {
    hipLaunchKernelGGL(k_rmsnorm_qx, dim3(rows), dim3(256), 0, st, x, w, eps, out_plain, xperm,
                       xsum, H, abort);
    return hipGetLastError();
}

// One wave per expert: the expert's router row stays in registers, every token row is dotted
// against it.  H % 512 == 0, H <= 4096.
__global__ __launch_bounds__(256) void k_router(const uint16_t* __restrict__ W,
                                                const uint16_t* __restrict__ x, float* logits,
                                                int M, int E, int H, const int* abort) {
    if (aborted(abort)) return;
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= E) return;
    const int nch = H / 512;
    u4v wr[8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
        if (c < nch) wr[c] = *(const u4v*)(W + (size_t)e * H + 512 * c + 8 * lane);
    for (int m = 0; m < M; ++m) {
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (c >= nch) break;
            const u4v xv = *(const u4v*)(x + (size_t)m * H + 512 * c + 8 * lane);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = dot2(wr[c][j], xv[j], acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) logits[(size_t)m * E + e] = acc;
    }
}

hipError_t launch_router(const uint16_t* W, const uint16_t* x, float* logits, int M, int E, int H,
                         const int* abort, hipStream_t st) {
    hipLaunchKernelGGL(k_router, dim3((E + 3) / 4), dim3(256), 0, st, W, x, logits, M, E, H,
                       abort);
    return hipGetLastError();
}

// Group pair indices 0..P-1 by expert id (ids in s_ids, LDS): experts in increasing id, an
// expert's pairs in no particular order (each pair's output is computed the same way wherever it
// is listed).  Ids outside [0, E) are left out.  Whole 256-thread block, thread t = expert t
// (one thread walking the experts and pairs took 21 us of a 72-pair product's 48).
__device__ void bucket_pairs(const int* s_ids, int P, int E, Buckets* bk, int* s_cnt,
                             int* s_slot) {
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    __shared__ int s_tot[4][2];
    s_cnt[t] = 0;
    __syncthreads();
    for (int p = t; p < P; p += 256) {
        const int e = s_ids[p];
        if (e >= 0 && e < E) atomicAdd(&s_cnt[e], 1);
    }
    __syncthreads();
    const int cnt = s_cnt[t], on = cnt > 0;
    int pos = cnt, u = on;  // inclusive sums over the experts up to t
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(pos, o, MJ_WAVE), z = __shfl_up(u, o, MJ_WAVE);
        if (lane >= o) {
            pos += y;
            u += z;
        }
    }
    if (lane == 63) {
        s_tot[wv][0] = pos;
        s_tot[wv][1] = u;
    }
    __syncthreads();
    for (int w = 0; w < wv; ++w) {
        pos += s_tot[w][0];
        u += s_tot[w][1];
    }
    s_slot[t] = pos - cnt;
    if (on) {
        bk->expert[u - 1] = t;
        bk->start[u - 1] = pos - cnt;
    }
    if (t == 255) {
        bk->start[u] = pos;
        bk->count = u;
    }
    __syncthreads();
    for (int p = t; p < P; p += 256) {
        const int e = s_ids[p];
        if (e >= 0 && e < E) bk->pair[atomicAdd(&s_slot[e], 1)] = p;
    }
}
static_assert(MJ_MAX_EXPERTS == 256, "an expert a thread");

__global__ __launch_bounds__(256) void k_bucket_inds(const int32_t* __restrict__ inds, int P,
                                                     Buckets* bk, const int* abort) {
    if (block_aborted(abort)) return;
    __shared__ int s_ids[MJ_MAX_PAIRS];
    __shared__ int s_cnt[MJ_MAX_EXPERTS];
    __shared__ int s_slot[MJ_MAX_EXPERTS];
    for (int p = threadIdx.x; p < P; p += blockDim.x) s_ids[p] = inds[p];
    __syncthreads();
    bucket_pairs(s_ids, P, MJ_MAX_EXPERTS, bk, s_cnt, s_slot);
}

hipError_t launch_bucket_inds(const int32_t* inds, int P, Buckets* bk, const int* abort,
                              hipStream_t st) {
    hipLaunchKernelGGL(k_bucket_inds, dim3(1), dim3(256), 0, st, inds, P, bk, abort);
    return hipGetLastError();
}

// Single block: softmax + top-k per row (one wave per row), then expert bucketing.
__global__ __launch_bounds__(256) void k_topk_bucket(const float* __restrict__ logits, int M,
                                                     int E, int k, int32_t* inds, float* scores,
                                                     Buckets* bk, const int* abort) {
    if (block_aborted(abort)) return;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    __shared__ int s_inds[MJ_MAX_PAIRS];
    __shared__ int s_cnt[MJ_MAX_EXPERTS];
    __shared__ int s_slot[MJ_MAX_EXPERTS];
    for (int m = wv; m < M; m += 4) {
        const float* lg = logits + (size_t)m * E;
        float lv[4], work[4];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = lane + 64 * i;
            lv[i] = e < E ? lg[e] : -INFINITY;
            mx = fmaxf(mx, lv[i]);
        }
        mx = wave_max(mx);
        float z = 0.0f, g[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = lane + 64 * i;
            g[i] = e < E ? expf(lv[i] - mx) : 0.0f;
            z += g[i];
            work[i] = lv[i];
        }
        z = wave_sum(z);
        float sel[8];
        int seli[8];
        for (int j = 0; j < k; ++j) {
            float bv = work[0];
            int bi = lane;
#pragma unroll
            for (int i = 1; i < 4; ++i)
                if (work[i] > bv) {
                    bv = work[i];
                    bi = lane + 64 * i;
                }
            wave_argmax(bv, bi);
            // owner lane marks it taken and publishes the gate
            float gsel = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (lane + 64 * i == bi) {
                    work[i] = -INFINITY;
                    gsel = g[i] / z;
                }
            gsel = __shfl(gsel, bi & 63, MJ_WAVE);
            sel[j] = gsel;
            seli[j] = bi;
        }
        if (lane == 0) {
            float ssum = 0.0f;
            for (int j = 0; j < k; ++j) ssum += sel[j];
            for (int j = 0; j < k; ++j) {
                inds[m * k + j] = seli[j];
                scores[m * k + j] = sel[j] / ssum;
                s_inds[m * k + j] = seli[j];
            }
        }
    }
    if (bk == nullptr) return;
    __syncthreads();
    bucket_pairs(s_inds, M * k, E, bk, s_cnt, s_slot);
}

hipError_t launch_topk_bucket(const float* logits, int M, int E, int k, int32_t* inds,
                              float* scores, Buckets* bk, const int* abort, hipStream_t st) {
    hipLaunchKernelGGL(k_topk_bucket, dim3(1), dim3(256), 0, st, logits, M, E, k, inds, scores,
                       bk, abort);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_score_combine(const uint16_t* __restrict__ down,
                                                       const float* __restrict__ scores,
                                                       const uint16_t* x_resid, uint16_t* y,
                                                       int M, int k, int H, const int* abort) {
    if (aborted(abort)) return;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= M * H) return;
    const int m = i / H, c = i % H;
    float acc = 0.0f;
    for (int j = 0; j < k; ++j) acc += h2f(down[((size_t)m * k + j) * H + c]) * scores[m * k + j];
    if (x_resid)
        y[i] = f2h(h2f(x_resid[i]) + hround(acc));
    else
        y[i] = f2h(acc);
}

// The same combine, 8 elements a thread (H % 8 == 0, k <= 8) with every load issued before
// the first wait: one memory round trip instead of one per expert.
__global__ __launch_bounds__(256) void k_score_combine8(const uint16_t* __restrict__ down,
                                                        const float* __restrict__ scores,
                                                        const uint16_t* x_resid, uint16_t* y,
                                                        int M, int k, int H, const int* abort) {
    const int i = 8 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= M * H) return;
    const int m = i / H, c = i % H;
    u4v d[8];
    float sc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int jj = min(j, k - 1);
        d[j] = *(const u4v*)(down + ((size_t)m * k + jj) * H + c);
        sc[j] = scores[m * k + jj];
    }
    const u4v xr = *(const u4v*)((x_resid ? x_resid : down) + (size_t)i);
    if (aborted(abort)) return;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (j < k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc[2 * q] += h2f(d[j][q] & 0xFFFFu) * sc[j];
                acc[2 * q + 1] += h2f(d[j][q] >> 16) * sc[j];
            }
        }
    }
    u4v o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (x_resid)
            o[q] = (uint32_t)f2h(h2f(xr[q] & 0xFFFFu) + hround(acc[2 * q])) |
                   ((uint32_t)f2h(h2f(xr[q] >> 16) + hround(acc[2 * q + 1])) << 16);
        else
            o[q] = (uint32_t)f2h(acc[2 * q]) | ((uint32_t)f2h(acc[2 * q + 1]) << 16);
    }
    *(u4v*)(y + (size_t)i) = o;
}

hipError_t launch_score_combine(const uint16_t* down, const float* scores, const uint16_t* x_resid,
                                uint16_t* y, int M, int k, int H, const int* abort,
                                hipStream_t st) {
    if (H % 8 == 0 && k >= 1 && k <= 8) {
        hipLaunchKernelGGL(k_score_combine8, dim3((M * H / 8 + 255) / 256), dim3(256), 0, st, down,
                           scores, x_resid, y, M, k, H, abort);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_score_combine, dim3((M * H + 255) / 256), dim3(256), 0, st, down, scores,
                       x_resid, y, M, k, H, abort);
    return hipGetLastError();
}

// The expert combine of one row followed by the next RMSNorm (of the next layer's attention,
// or the final norm), H = 2048: one 256-thread block per row, thread t owns elements
// 8t .. 8t+7.  The combine is k_score_combine's arithmetic, the norm k_rmsnorm_qx's.  Every
// load is issued before the first wait (the k <= 8 expert rows at clamped indices, their
// weights, the residual, the norm weights and the abort word): one memory round trip, not one
// per expert.
__global__ __launch_bounds__(256) void k_combine_norm(const uint16_t* __restrict__ down,
                                                      const float* __restrict__ scores,
                                                      const uint16_t* x_resid, uint16_t* y, int k,
                                                      NormOut no, const int* abort) {
    const int r = blockIdx.x, t = threadIdx.x;
    constexpr int H = 2048;
    u4v d[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
        d[j] = *(const u4v*)(down + ((size_t)r * k + min(j, k - 1)) * H + 8 * t);
    // the weights as one vector load (lane j holds weight j), not eight scalar ones
    const float scv = scores[r * k + min(t & 7, k - 1)];
    const u4v xr = *(const u4v*)((x_resid ? x_resid : down) + (size_t)r * H + 8 * t);
    const u4v wn = *(const u4v*)(no.w + 8 * t);
    if (aborted(abort)) return;
    float sc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) sc[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(scv), j));
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (j < k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc[2 * q] += h2f(d[j][q] & 0xFFFFu) * sc[j];
                acc[2 * q + 1] += h2f(d[j][q] >> 16) * sc[j];
            }
        }
    }
    u4v hv;
    if (x_resid) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            hv[q] = (uint32_t)f2h(h2f(xr[q] & 0xFFFFu) + hround(acc[2 * q])) |
                    ((uint32_t)f2h(h2f(xr[q] >> 16) + hround(acc[2 * q + 1])) << 16);
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            hv[q] = (uint32_t)f2h(acc[2 * q]) | ((uint32_t)f2h(acc[2 * q + 1]) << 16);
    }
    *(u4v*)(y + (size_t)r * H + 8 * t) = hv;
    norm_row_2048_w(hv, wn, no, r);
}

hipError_t launch_combine_norm(const uint16_t* down, const float* scores, const uint16_t* x_resid,
                               uint16_t* y, int M, int k, int H, const NormOut& no,
                               const int* abort, hipStream_t st) {
    if (H != 2048 || k < 1 || k > 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_combine_norm, dim3(M), dim3(256), 0, st, down, scores, x_resid, y, k, no,
                       abort);
    return hipGetLastError();
}

#define RT_H 2048

// ---------------------------------------------------------------------------------------
// MoE front, two launches:
//   k_route_logits  one 256-thread block per (row, group of RS_EPB experts), M * E / RS_EPB
//                   blocks: RMSNorm of the row (the group-0 block writes it out, plain and in
//                   qx order with its block sums) and the logits of the group's experts.  The
//                   router matrix is read in 32 KB pieces by many CUs (a single CU streams only
//                   a few tens of GB/s).
//   k_route_topk    one wave per row: top-k of the row's logits, renormalised scores.
// The kernel boundary orders the two: a grid-wide hand-off inside one kernel costs more than the
// launch with a device-scope release (an L2 write-back on this chip: 7.8 us at 72 blocks, two
// launches 3.5), and about as much without one (device-coherent stores and one counter: 2.5 us at 144
// blocks, 3.9 at 256; an empty launch 2.45).
// Arithmetic as maple_rms_norm / maple_batched_gemv / maple_route_top8: fp32 sums (the logit
// sums in v_dot2 lane partials and a fixed shuffle tree), softmax with max subtraction, top-k
// by logit with the lowest index winning ties, weights renormalised over the k in rank order.
// The top-k ranks every expert against all E logits (broadcast LDS reads), so the selection
// comes out sorted without a chain of cross-lane reductions.
// ---------------------------------------------------------------------------------------
#define RS_EPB 8  // router rows (experts) per block: two per wave

__global__ __launch_bounds__(256) void k_route_logits(RouteArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int E = a.E, S = E / RS_EPB;
    const int r = blockIdx.x / S, grp = blockIdx.x - r * S;
    __shared__ __align__(16) uint16_t xn[RT_H];
    __shared__ float s_ss[4];
    if (aborted(a.abort)) return;

    // router rows of this wave first (k = 512 c + 8 lane .. +7), then the row
    const int e0 = grp * RS_EPB + 2 * wv;
    u4v wr[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            wr[j][c] = *(const u4v*)(a.W + (size_t)(e0 + j) * RT_H + 512 * c + 8 * lane);
    u4v xv = *(const u4v*)(a.x + (size_t)r * RT_H + 8 * tid);
    u4v nw = {0u, 0u, 0u, 0u};
    if (a.norm_w) nw = *(const u4v*)(a.norm_w + 8 * tid);

    if (a.norm_w) {
        float ss = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float x0 = h2f(xv[q] & 0xFFFFu), x1 = h2f(xv[q] >> 16);
            ss += x0 * x0;
            ss += x1 * x1;
        }
        ss = wave_sum(ss);
        if (lane == 0) s_ss[wv] = ss;
        __syncthreads();
        const float tot = (s_ss[0] + s_ss[1]) + (s_ss[2] + s_ss[3]);
        const float inv = 1.0f / sqrtf(tot / (float)RT_H + a.eps);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float x0 = h2f(xv[q] & 0xFFFFu) * inv * h2f(nw[q] & 0xFFFFu);
            const float x1 = h2f(xv[q] >> 16) * inv * h2f(nw[q] >> 16);
            xv[q] = (uint32_t)f2h(x0) | ((uint32_t)f2h(x1) << 16);
        }
    }
    *(u4v*)(xn + 8 * tid) = xv;
    // the fused MoE launch's act rows: the "not yet written" marker, before that launch starts
    for (int i = blockIdx.x * 256 + tid; i < a.act_n16; i += gridDim.x * 256)
        ((u4v*)a.act_mark)[i] = (u4v){~0u, ~0u, ~0u, ~0u};
    if (grp == 0) {
        if (a.xn) *(u4v*)(a.xn + (size_t)r * RT_H + 8 * tid) = xv;
        if (a.xperm)
            emit_qx(xv, lane, a.xperm + (size_t)r * RT_H, a.xsum + (size_t)r * (RT_H / 64), 8 * tid);
    }
    __syncthreads();

    u4v xa[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) xa[c] = *(const u4v*)(xn + 512 * c + 8 * lane);
    float acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        acc[j] = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[j] = dot2(wr[j][c][q], xa[c][q], acc[j]);
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] += __shfl_xor(acc[j], m, MJ_WAVE);
    if (lane == 0) *(float2*)(a.logits + (size_t)r * E + e0) = make_float2(acc[0], acc[1]);
}

// The logits of a wide pass, from rows already normed: a wave keeps four experts' router rows in
// registers over RW_ROWS rows, two at a time.  Its eight sums meet by halves: at each of the first
// three lane distances a lane keeps half of its sums and takes the other lane's part of them, so the
// additions are those of k_route_logits' tree with 10 lane moves for eight sums instead of 48.
// Norming again in each of 32 blocks a row, with an LDS copy of it, took 17 us for 200 rows of 256
// experts; the norm launch and this one 14.4.
#define RW_ROWS 8
__global__ __launch_bounds__(256) void k_route_wide(RouteArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int E = a.E, G = (E + 15) / 16;
    const int r0 = blockIdx.x / G * RW_ROWS, e0 = blockIdx.x % G * 16 + 4 * wv;
    if (aborted(a.abort) || e0 >= E) return;
    u4v wr[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            wr[j][c] = *(const u4v*)(a.W + (size_t)min(e0 + j, E - 1) * RT_H + 512 * c + 8 * lane);
    u4v xa[2][2][4];
    auto request = [&](int r, u4v (&x)[2][4]) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                x[i][c] = *(const u4v*)(a.x + (size_t)min(r + i, a.M - 1) * RT_H + 512 * c + 8 * lane);
    };
    request(r0, xa[0]);
#pragma unroll
    for (int it = 0; it < RW_ROWS / 2; ++it) {
        const int r = r0 + 2 * it;
        if (r >= a.M) break;
        if (it + 1 < RW_ROWS / 2) request(r + 2, xa[(it + 1) & 1]);
        float v[8];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float acc = 0.0f;
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc = dot2(wr[j][c][q], xa[it & 1][i][c][q], acc);
                v[4 * i + j] = acc;
            }
#pragma unroll
        for (int m = 32, n = 4; m > 4; m >>= 1, n >>= 1) {
            const bool up = (lane & m) != 0;
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const float keep = up ? v[i + n] : v[i], send = up ? v[i] : v[i + n];
                v[i] = keep + __shfl_xor(send, m, MJ_WAVE);
            }
        }
#pragma unroll
        for (int m = 4; m > 0; m >>= 1) v[0] += __shfl_xor(v[0], m, MJ_WAVE);
        // lane 8 s: sum s = 4 i + j (bit 5 of the lane chose i, bits 4 and 3 j)
        const int row = r + (lane >> 5), e = e0 + ((lane >> 3) & 3);
        if ((lane & 7) == 0 && row < a.M && e < E) a.logits[(size_t)row * E + e] = v[0];
    }
}

// inds and scores of every row: one wave a row, four rows a block.  (One 16-wave block for the
// whole pass ranked up to four rows a wave on one CU: 22.7 us for 64 rows of 256 experts, 10.0 us
// of 64.)
#define RT_WAVES 4
template <int NI>
__global__ __launch_bounds__(64 * RT_WAVES) void k_route_topk(RouteArgs a) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, E = a.E, k = a.k;
    __shared__ __align__(16) float s_row[RT_WAVES][64 * NI];
    __shared__ __align__(16) float s_gate[RT_WAVES][8];
    __shared__ int s_ind[RT_WAVES][8];
    const int r = blockIdx.x * RT_WAVES + wv;
    float v[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
        v[i] = a.logits[min(r, a.M - 1) * E + min(lane + 64 * i, E - 1)];
    if (aborted(a.abort) || r >= a.M) return;
#pragma unroll
    for (int i = 0; i < NI; ++i)
        s_row[wv][lane + 64 * i] = lane + 64 * i < E ? v[i] + 0.0f : -INFINITY;
    __builtin_amdgcn_wave_barrier();
    int e = 0;
    float gate = 0.0f;
    row_topk<NI>(s_row[wv], E, k, s_ind[wv], s_gate[wv], e, gate);
    if (lane < k) {
        a.inds[r * k + lane] = e;
        a.scores[r * k + lane] = gate;
    }
}

bool route_supported(int H, int E, int k) {
    return H == RT_H && E >= RS_EPB && E <= MJ_MAX_EXPERTS && E % RS_EPB == 0 && k >= 1 &&
           k <= 8 && k <= E;
}

hipError_t launch_route_logits(const RouteArgs& a, int H, hipStream_t st) {
    if (!route_supported(H, a.E, a.k) || a.M < 1 || a.M > MJ_WIDE_ROWS) return hipErrorInvalidValue;
    if (!a.logits) return hipErrorInvalidValue;
    if (a.M <= MJ_ROWS) {
        hipLaunchKernelGGL(k_route_logits, dim3(a.M * (a.E / RS_EPB)), dim3(256), 0, st, a);
        return hipGetLastError();
    }
    // a wide pass: the rows normed by a launch of their own (into xn, and in qx order)
    if (!a.norm_w || !a.xn || !a.xperm || a.act_n16 != 0) return hipErrorInvalidValue;
    hipError_t e = launch_rmsnorm_qx(a.x, a.norm_w, a.eps, a.xn, a.xperm, a.xsum, a.M, H, a.abort, st);
    if (e != hipSuccess) return e;
    RouteArgs w = a;
    w.x = a.xn;
    hipLaunchKernelGGL(k_route_wide,
                       dim3((a.M + RW_ROWS - 1) / RW_ROWS * ((a.E + 15) / 16)), dim3(256), 0, st, w);
    return hipGetLastError();
}

hipError_t launch_route_topk(const RouteArgs& a, hipStream_t st) {
    if (a.E < 1 || a.E > MJ_MAX_EXPERTS || a.k < 1 || a.k > 8 || a.k > a.E || a.M < 1 ||
        a.M > MJ_WIDE_ROWS)
        return hipErrorInvalidValue;
    const dim3 grid((a.M + RT_WAVES - 1) / RT_WAVES), block(64 * RT_WAVES);
    if (a.E <= 64)
        hipLaunchKernelGGL(k_route_topk<1>, grid, block, 0, st, a);
    else
        hipLaunchKernelGGL(k_route_topk<MJ_MAX_EXPERTS / 64>, grid, block, 0, st, a);
    return hipGetLastError();
}

// The slot tables of a wide pass's two expert products, from its pairs' expert ids: one block,
// thread t < 256 numbering expert t's slots by sums across the experts, then a pair a thread
// taking the next place of its expert (a pair whose id is outside [0, E) has none).  The places' order varies from run to run, which moves rows
// within a slot and changes no value.
__global__ __launch_bounds__(1024) void k_wide_slots(const int32_t* __restrict__ inds, int P,
                                                     int E, SlotTab up, SlotTab dn,
                                                     const int* abort) {
    __shared__ int s_cnt[MJ_MAX_EXPERTS], s_at[MJ_MAX_EXPERTS], s_first[2][MJ_MAX_EXPERTS];
    __shared__ int s_tot[2][4];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    constexpr int PT = MJ_WIDE_PAIRS / 1024;
    int id[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) id[i] = t + 1024 * i < P ? inds[t + 1024 * i] : -1;
    if (block_aborted(abort)) return;
    if (t < MJ_MAX_EXPERTS) s_cnt[t] = s_at[t] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i)
        if ((unsigned)id[i] < (unsigned)E) atomicAdd(&s_cnt[id[i]], 1);
    __syncthreads();
    int incl[2] = {0, 0}, parts[2] = {0, 0};
    if (t < MJ_MAX_EXPERTS) {
        const int c = s_cnt[t];
        parts[0] = (c + up.ps - 1) / up.ps;
        parts[1] = (c + dn.ps - 1) / dn.ps;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            incl[x] = parts[x];
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl[x], o, MJ_WAVE);
                if (lane >= o) incl[x] += y;
            }
            if (lane == 63) s_tot[x][wv] = incl[x];
        }
    }
    __syncthreads();
    if (t < MJ_MAX_EXPERTS) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            for (int w = 0; w < wv; ++w) incl[x] += s_tot[x][w];
            s_first[x][t] = incl[x] - parts[x];
        }
    }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const SlotTab& tab = x ? dn : up;
        const int n = ((s_tot[x][0] + s_tot[x][1]) + s_tot[x][2]) + s_tot[x][3];
        for (int sl = n + t; sl < tab.n; sl += 1024) *(int2*)(tab.rec + 16 * sl) = make_int2(0, 0);
    }
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int e = id[i], p = t + 1024 * i;
        if ((unsigned)e >= (unsigned)E) continue;
        const int c = s_cnt[e], at = atomicAdd(&s_at[e], 1);
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            // the first `more` slots take one pair more than the others
            const SlotTab& tab = x ? dn : up;
            const int np = (c + tab.ps - 1) / tab.ps, base = c / np, more = c - base * np;
            const int lead = more * (base + 1);
            const int sl = at < lead ? at / (base + 1) : more + (at - lead) / base;
            const int off = at < lead ? at - sl * (base + 1) : (at - lead) - (sl - more) * base;
            const int cnt = base + (sl < more ? 1 : 0);
            int32_t* rec = tab.rec + 16 * (s_first[x][e] + sl);
            rec[off] = p | (off == 0 ? e << 16 : off == 1 ? cnt << 16 : 0);
            if (cnt == 1) rec[1] = 1 << 16;
        }
    }
}

hipError_t launch_wide_slots(const int32_t* inds, int P, int E, const SlotTab& up,
                             const SlotTab& dn, const int* abort, hipStream_t st) {
    for (const SlotTab* tab : {&up, &dn})
        if (tab->ps < 1 || tab->ps > 16 || tab->n < slot_tab_size(MJ_MAX_EXPERTS, tab->ps))
            return hipErrorInvalidValue;
    if (P < 1 || P > MJ_WIDE_PAIRS || E < 1 || E > MJ_MAX_EXPERTS) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_wide_slots, dim3(1), dim3(1024), 0, st, inds, P, E, up, dn, abort);
    return hipGetLastError();
}
