// sample.hip -- full-vocabulary speculative sampling (rejection sampling) on the device.
//
// Rules: SpeculativeSampling.tryAccept / walkDraft (SpeculativeSampling.swift:27-99) with
// LogitsProcessor.probabilities / samplePrepared (LogitsProcessor.swift:116-189):
//   p = softmax(logits * (1/T));  accept draft d iff q > 0, p_d > 0 and u0 <= min(1, p_d / q);
//   on reject sample the residual (point q: p with p_d -> max(0, p_d - q); uniform q:
//   max(p - q, 0)) by a cumulative walk to u1 * sum; after a full accept sample the bonus from
//   the last row by a walk to u0 * sum of exps.
// LogitsProcessor options: penalties (prepare, LogitsProcessor.swift:57-104) on every row, the
// seen set and counts growing with the drafts accepted before it (walkDraft 86-87);
// samplePrepared's nucleus (137-154) for the bonus and for a residual of zero mass: tokens
// ranked by e descending, the lower id first on ties, kept up to the first ranked prefix whose
// mass reaches top_p * Z, sampled in id order.  The masses are summed exactly, as integers
// trunc(e * 2^40), so no order is needed: the cut is found by a radix selection over the e bits
// (three digit rounds of histograms of counts and masses), not by sorting the row.
// Every float operation below happens in a fixed order (chunks of 16 summed sequentially,
// blocks of 64 chunks summed sequentially, block totals summed sequentially; exp evaluated by
// canon_expf; IEEE divisions) so the CPU oracle reproduces each decision bit for bit.
#pragma clang fp contract(off)
#include "mj_device.h"
#include "mj_internal.h"

#define CH 16
#define BLK 64
#define MAX_CHUNKS 12288  // V <= 196608
#define RMB 32            // blocks a row's maximum is split over
#define DEC_STAGE (MJ_ROWS * (MAX_CHUNKS / BLK))  // every row's block sums, in LDS

// Hand-off from the accept decisions to the residual walk: phase 1 = row fr was rejected and
// its residual still has to be summed (k_resid_sums) and walked (k_resid_walk).
struct SampleState {
    int phase, fr, d, pad;
    float q, Zr, pad2, pad3;
};
static_assert(sizeof(SampleState) == 32, "state fits its 8 floats");

struct SampleArgs {
    const float* src;      // [rows][V] the logits given
    float* logits;         // [rows][V] the logits sampled from: src, or where its rows go penalised
    int rows, V;
    const int32_t* draft;  // [rows-1]
    float invT;
    int q_mode;            // 0 point, 1 uniform
    float q_uniform;       // 1/V
    const float* q_point;  // [rows-1] or nullptr (= 1)
    uint64_t seed, counter;
    float* rowmax;         // [rows]
    float* bsum;           // [rows][nblocks] block sums of e
    int nblocks;
    float* mpart;          // [rows][RMB] partial row maxima
    const float* head_max; // [rows] row maxima already known (no penalties), or nullptr
    float* rbs;            // [nblocks] block sums of the residual of the rejected row
    struct SampleState* state;
    int32_t* out;          // [2] or nullptr
    StepResult* res;       // or nullptr
    const StepDesc* sd;    // when set: temperature, q, seed, counter, draft, options from it
    const int* abort;
    SampleOpts o;
    NucleusBuf nb;         // nb.st == nullptr: no nucleus
};

// Effective per-call parameters (from the step descriptor when one is given).
__device__ __forceinline__ SampleArgs resolve(SampleArgs a) {
    if (a.sd) {
        a.invT = __fdiv_rn(1.0f, fmaxf(a.sd->temperature, 1e-5f));
        a.q_mode = a.sd->q_mode;
        a.q_uniform = a.sd->q_uniform;
        a.q_point = a.sd->has_qpoint ? a.sd->q_point : nullptr;
        a.seed = a.sd->seed;
        a.counter = a.sd->counter;
        a.draft = a.sd->tokens + 1;
        a.o.top_p = a.sd->top_p;
        a.o.rep = a.sd->rep;
        a.o.pres = a.sd->pres;
        a.o.freq = a.sd->freq;
        a.o.n_hist = a.sd->n_hist;
    }
    return a;
}

__device__ __forceinline__ bool nucleus_on(const SampleArgs& a) {
    return a.nb.st != nullptr && a.o.top_p < 1.0f - 1e-6f;
}

// LogitsProcessor.prepare for one token: repetition, presence, frequency (in that order)
__device__ __forceinline__ float penalize1(float x, int count, float rep, float pres, float freq) {
    if (fabsf(rep - 1.0f) > 1e-6f && rep > 0.0f) x = x > 0.0f ? __fdiv_rn(x, rep) : x * rep;
    if (pres != 0.0f) x = x - pres;
    if (freq != 0.0f && count > 0) x = x - freq * (float)count;
    return x;
}

__device__ __forceinline__ void row_uniforms(const SampleArgs& a, int row, float& u0, float& u1) {
    uint32_t c[4] = {(uint32_t)row, (uint32_t)a.counter, (uint32_t)(a.counter >> 32), 0x6d6a6a76u};
    philox4x32_10(c, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
    u0 = u01(c[0]);
    u1 = u01(c[1]);
}

__device__ __forceinline__ float e_of(const SampleArgs& a, float x, float mxs) {
    const float s = x * a.invT;
    return canon_expf(s - mxs);
}

__device__ __forceinline__ float e_at(const SampleArgs& a, int row, int v, float mxs) {
    return e_of(a, a.logits[(size_t)row * a.V + v], mxs);
}

// residual mass at v given e_v (p_v = e_v / Z)
__device__ __forceinline__ float r_of(const SampleArgs& a, float e, int v, float Z, float q,
                                      int d) {
    const float pv = __fdiv_rn(e, Z);
    if (a.q_mode == 1) return fmaxf(pv - q, 0.0f);
    if (v == d && q > 0.0f) return fmaxf(0.0f, pv - q);
    return pv;
}

// Rows of 16-byte aligned logits (float4 requests) or not (one float a request).
__device__ __forceinline__ bool rows_aligned(const SampleArgs& a) {
    return ((a.V & 3) | ((uintptr_t)a.logits & 15)) == 0;
}

// The CH logits of chunk c of a row, requested together; indices past the row's end clamp to
// its last element (callers use only those below V).
__device__ __forceinline__ void chunk_logits(const SampleArgs& a, int row, int c, float x[CH]) {
    const float* rp = a.logits + (size_t)row * a.V;
    if (rows_aligned(a)) {
        const float4* p4 = (const float4*)rp;
        const int last = (a.V >> 2) - 1;
#pragma unroll
        for (int k = 0; k < CH / 4; ++k) {
            const float4 f = p4[min(c * (CH / 4) + k, last)];
            x[4 * k] = f.x;
            x[4 * k + 1] = f.y;
            x[4 * k + 2] = f.z;
            x[4 * k + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < CH; ++k) x[k] = rp[min(c * CH + k, a.V - 1)];
    }
}

// Chunk c's element values -- e, or the residual (resid) -- into x, and their sum in element
// order.
__device__ __forceinline__ float chunk_vals(const SampleArgs& a, int row, int c, bool resid,
                                            float mxs, float Z, float q, int d, float x[CH]) {
    chunk_logits(a, row, c, x);
    const int v0 = c * CH;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        float e = e_of(a, x[k], mxs);
        if (resid) e = r_of(a, e, v0 + k, Z, q, d);
        x[k] = e;
        if (v0 + k < a.V) s = s + e;
    }
    return s;
}

// n >= 1 floats from src into LDS by nt threads, eight requests a thread in flight.
__device__ __forceinline__ void stage_lds(float* dst, const float* src, int n, int t, int nt) {
    for (int base = t; base < n; base += nt * 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = src[min(base + nt * k, n - 1)];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (base + nt * k < n) dst[base + nt * k] = v[k];
    }
}

// One thread: p[0..n) (n >= 1) replaced by its running totals in order, p[b] = ((p_0 + p_1) +
// ...) + p_b from 0.0f; returns the total.
__device__ __forceinline__ float running_totals(float* p, int n) {
    float z = 0.0f;
    for (int b0 = 0; b0 < n; b0 += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = p[min(b0 + k, n - 1)];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (b0 + k < n) {
                z = z + v[k];
                p[b0 + k] = z;
            }
    }
    return z;
}

// First lane of the (whole, converged) wave whose `hit` holds, or -1.
__device__ __forceinline__ int wave_first(bool hit) {
    const uint64_t m = __ballot(hit);
    return m ? __ffsll((unsigned long long)m) - 1 : -1;
}

#define RM_UNROLL 6  // float4 requests a thread: a slice of V / RMB <= 6144 floats in one round

// Without penalties: the slices' maxima alone, each thread its whole share of a slice at once
// (indices clamp to the slice's last element, and a repeated one leaves a maximum unchanged).  Through
// k_row_prep's copy in LDS, which bounds the blocks of a CU to six, 64 rows of 151936 were accepted in
// 53.8 us and 9 in 28.4; 38.2 and 23.9 so.
__global__ __launch_bounds__(256) void k_row_max(SampleArgs a) {
    if (aborted(a.abort)) return;
    const int i = blockIdx.x / RMB, j = blockIdx.x % RMB, t = threadIdx.x;
    const float* rp = a.logits + (size_t)i * a.V;
    float m = -INFINITY;
    if (rows_aligned(a)) {
        const int V4 = a.V >> 2, span = (V4 + RMB - 1) / RMB;
        const int v0 = j * span, v1 = min(V4, v0 + span);
        for (int v = v0 + t; v < v1; v += 256 * RM_UNROLL) {
            float4 f[RM_UNROLL];
#pragma unroll
            for (int k = 0; k < RM_UNROLL; ++k)
                f[k] = *(const float4*)(rp + 4 * min(v + 256 * k, v1 - 1));
#pragma unroll
            for (int k = 0; k < RM_UNROLL; ++k)
                m = fmaxf(m, fmaxf(fmaxf(f[k].x, f[k].y), fmaxf(f[k].z, f[k].w)));
        }
    } else {
        const int span = (a.V + RMB - 1) / RMB;
        const int v0 = j * span, v1 = min(a.V, v0 + span);
        for (int v = v0 + t; v < v1; v += 256 * 8) {
            float f[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) f[k] = rp[min(v + 256 * k, v1 - 1)];
#pragma unroll
            for (int k = 0; k < 8; ++k) m = fmaxf(m, f[k]);
        }
    }
    m = wave_max(m);
    __shared__ float sm[4];
    if ((t & 63) == 0) sm[t >> 6] = m;
    __syncthreads();
    if (t == 0) a.mpart[i * RMB + j] = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
}

// The rows made ready, in RMB slices a row: block (row i, j) takes its slice of the given logits
// (src) into LDS, applies row i's penalties to the slice's tokens, writes the slice to `logits` (the
// same buffer, or the copy that keeps the caller's), and the slice's maximum (exact in any order;
// the sums kernel folds the RMB partials).  The penalties: every history token, then every draft
// d < i that is neither earlier among the drafts nor in the history, each once with its total count
// (history count + occurrences among drafts 0 .. i-1).  The history is ascending: a longer one is
// searched for the slice's part by 256 samples of it.  Slice, history and drafts are requested
// together.  (A copy, one block a row for the penalties, then the maxima: acceptance of 9 rows of
// 151936 with a history of 1500 79.2 us, now 69.7.)
#define RP_HIST 8    // history entries a thread requests at once
#define RP_SLICE (MAX_CHUNKS * CH / RMB)
__global__ __launch_bounds__(256) void k_row_prep(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    const bool rep_on = fabsf(a.o.rep - 1.0f) > 1e-6f && a.o.rep > 0.0f;
    const bool pen = rep_on || a.o.pres != 0.0f || a.o.freq != 0.0f;
    const int i = blockIdx.x / RMB, j = blockIdx.x % RMB, t = threadIdx.x;
    const float* src = a.src + (size_t)i * a.V;
    float* dst = a.logits + (size_t)i * a.V;
    const bool al = ((a.V & 3) | (((uintptr_t)a.src | (uintptr_t)a.logits) & 15)) == 0;
    const int span = al ? ((a.V >> 2) + RMB - 1) / RMB * 4 : (a.V + RMB - 1) / RMB;
    const int v0 = min(j * span, a.V), v1 = min(v0 + span, a.V), n = v1 - v0;
    __shared__ __align__(16) float s_l[RP_SLICE];
    __shared__ int s_draft[MJ_ROWS];
    __shared__ int s_inh[MJ_ROWS];  // draft d equals a history token of the slice
    static_assert(RM_UNROLL * 4 * 256 >= RP_SLICE, "a slice in one round");
    // (an empty slice still requests element 0 of its row)
    const int last = max(n, 1) - 1, vb = n > 0 ? v0 : 0;
    float4 f[RM_UNROLL];
    if (al) {
#pragma unroll
        for (int k = 0; k < RM_UNROLL; ++k)
            f[k] = *(const float4*)(src + vb + 4 * min(t + 256 * k, last >> 2));
    }
    const int nh = pen ? a.o.n_hist : 0;
    int h0 = 0, h1 = nh;
    int tok[RP_HIST], cnt[RP_HIST];
    auto request = [&](int j0) {
#pragma unroll
        for (int u = 0; u < RP_HIST; ++u) {
            const int e = min(j0 + 256 * u, nh - 1);
            tok[u] = a.o.hist_tok[e];
            cnt[u] = a.o.hist_cnt[e];
        }
    };
    if (pen && t < i) s_draft[t] = a.draft[t];
    if (t < MJ_ROWS) s_inh[t] = 0;
    if (nh > 256 * RP_HIST) {
        const int step = (nh + 255) / 256;
        const bool in = t * step < nh;
        const int smp = a.o.hist_tok[in ? t * step : 0];
        const int c0 = __syncthreads_count(in && smp < v0), c1 = __syncthreads_count(in && smp < v1);
        h0 = max(c0 - 1, 0) * step;
        h1 = min(c1 * step, nh);
    }
    if (h0 < h1) request(h0 + t);
    if (al) {
#pragma unroll
        for (int k = 0; k < RM_UNROLL; ++k)
            if (4 * (t + 256 * k) < n) *(float4*)(s_l + 4 * (t + 256 * k)) = f[k];
    } else {
        for (int b = t; b < n; b += 256 * 8) {
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k] = src[v0 + min(b + 256 * k, n - 1)];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (b + 256 * k < n) s_l[b + 256 * k] = x[k];
        }
    }
    __syncthreads();
    if (pen) {
        for (int j0 = h0 + t; j0 < h1; j0 += 256 * RP_HIST) {
            if (j0 != h0 + t) request(j0);
#pragma unroll
            for (int u = 0; u < RP_HIST; ++u) {
                if (j0 + 256 * u >= h1 || tok[u] < v0 || tok[u] >= v1) continue;
                for (int d = 0; d < i; ++d)
                    if (s_draft[d] == tok[u]) {
                        ++cnt[u];
                        s_inh[d] = 1;
                    }
                float& x = s_l[tok[u] - v0];
                x = penalize1(x, cnt[u], a.o.rep, a.o.pres, a.o.freq);
            }
        }
        __syncthreads();
        if (t < i) {
            const int tk = s_draft[t];
            bool first = tk >= v0 && tk < v1 && !s_inh[t];
            for (int e = 0; e < t; ++e) first = first && s_draft[e] != tk;
            if (first) {
                int c = 0;
                for (int e = 0; e < i; ++e) c += s_draft[e] == tk;
                s_l[tk - v0] = penalize1(s_l[tk - v0], c, a.o.rep, a.o.pres, a.o.freq);
            }
        }
        __syncthreads();
    }
    const bool wr = pen || a.src != a.logits;
    float m = -INFINITY;
    if (al) {
        for (int b = 4 * t; b < n; b += 4 * 256) {
            const float4 x = *(const float4*)(s_l + b);
            m = fmaxf(m, fmaxf(fmaxf(x.x, x.y), fmaxf(x.z, x.w)));
            if (wr) *(float4*)(dst + v0 + b) = x;
        }
    } else {
        for (int b = t; b < n; b += 256) {
            m = fmaxf(m, s_l[b]);
            if (wr) dst[v0 + b] = s_l[b];
        }
    }
    m = wave_max(m);
    __shared__ float sm[4];
    if ((t & 63) == 0) sm[t >> 6] = m;
    __syncthreads();
    if (t == 0) a.mpart[i * RMB + j] = fmaxf(fmaxf(sm[0], sm[1]), fmaxf(sm[2], sm[3]));
}

// Block sums of e_v: one 64-thread block per (row, 1024-element block), lane = chunk.  The
// row maximum (the lm_head's, or folded from the partial maxima) and the chunk's logits are
// requested together (clamped indices: every lane loads, lanes past the end contribute nothing).
__global__ __launch_bounds__(64) void k_sample_sums(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    const int row = blockIdx.x / a.nblocks, b = blockIdx.x % a.nblocks;
    const int lane = threadIdx.x;
    const int nch = (a.V + CH - 1) / CH;
    const int chunk = b * BLK + lane;
    float x[CH];
    chunk_logits(a, row, min(chunk, nch - 1), x);
    float mx;
    if (a.head_max)
        mx = a.head_max[row];
    else
        mx = wave_max(a.mpart[row * RMB + (lane & (RMB - 1))]);
    if (b == 0 && lane == 0) a.rowmax[row] = mx;
    const float mxs = mx * a.invT;
    const int v0 = chunk * CH;
    float cs = 0.0f;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const float e = e_of(a, x[k], mxs);
        if (v0 + k < a.V) cs = cs + e;
    }
    __shared__ float s[BLK];
    s[lane] = chunk < nch ? cs : 0.0f;
    __syncthreads();
    if (lane == 0) {
        float bs = 0.0f;
        for (int c = 0; c < BLK; ++c)
            if (b * BLK + c < nch) bs = bs + s[c];
        a.bsum[(size_t)row * a.nblocks + b] = bs;
    }
}

// The outcome (acc drafts accepted, then tok), written by the 64 lanes of one wave: lane i
// writes path[i] and emit[i] (the accepted drafts are read together).
__device__ __forceinline__ void write_result(const SampleArgs& a, int acc, int tok) {
    const int i = threadIdx.x & 63;
    if (a.out && i == 0) {
        a.out[0] = acc;
        a.out[1] = tok;
    }
    if (a.res) {
        if (i == 0) {
            a.res->accepted = acc;
            a.res->token = tok;
        }
        if (i <= acc) {
            a.res->path[i] = i;
            a.res->emit[i] = i < acc ? a.draft[i] : tok;
        }
    }
}

// Walk of a row to tgt over its mass (vals(c, x): chunk c's element values into x, their sum in
// element order, c clamped by the caller), given the running totals of its block sums (pref[b] = ((s_0 + s_1) + ...) + s_b, the totals a sequential walk
// forms): the first block whose running total reaches tgt (the last element if none), in it the
// first chunk (the block's 64 chunk sums recomputed in the same order, running on from the total
// before the block; the block's last element if none), then the first element of that chunk;
// writes (fr, token).  Block of 256 threads; the block's chunk sums and element values are
// computed once, and the running totals of a level are formed redundantly by every lane of
// wave 0 so that the first lane reaching tgt is found by one ballot.
template <class F>
__device__ __forceinline__ void walk_write(const SampleArgs& a, int fr, float tgt,
                                           const float* pref, F vals) {
    const int t = threadIdx.x;
    const int nch = (a.V + CH - 1) / CH, nb = a.nblocks;
    __shared__ __align__(16) float cs[BLK];
    __shared__ __align__(16) float ev[BLK][CH + 4];
    __shared__ int s_blk;
    if (t == 0) s_blk = nb;
    __syncthreads();
    if (t < nb && tgt <= pref[t]) atomicMin(&s_blk, t);  // nb <= MAX_CHUNKS / BLK <= 256
    __syncthreads();
    const int blk = s_blk;
    if (blk == nb) {  // block-uniform
        if (t < 64) write_result(a, fr, a.V - 1);
        return;
    }
    const int c0 = blk * BLK, n = min(BLK, nch - c0);
    const float P = blk > 0 ? pref[blk - 1] : 0.0f;
    if (t < BLK) {
        float x[CH];
        cs[t] = vals(min(c0 + t, nch - 1), x);
        float4* e4 = (float4*)ev[t];
#pragma unroll
        for (int k = 0; k < CH / 4; ++k)
            e4[k] = make_float4(x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]);
    }
    __syncthreads();
    if (t >= 64) return;  // wave 0 finishes (wave-uniform)
    // chunk level: lane k keeps the running total after chunk k
    float Q = P, Qk = 0.0f;
#pragma unroll
    for (int k = 0; k < BLK; ++k) {
        Q = Q + cs[k];
        Qk = t == k ? Q : Qk;
    }
    const int ci = wave_first(t < n && tgt <= Qk);
    int tok;
    if (ci < 0) {
        tok = min((c0 + n) * CH, a.V) - 1;
    } else {
        const int cc = c0 + ci;
        const int ne = min(CH, a.V - cc * CH);
        float R = ci > 0 ? __shfl(Qk, ci - 1) : P, Rk = 0.0f;
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            R = R + ev[ci][k];
            Rk = t == k ? R : Rk;
        }
        const int ei = wave_first(t < ne && tgt <= Rk);
        tok = cc * CH + (ei < 0 ? ne - 1 : ei);
    }
    write_result(a, fr, tok);  // wave 0
}

// Single block: row totals (with their running totals kept for a walk) and the accept
// decisions, one row a lane; the first rejected row ends the chain.  A full accept samples the
// bonus here (or leaves it to the nucleus kernels); a reject hands row fr to k_resid_sums /
// k_resid_walk through the state.
__global__ __launch_bounds__(256) void k_sample_decide(SampleArgs a) {
    if (block_aborted(a.abort)) return;
    a = resolve(a);
    const int t = threadIdx.x;
    const int D = a.rows - 1;
    const int per = a.nblocks;
    __shared__ float Z[MJ_ROWS];
    __shared__ float pref[DEC_STAGE];  // row r's block sums at r * per, then their running totals
    __shared__ int s_fr;
    // the drafts' e values and every row's block sums, requested together
    int d = -1;
    float ed = 0.0f;
    if (t < D) {
        d = a.draft[t];
        if (d >= 0 && d < a.V)
            ed = e_of(a, a.logits[(size_t)t * a.V + d], a.rowmax[t] * a.invT);
    }
    stage_lds(pref, a.bsum, a.rows * per, t, 256);
    __syncthreads();
    if (t < a.rows) Z[t] = running_totals(pref + t * per, per);
    __syncthreads();
    if (t < 64) {  // wave 0: one draft a lane (D < MJ_ROWS == 64)
        bool rej = false;
        if (t < D) {
            const float p = (d >= 0 && d < a.V) ? __fdiv_rn(ed, Z[t]) : 0.0f;
            float q = a.q_mode == 1 ? a.q_uniform : (a.q_point ? a.q_point[t] : 1.0f);
            q = fmaxf(0.0f, q);
            float u0, u1;
            row_uniforms(a, t, u0, u1);
            rej = !(q > 0.0f && p > 0.0f && u0 <= fminf(1.0f, __fdiv_rn(p, q)));
        }
        const int f = wave_first(rej);
        const int fr = f < 0 ? D : f;
        if (t == 0) {
            s_fr = fr;
            if (fr < D) {
                float q = a.q_mode == 1 ? a.q_uniform : (a.q_point ? a.q_point[fr] : 1.0f);
                *a.state = SampleState{1, fr, a.draft[fr], 0, fmaxf(0.0f, q), Z[fr], 0.0f, 0.0f};
            } else {
                *a.state = SampleState{0, fr, -1, 0, 0.0f, Z[fr], 0.0f, 0.0f};
            }
        }
    }
    __syncthreads();
    const int fr = s_fr;
    if (fr < D) return;  // the residual kernels finish (block-uniform)
    // the bonus: sample the last row by a walk to u0 * Z over e (samplePrepared)
    float u0, u1;
    row_uniforms(a, fr, u0, u1);
    if (nucleus_on(a)) {
        if (t == 0) *a.nb.st = NucState{1, fr, fr, u0, Z[fr]};
        return;  // block-uniform
    }
    if (t == 0 && a.nb.st) a.nb.st->need = 0;
    const float mxs = a.rowmax[fr] * a.invT, Zf = Z[fr];
    walk_write(a, fr, u0 * Zf, pref + fr * per, [&](int c, float x[CH]) {
        return chunk_vals(a, fr, c, false, mxs, Zf, 0.0f, -1, x);
    });
}

// Residual block sums of the rejected row (same chunk / block order as the e sums): one 64-thread
// block per 1024-element block, lane = chunk.
__global__ __launch_bounds__(64) void k_resid_sums(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    const SampleState st = *a.state;
    if (st.phase != 1) return;
    const int b = blockIdx.x, lane = threadIdx.x;
    const int nch = (a.V + CH - 1) / CH;
    const int chunk = b * BLK + lane;
    const float mxs = a.rowmax[st.fr] * a.invT;
    float x[CH];
    const float cs = chunk_vals(a, st.fr, min(chunk, nch - 1), true, mxs, st.Zr, st.q, st.d, x);
    __shared__ float sc[BLK];
    sc[lane] = chunk < nch ? cs : 0.0f;
    __syncthreads();
    if (lane == 0) {
        float bs = 0.0f;
        for (int c = 0; c < BLK; ++c)
            if (b * BLK + c < nch) bs = bs + sc[c];
        a.rbs[b] = bs;
    }
}

// Round r's histogram of the nucleus selection (NUC_HBINS bins kept for each) set empty.
#define NUC_HBINS 2048
__device__ __forceinline__ void nuc_clear(const NucleusBuf& nb, int r, int t) {
#pragma unroll
    for (int k = 0; k < NUC_HBINS / 256; ++k) {
        nb.hcnt[NUC_HBINS * r + 256 * k + t] = 0u;
        nb.hmass[NUC_HBINS * r + 256 * k + t] = 0ull;
    }
}

// The rejected row's sample: the residual total S, then a walk to u1 * S over the residual, or,
// with no residual mass, samplePrepared of the row (nucleus kernels, or a walk to u1 * Z over e
// with the row's block sums).
__global__ __launch_bounds__(256) void k_resid_walk(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    const SampleState st = *a.state;
    const int t = threadIdx.x;
    // the nucleus selection's first histogram starts empty (its kernel adds to it next)
    if (a.nb.st) nuc_clear(a.nb, 0, t);
    if (st.phase != 1) return;
    __shared__ float s_S;
    __shared__ float pref[MAX_CHUNKS / BLK];
    stage_lds(pref, a.rbs, a.nblocks, t, 256);
    __syncthreads();
    if (t == 0) s_S = running_totals(pref, a.nblocks);
    __syncthreads();
    const float S = s_S;
    float u0, u1;
    row_uniforms(a, st.fr, u0, u1);
    const bool walk_resid = S > 0.0f;
    if (nucleus_on(a) && !walk_resid) {
        if (t == 0) *a.nb.st = NucState{1, st.fr, st.fr, u1, st.Zr};
        return;  // block-uniform
    }
    if (t == 0 && a.nb.st) a.nb.st->need = 0;
    if (!walk_resid) {  // block-uniform: the row's e block sums instead
        stage_lds(pref, a.bsum + (size_t)st.fr * a.nblocks, a.nblocks, t, 256);
        __syncthreads();
        if (t == 0) running_totals(pref, a.nblocks);
        __syncthreads();
    }
    const float mxs = a.rowmax[st.fr] * a.invT;
    walk_write(a, st.fr, walk_resid ? u1 * S : u1 * st.Zr, pref, [&](int c, float x[CH]) {
        return chunk_vals(a, st.fr, c, walk_resid, mxs, st.Zr, st.q, st.d, x);
    });
}

// ---- nucleus (samplePrepared, LogitsProcessor.swift:137-164) --------------------------------
// The cut, by radix selection.  The e of the nucleus row are non-negative floats, so their bits
// order as their values.  Round r (0..2) histograms digit r (bits 31..21, 20..10, 9..0) of the keys
// that match the digits already chosen: a count and an exact mass (sum of trunc(e * 2^40)) per
// digit value.  Scanning a round's digits from the top, the cut lies in the first digit whose
// mass, added to the mass of the keys above it, reaches the target; after three rounds the cut
// key is known exactly, and among the keys equal to it (ties, taken in id order) the cut is the
// j-th, j the fewest that reach the target.  NUC_BLOCKS blocks of 256 threads cover up to
// NUC_BLOCKS * 2048 ids, block b ids [2048 b, 2048 b + 2048); the last round also keeps each
// block's digit counts so the j-th tie is found without another pass.
// Every kernel scans the histogram before it with its whole block (a thread's digits, then sums
// across lanes); the state after a scan is left for the next kernel.  (One thread's walk of the
// digits, three and four histograms a round, took 21, 30 and 37 us; the kept sums and the walk on
// one CU, element by element, 164 us of a 152k-id row.)
#define NUC_BLOCKS 96
#define NUC_PER_BLOCK 2048

template <int R>
struct NucDigit {  // of round R
    static constexpr int BITS = R < 2 ? 11 : 10, BINS = 1 << BITS;
    static constexpr int SHIFT = R == 0 ? 21 : R == 1 ? 10 : 0;
    static constexpr int OFF = R * NUC_HBINS;  // first bin in hcnt / hmass
};

__device__ __forceinline__ uint64_t nuc_fixed(float e) {
    return (uint64_t)(e * 0x1p40f);  // exact scaling, then truncation (e <= 1)
}

__device__ __forceinline__ uint64_t nuc_target(const SampleArgs& a, float Z) {
    const float tp = a.o.top_p < 0.0f ? 0.0f : (a.o.top_p > 1.0f ? 1.0f : a.o.top_p);
    return nuc_fixed(tp * Z);
}

__device__ __forceinline__ uint64_t shfl_up64(uint64_t v, int o) {
    const uint32_t lo = __shfl_up((uint32_t)v, o, MJ_WAVE);
    const uint32_t hi = __shfl_up((uint32_t)(v >> 32), o, MJ_WAVE);
    return ((uint64_t)hi << 32) | lo;
}

// The selection after round R's histogram, from the state before it: prefix gains the digit, and
// above the mass of the keys ranked above that digit's; some = false when the target exceeds the
// row's whole mass (every key is kept).  Block of 256 threads, all of them get the result; thread t
// holds bins BINS - 1 - t PER .. downwards.
template <int R>
__device__ NucSel nuc_scan(const NucleusBuf& nb, NucSel s, uint64_t F) {
    using Dg = NucDigit<R>;
    constexpr int PER = Dg::BINS / 256;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int lo = Dg::OFF + Dg::BINS - (t + 1) * PER;  // the thread's lowest bin
    uint32_t cnt[PER];
    uint64_t mass[PER];
#pragma unroll
    for (int k = 0; k < PER; k += 4) {
        const u4v c = *(const u4v*)(nb.hcnt + lo + k);
#pragma unroll
        for (int j = 0; j < 4; ++j) cnt[k + j] = c[j];
    }
#pragma unroll
    for (int k = 0; k < PER; k += 2) {
        const u4v m = *(const u4v*)(nb.hmass + lo + k);
        mass[k] = ((uint64_t)m[1] << 32) | m[0];
        mass[k + 1] = ((uint64_t)m[3] << 32) | m[2];
    }
    uint64_t own = 0ull;
#pragma unroll
    for (int k = 0; k < PER; ++k) own += mass[k];
    uint64_t incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t y = shfl_up64(incl, o);
        if (lane >= o) incl += y;
    }
    __shared__ uint64_t s_w[4];
    __shared__ uint64_t s_above;
    __shared__ int s_bin;  // bins below the top
    if (lane == 63) s_w[wv] = incl;
    if (t == 0) s_bin = Dg::BINS;
    __syncthreads();
    uint64_t above = s.above + incl - own;
    for (int w = 0; w < wv; ++w) above += s_w[w];
    // the thread's first bin from the top that reaches the target
    int hit = Dg::BINS;
    uint64_t ha = 0ull;
#pragma unroll
    for (int k = PER - 1; k >= 0; --k) {
        if (hit == Dg::BINS && cnt[k] != 0u && above + mass[k] >= F) {
            hit = t * PER + PER - 1 - k;
            ha = above;
        }
        above += mass[k];
    }
    if (hit < Dg::BINS) atomicMin(&s_bin, hit);
    __syncthreads();
    if (hit < Dg::BINS && hit == s_bin) s_above = ha;
    __syncthreads();
    const int bin = s_bin;
    if (bin == Dg::BINS) s.some = 0;
    if (s.some) {
        s.prefix = (s.prefix << Dg::BITS) | (uint32_t)(Dg::BINS - 1 - bin);
        s.above = s_above;
    }
    return s;
}

// Round R of the selection; round 0 also computes the row's keys (e bits).
template <int R>
__global__ __launch_bounds__(256) void k_nucleus_round(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    using Dg = NucDigit<R>;
    const int t = threadIdx.x, b = blockIdx.x;
    // the next round's histogram starts empty
    if constexpr (R < 2)
        if (b == 0) nuc_clear(a.nb, R + 1, t);
    const NucState st = *a.nb.st;
    if (!st.need) return;
    constexpr int PT = NUC_PER_BLOCK / 256;
    // the thread's ids' logits (round 0) or keys, requested together ahead of the scan
    const float* lr = a.logits + (size_t)st.row * a.V;
    uint32_t key[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int v = min(b * NUC_PER_BLOCK + 256 * i + t, a.V - 1);
        key[i] = R == 0 ? __float_as_uint(lr[v]) : a.nb.keys[v];
    }
    __shared__ uint32_t s_cnt[Dg::BINS];
    __shared__ unsigned long long s_mass[Dg::BINS];
#pragma unroll
    for (int k = 0; k < Dg::BINS / 256; ++k) {
        s_cnt[256 * k + t] = 0u;
        s_mass[256 * k + t] = 0ull;
    }
    NucSel sel{0ull, 0u, 1};
    if constexpr (R == 2) sel = a.nb.sel[0];
    if constexpr (R > 0) {
        if (sel.some) sel = nuc_scan<(R > 0 ? R - 1 : 0)>(a.nb, sel, nuc_target(a, st.Z));
        if (b == 0 && t == 0) a.nb.sel[R - 1] = sel;
    }
    __syncthreads();
    if (!sel.some) return;  // block-uniform: every key is kept
    const float mxs = a.rowmax[st.row] * a.invT;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int v = b * NUC_PER_BLOCK + 256 * i + t;
        if (v >= a.V) break;
        if constexpr (R == 0) {
            key[i] = __float_as_uint(e_of(a, __uint_as_float(key[i]), mxs));
            a.nb.keys[v] = key[i];
        } else {
            if ((key[i] >> (Dg::SHIFT + Dg::BITS)) != sel.prefix) continue;
        }
        const int d = (key[i] >> Dg::SHIFT) & (Dg::BINS - 1);
        atomicAdd(&s_cnt[d], 1u);
        atomicAdd(&s_mass[d], (unsigned long long)nuc_fixed(__uint_as_float(key[i])));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < Dg::BINS / 256; ++k) {
        const int d = 256 * k + t;
        if (s_cnt[d] != 0u) {
            atomicAdd(a.nb.hcnt + Dg::OFF + d, s_cnt[d]);
            atomicAdd((unsigned long long*)(a.nb.hmass + Dg::OFF + d), s_mass[d]);
        }
        if constexpr (R == 2) a.nb.hblk[Dg::BINS * b + d] = s_cnt[d];
    }
}

// e of id v if the nucleus keeps it (a key above the cut, or the cut key up to the cut id), else 0
__device__ __forceinline__ float nuc_kept(uint32_t k, int v, uint32_t ck, int cid) {
    return (k > ck || (k == ck && v <= cid)) ? __uint_as_float(k) : 0.0f;
}

// The cut, and block sums of the kept e in the canonical order: one 256-thread block per 1024 ids
// (chunks of CH by the first wave).  Every block finds the cut for itself.
__global__ __launch_bounds__(256) void k_nucleus_sums(SampleArgs a) {
    if (block_aborted(a.abort)) return;
    a = resolve(a);
    const NucState st = *a.nb.st;
    if (!st.need) return;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, b = blockIdx.x;
    const int nch = (a.V + CH - 1) / CH, chunk = b * BLK + t;
    uint32_t k16[CH];  // the chunk's keys (clamped), requested ahead of the scan
    if (t < BLK) {
#pragma unroll
        for (int k = 0; k < CH; ++k) k16[k] = a.nb.keys[min(chunk * CH + k, a.V - 1)];
    }
    using Dg = NucDigit<2>;
    const uint64_t F = nuc_target(a, st.Z);
    NucSel sel = a.nb.sel[1];
    if (sel.some) sel = nuc_scan<2>(a.nb, sel, F);  // (block-uniform)
    uint32_t ck = 0u;   // the cut key
    int cid = a.V - 1;  // the cut id: with every key (or every tie) kept, the last
    if (sel.some) {
        ck = sel.prefix;
        // ties of the cut key, in id order: j of them reach the target (at least one)
        const uint64_t m = nuc_fixed(__uint_as_float(ck));
        const uint64_t need = F > sel.above ? F - sel.above : 0ull;
        const int j = need == 0ull ? 1 : (int)((need + m - 1) / m);
        const int d = ck & (Dg::BINS - 1);
        if (j < (int)a.nb.hcnt[Dg::OFF + d]) {  // block-uniform
            // the block of ids holding the j-th tie: running counts of the NUC_BLOCKS blocks
            __shared__ int s_b[4], s_blk, s_before, s_id;
            int c = t < NUC_BLOCKS ? (int)a.nb.hblk[Dg::BINS * t + d] : 0;
            auto block_incl = [&](int v) {  // inclusive sum over the block's threads
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int y = __shfl_up(v, o, MJ_WAVE);
                    if (lane >= o) v += y;
                }
                __syncthreads();
                if (lane == 63) s_b[wv] = v;
                __syncthreads();
                for (int w = 0; w < wv; ++w) v += s_b[w];
                return v;
            };
            int incl = block_incl(c);
            if (c > 0 && incl - c < j && j <= incl) {
                s_blk = t;
                s_before = incl - c;
            }
            __syncthreads();
            // the j-th tie in it: eight ids a thread
            const int jl = j - s_before, v0 = s_blk * NUC_PER_BLOCK + 8 * t;
            uint32_t eq = 0u;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                eq |= (uint32_t)(v0 + k < a.V && a.nb.keys[min(v0 + k, a.V - 1)] == ck) << k;
            c = __popc(eq);
            incl = block_incl(c);
            if (c > 0 && incl - c < jl && jl <= incl) {
                uint32_t e = eq;
                for (int k = incl - c + 1; k < jl; ++k) e &= e - 1u;
                s_id = v0 + __ffs(e) - 1;
            }
            __syncthreads();
            cid = s_id;
        }
    }
    if (b == 0 && t == 0) *a.nb.cut = NucCut{ck, cid};
    __shared__ float s[BLK];
    if (t >= BLK) return;  // the first wave sums
    float cs = 0.0f;
#pragma unroll
    for (int k = 0; k < CH; ++k)
        if (chunk * CH + k < a.V) cs = cs + nuc_kept(k16[k], chunk * CH + k, ck, cid);
    s[t] = chunk < nch ? cs : 0.0f;
    __builtin_amdgcn_wave_barrier();
    if (t == 0) {
        float bs = 0.0f;
        for (int c = 0; c < BLK; ++c)
            if (b * BLK + c < nch) bs = bs + s[c];
        a.rbs[b] = bs;
    }
}

// The sample: a walk in id order to u * (kept mass), one 256-thread block.
__global__ __launch_bounds__(256) void k_nucleus_pick(SampleArgs a) {
    if (aborted(a.abort)) return;
    a = resolve(a);
    const NucState st = *a.nb.st;
    if (!st.need) return;
    const NucCut cut = *a.nb.cut;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const uint32_t* keys = a.nb.keys;
    __shared__ float s_S;
    __shared__ float pref[MAX_CHUNKS / BLK];
    stage_lds(pref, a.rbs, a.nblocks, t, 256);
    __syncthreads();
    if (t == 0) s_S = running_totals(pref, a.nblocks);
    __syncthreads();
    const float S = s_S;
    if (S > 0.0f) {
        walk_write(a, st.acc, st.u * S, pref, [&](int c, float x[CH]) {
            uint32_t k16[CH];
#pragma unroll
            for (int k = 0; k < CH; ++k) k16[k] = keys[min(c * CH + k, a.V - 1)];
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < CH; ++k) {
                x[k] = nuc_kept(k16[k], c * CH + k, cut.key, cut.id);
                if (c * CH + k < a.V) sum = sum + x[k];
            }
            return sum;
        });
        return;
    }
    // no kept mass: the top-ranked token, the largest key, the lowest id among equal keys
    __shared__ uint32_t s_k[4];
    __shared__ int s_v[4];
    uint32_t bk = 0u;
    int bi = a.V;
    for (int v = t; v < a.V; v += 256) {
        const uint32_t k = keys[v];
        if (k > bk || (k == bk && v < bi)) {
            bk = k;
            bi = v;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t ok = __shfl_xor(bk, o, MJ_WAVE);
        const int oi = __shfl_xor(bi, o, MJ_WAVE);
        if (ok > bk || (ok == bk && oi < bi)) {
            bk = ok;
            bi = oi;
        }
    }
    if (lane == 0) {
        s_k[wv] = bk;
        s_v[wv] = bi;
    }
    __syncthreads();
    for (int w = 0; w < 4; ++w)
        if (s_k[w] > bk || (s_k[w] == bk && s_v[w] < bi)) {
            bk = s_k[w];
            bi = s_v[w];
        }
    if (t < 64) write_result(a, st.acc, bi < a.V ? bi : 0);
}

static size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t nucleus_bytes(int V) {
    return up256((size_t)V * 4) + up256(3 * NUC_HBINS * 4) + up256(3 * NUC_HBINS * 8) +
           up256((size_t)NUC_BLOCKS * NucDigit<2>::BINS * 4) + up256(sizeof(NucState)) +
           up256(2 * sizeof(NucSel)) + up256(sizeof(NucCut));
}

void nucleus_layout(void* base, int V, NucleusBuf& nb) {
    char* p = (char*)base;
    auto take = [&](size_t n) {
        char* q = p;
        p += up256(n);
        return (void*)q;
    };
    nb.keys = (uint32_t*)take((size_t)V * 4);
    nb.hcnt = (uint32_t*)take(3 * NUC_HBINS * 4);
    nb.hmass = (uint64_t*)take(3 * NUC_HBINS * 8);
    nb.hblk = (uint32_t*)take((size_t)NUC_BLOCKS * NucDigit<2>::BINS * 4);
    nb.st = (NucState*)take(sizeof(NucState));
    nb.sel = (NucSel*)take(2 * sizeof(NucSel));
    nb.cut = (NucCut*)take(sizeof(NucCut));
}

hipError_t launch_accept_sampled(float* logits, int rows, int V, const int32_t* draft,
                                 float temperature, int q_mode, const float* q_point,
                                 uint64_t seed, uint64_t counter, const SampleOpts& o,
                                 const NucleusBuf* nb, float* rowmax, float* bsum, int32_t* out,
                                 StepResult* res, const StepDesc* sd, const int* abort,
                                 hipStream_t st, const float* head_max, const float* src) {
    if (head_max && src) return hipErrorInvalidValue;
    SampleArgs a{};
    a.sd = sd;
    a.src = src ? src : logits;
    a.logits = logits;
    a.rows = rows;
    a.V = V;
    a.draft = draft;
    a.invT = 1.0f / fmaxf(temperature, 1e-5f);
    a.q_mode = q_mode;
    a.q_uniform = 1.0f / (float)V;
    a.q_point = q_point;
    a.seed = seed;
    a.counter = counter;
    a.rowmax = rowmax;
    a.nblocks = ((V + CH - 1) / CH + BLK - 1) / BLK;
    // the bsum buffer (sample_scratch_floats, 16-byte aligned): the hand-off state, block sums,
    // partial maxima, residual block sums
    a.state = (SampleState*)bsum;
    a.bsum = bsum + 8;
    a.mpart = a.bsum + (size_t)rows * a.nblocks;
    a.rbs = a.mpart + (size_t)rows * RMB;
    a.out = out;
    a.res = res;
    a.abort = abort;
    a.o = o;
    if (nb) a.nb = *nb;
    a.head_max = head_max;
    if (V > MAX_CHUNKS * CH || V > NUC_BLOCKS * NUC_PER_BLOCK || rows > MJ_ROWS)
        return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    if (!head_max) {
        // (a pass's options are on the device: one without penalties comes with head_max)
        const bool pen = sd != nullptr || src != nullptr ||
                         (fabsf(o.rep - 1.0f) > 1e-6f && o.rep > 0.0f) || o.pres != 0.0f ||
                         o.freq != 0.0f;
        if (pen)
            hipLaunchKernelGGL(k_row_prep, dim3(rows * RMB), dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL(k_row_max, dim3(rows * RMB), dim3(256), 0, st, a);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_sample_sums, dim3(rows * a.nblocks), dim3(64), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sample_decide, dim3(1), dim3(256), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_resid_sums, dim3(a.nblocks), dim3(64), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_resid_walk, dim3(1), dim3(256), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess || !nb) return e;
    hipLaunchKernelGGL(k_nucleus_round<0>, dim3(NUC_BLOCKS), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_nucleus_round<1>, dim3(NUC_BLOCKS), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_nucleus_round<2>, dim3(NUC_BLOCKS), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_nucleus_sums, dim3(a.nblocks), dim3(256), 0, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_nucleus_pick, dim3(1), dim3(256), 0, st, a);
    return hipGetLastError();
}

int sample_nblocks(int V) { return ((V + CH - 1) / CH + BLK - 1) / BLK; }

// floats of the buffer passed as bsum: 8 for the state, rows x nblocks block sums, rows x RMB
// partial maxima, nblocks residual block sums
size_t sample_scratch_floats(int rows, int V) {
    const size_t nb = (size_t)sample_nblocks(V);
    return 8 + (size_t)rows * nb + (size_t)rows * RMB + nb;
}
