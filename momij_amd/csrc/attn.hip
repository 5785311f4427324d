// attn.hip -- sliding-window attention over the fp16 KV cache for a pass of M verify rows
// arranged as a chain or a draft tree.
//
// k_attn_chunk      maple_sdpa_d128 math (SeedlessMetal.swift:2919-2997): softmax(q k^T /
//                   sqrt(128)) v in fp32, GQA.  Split-K over 64-key chunks ("flash decoding");
//                   one 256-thread block per (kv head, chunk or group of four, two or four of the
//                   pass's 16-vector query tiles) stages its Q (row x head of the kv group), K and
//                   V^T in LDS and runs QK^T and PV on v_mfma_f32_16x16x32_f16.
//                   Mask: committed positions inside the row's window [P-W+1, L-1]
//                   (AttentionMasks.swift:10-27) plus the row's ancestors and itself; a chain is
//                   the causal M-row pass.
//                   The block also finishes the projection's raw q and k rows as
//                   maple_qk_norm_rope + maple_write_kv_pair do (2794-2901): per-head RMSNorm(eps)
//                   * w, non-traditional half-split RoPE on the first rope_dim dims at the row's
//                   position L + depth(r) (angles from the pass's RoPE table).  Queries are
//                   finished by every block that takes them (they are small); the pass's own keys
//                   by the blocks whose chunk holds them, the first of which also appends them
//                   (K finished, V as projected) at slot (L + r) % C.  Of a wide prefill pass
//                   k_attn_finish does both in place before, and k_attn_combine appends.
// k_attn_combine    merges the chunk partials per (row, head) and writes the output in the qx
//                   format consumed by the o-projection.
#include <algorithm>

#include "mj_device.h"
#include "mj_internal.h"

#define HD 128
#define AK 64     // keys per chunk
#define QSTR 136  // LDS row stride (halves) of Q and K tiles
#define VSTR 72   // LDS row stride (halves) of V^T and P tiles

// Chunks of a pass.  Keys are placed by absolute position: chunk c0 + c holds positions
// [AK (c0 + c), AK (c0 + c) + AK - 1], key lane = position % AK.  The committed window
// [lo, L - 1] is laid out that way; so are a chain pass's own rows (row r at position L + r).
// A tree pass's own rows (positions repeat across siblings) follow in chunks of their own, by
// row index.  With keys placed by position, a row's chunk partials and their merge order depend
// only on the row's position, not on the other rows of the pass: a chain verify row computes
// bit for bit what a one-row pass at its position computes.
struct ChunkGeom {
    int64_t lo, hi;  // positions placed by position: [lo, hi]
    int64_t c0;      // absolute index of the first chunk
    int n_abs, nch;  // chunks placed by position; all chunks
};

__host__ __device__ inline ChunkGeom chunk_geom(int window, int64_t L, int M, bool chain) {
    ChunkGeom g;
    g.lo = window > 0 ? (L - window + 1 > 0 ? L - window + 1 : 0) : 0;
    g.hi = chain ? L + M - 1 : L - 1;
    g.c0 = g.lo / AK;
    g.n_abs = g.hi >= g.lo ? (int)(g.hi / AK - g.c0 + 1) : 0;
    g.nch = g.n_abs + (chain ? 0 : (M + AK - 1) / AK);
    return g;
}

int attn_max_chunks(int window, int64_t L_max, int M) {
    // position-aligned chunks: one more than the keys span, one for a tree's own rows
    const int64_t keys = (window > 0 ? (int64_t)window - 1 : L_max) + M;
    return (int)((keys + AK - 1) / AK) + 2;
}

// Groups of AG chunks, by absolute chunk index (a tree's own chunks are a group after them).  A
// group's partial is its chunks merged in increasing order (merge_part), whether one block
// computed them all or the combine merges the chunks of several: a row's result does not depend on
// which.
#define AG 4
__host__ __device__ inline int group_count(const ChunkGeom& g) {
    return (g.n_abs > 0 ? (int)((g.c0 + g.n_abs - 1) / AG - g.c0 / AG + 1) : 0) +
           (g.nch > g.n_abs ? 1 : 0);
}
// chunks cb .. ce - 1 of group j (none past the last group)
__device__ __forceinline__ void group_chunks(const ChunkGeom& g, int j, int& cb, int& ce) {
    const int64_t a0 = (g.c0 / AG + j) * AG - g.c0;  // first chunk of the group, may be < 0
    cb = a0 < 0 ? 0 : (int)a0;
    ce = (int)(a0 + AG < g.n_abs ? a0 + AG : g.n_abs);
    if (a0 >= g.n_abs) {  // past the chunks placed by position
        const bool own = j == group_count(g) - 1 && g.nch > g.n_abs;
        cb = own ? g.n_abs : g.nch;
        ce = g.nch;
    }
}
// Weights of the merge of a further part (maximum m) into a running one (mg): the new maximum
// replaces mg, the running sums scale by fa, the part's by fb.  Empty parts (-inf) leave exact
// values alone.
__device__ __forceinline__ void merge_part(float& mg, float m, float& fa, float& fb) {
    const float mn = fmaxf(mg, m);
    fa = mg == mn ? 1.0f : __builtin_amdgcn_exp2f(mg - mn);
    fb = m == mn ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
    mg = mn;
}

// DPP lane moves (no LDS round trip): quad_perm [1,0,3,2] (xor 1) 0xB1, [2,3,0,1] (xor 2)
// 0x4E; row_half_mirror 0x141
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// sum over each group of 8 lanes (the same bits in every lane of the group)
__device__ __forceinline__ float lane8_sum(float v) {
    v += dpp<0xB1>(v);
    v += dpp<0x4E>(v);
    v += dpp<0x141>(v);
    return v;
}
// max / sum over lanes i, i ^ 16, i ^ 32, i ^ 48 (v_permlane16_swap: rows 2k + 1 of the first
// operand trade places with rows 2k of the second; v_permlane32_swap: the upper half of the
// first with the lower half of the second; with both operands v each returns the (lower,
// upper) pair of values, so every lane combines them in the same order)
__device__ __forceinline__ float xrow_max(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float xrow_sum(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ void unpack8(const u4v v, float x[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        x[2 * j] = h2f(v[j] & 0xFFFFu);
        x[2 * j + 1] = h2f(v[j] >> 16);
    }
}
__device__ __forceinline__ u4v pack8(const float x[8]) {
    u4v o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (uint32_t)f2h(x[2 * j]) | ((uint32_t)f2h(x[2 * j + 1]) << 16);
    return o;
}

// One vector's RMSNorm and RoPE over eight lanes: a lane holds dims 8 pa + i (xa) and, X parts above,
// the dims they rotate with (xb), with their norm weights; cs: the row's angles.
template <int HALF>
__device__ __forceinline__ void finish_vec(float xa[8], float xb[8], const float wa[8],
                                           const float wb[8], const float2* cs_row, int pa,
                                           float eps) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(xa[i], xa[i], ss);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(xb[i], xb[i], ss);
    ss = lane8_sum(ss);
    const float scl = 1.0f / sqrtf(ss / (float)HD + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        xa[i] = xa[i] * scl * wa[i];
        xb[i] = xb[i] * scl * wb[i];
    }
    if constexpr (HALF > 0) {
        // dims 8 pa + i < half pair with 8 pa + i + half
        const bool rot = 8 * pa < HALF;
        const float2* cs = cs_row + (rot ? 8 * pa : 0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float2 c2 = cs[i];
            const float cx = rot ? c2.x : 1.0f, sy = rot ? c2.y : 0.0f;
            // (the fused products spelled out: the same wherever this is inlined)
            const float ra = fmaf(xa[i], cx, -(xb[i] * sy)), rb = fmaf(xb[i], cx, xa[i] * sy);
            xa[i] = ra;
            xb[i] = rb;
        }
    }
}

// Work of one block (kv head g, chunk c), 256 threads:
//   loads, every one issued before the first wait (all unconditional, at clamped addresses):
//     K: key t / 4, dims 32 (t % 4) ..      (the layout the own-key norm reduces over)
//     V: keys 4 (t % 16) .. + 3, dims 8 (t / 16) ..   (transposed in registers, 8-byte LDS rows)
//     Q: parts of 8 dims, four per thread (one round up to 16 rows)
//     the pass's RoPE table rows, staged in LDS once for the block's queries and own keys
//   barrier; q and the own keys finished (RMSNorm, RoPE) into LDS, own K / V appended; barrier
//   S^T = K Q^T on MFMA (A = 16 keys, B = 16 query vectors): lane (n, q) holds query vector n
//   against keys 16 kt + 4 q + r, so a query's mask, max and sum stay in its lane (plus two
//   cross-lane steps) and its probabilities are already the A operand of the PV product: that
//   product's k-slot 8 q + u takes key 32 j + 4 q + u (u < 4) or 32 j + 16 + 4 q + u - 4.
//   Scores are kept in log2 units (scale * log2 e), so p = exp2(s - m); the partial max is
//   stored in the same units.
#define LOG2E 1.44269504088896341f
// LDS of the RoPE table: M * half angles rounded up to whole 64-lane staging rounds
__host__ __device__ inline int tab_floats2(int M, int half) {
    return ((M * half / 2 + 63) / 64) * 64 * 2;
}
// HALF: rope_dim / 2 (0: no RoPE).  JR: finishing jobs (8 a vector) a thread requests before the
// first barrier; jobs past 256 JR go in further rounds, each a dependent load round trip, so
// passes with more of them take JR = 3.
// CG: chunks a block takes, 1, or AG (the chunks of a group in turn, the next one's K and V
// requested before the current one's products; the block's tiles are then at most one a wave).
// WIDE: the 64-row parts of a wide prefill pass in one launch, part z = blockIdx.z.  Queries and own
// keys are finished in place in the projection rows before it (k_attn_finish), so the keys of every
// pass row come from there, the older ones from the cache, and nothing is appended (k_attn_combine
// does, once nobody reads what the append overwrites).
template <int HALF, int JR, int CG, bool WIDE = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_chunk(AttnArgs a) {
    constexpr int NT = 256;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int g = blockIdx.x / a.parts, part = blockIdx.x % a.parts;
    const int z = WIDE ? blockIdx.z : 0;
    const StepDesc* sd = a.sd + z;
    const int64_t L = sd->L;
    const int M = WIDE ? sd->M : a.M;
    const int row0 = MJ_ROWS * z;  // the pass's rows before this part
    const int gqa = a.nQ / a.nKV;
    // the block's query vectors qv0 .. qv0 + nqv - 1: tpp tiles of 16 a block
    const int qv0 = 16 * a.tpp * blockIdx.y, nqt_all = (M * gqa + 15) / 16;
    const int nqt = min(a.tpp, nqt_all - a.tpp * (int)blockIdx.y);
    if (WIDE && nqt <= 0) return;  // whole block (a shorter last part)
    const int nqv = min(16 * nqt, M * gqa - qv0);
    // partials are laid out over the tiles of a whole part
    const int nqt_part = WIDE ? (MJ_ROWS * gqa + 15) / 16 : nqt_all;
    const int qkvN = (a.nQ + 2 * a.nKV) * HD;
    constexpr int half = HALF;
    const ChunkGeom cg = chunk_geom(a.window, L, M, sd->chain != 0);
    int c = part, ce = part + 1;
    if constexpr (CG > 1) group_chunks(cg, part, c, ce);
    if (c >= cg.nch) return;  // whole block
    // Positions are taken relative to L, in 32 bits (|p - L| < C < 2^23).  Key lane k of the
    // current chunk sits at rel = crel + k (chunks placed by position) and is of class -2 none,
    // -1 committed, else own row (its index); all by selects, no branches.
    const int C = (int)a.C, lo = (int)(cg.lo - L), hi = (int)(cg.hi - L);
    const int Lm = (int)((uint64_t)L >> 32 ? L % a.C : (int64_t)((uint32_t)L % (uint32_t)C));
    bool by_pos = true, own_chunk = false;
    int crel = 0, arow = 0;  // rel of lane 0; own row of lane 0 (a tree's chunks)
    auto set_chunk = [&]() {
        by_pos = c < cg.n_abs;
        crel = by_pos ? (int)((cg.c0 + c) * AK - L) : 0;
        arow = (c - cg.n_abs) * AK;
        // the pass's own rows fall in the current chunk
        own_chunk = by_pos ? crel + AK - 1 >= 0 && crel <= hi : true;
    };
    set_chunk();
    auto slot_of = [&](int rel) -> int {  // ring slot
        int sl = Lm + rel;
        sl += sl < 0 ? C : 0;
        sl -= sl >= C ? C : 0;
        return sl;
    };
    auto key_of = [&](int k) -> int {
        const int rel = crel + k, ar = arow + k;
        const int cp = (rel < lo) | (rel > hi) ? -2 : rel < 0 ? -1 : rel;
        const int ct = ar < M ? ar : -2;
        return by_pos ? cp : ct;
    };

    extern __shared__ uint16_t lds[];
    uint16_t* Qs = lds;                          // [nqt*16][QSTR]
    uint16_t* Ks = Qs + nqt * 16 * QSTR;         // [AK][QSTR]
    uint16_t* Vt = Ks + AK * QSTR;               // [HD][VSTR]
    float2* tab = (float2*)(Vt + HD * VSTR);     // [M][half] RoPE angles of the pass's rows
    int* kmeta = (int*)(tab + tab_floats2(M, half));  // [AK] key: (p - L) * 128 + (class + 2)
    int* rlo = kmeta + AK;                       // [MJ_ROWS] window start of a row, - L
    uint64_t* ranc = (uint64_t*)(rlo + MJ_ROWS);  // [MJ_ROWS] ancestor masks
    uint16_t* qnw_s = (uint16_t*)(ranc + MJ_ROWS);  // [HD] q norm weights
    uint16_t* knw_s = qnw_s + HD;                  // [HD] k norm weights
    int* s_abort = (int*)(knw_s + HD);

    // ---- K: key kk = t / 4, dims 32 dq ..;  V: keys 4 vg .. 4 vg + 3, dims 8 vd ..
    const int kk = t >> 2, dq = t & 3;
    const int vg = t & 15, vd = t >> 4;
    u4v kv[4], vv[4];
    int kcls = -2, vcls[4];
    // each 8-dim part from the projection (own rows) or the cache, at clamped slots
    auto src_of = [&](int cls, int k, const uint16_t* own, const uint16_t* cache) {
        const int pr = WIDE ? row0 + crel + k : cls;  // pass row
        const bool inp = WIDE ? cls != -2 && pr >= 0 : cls >= 0;
        const int sl = cls == -1 && !inp ? slot_of(crel + k) : 0;
        const uint32_t off = inp ? (uint32_t)(pr * qkvN) : (uint32_t)(sl * HD);
        return (inp ? own : cache) + off;
    };
    const uint16_t* const kown = a.qkv + (a.nQ + g) * HD;
    const uint16_t* const vown = kown + a.nKV * HD;
    const uint16_t* const kcg = a.kc + (size_t)g * a.C * HD;
    const uint16_t* const vcg = a.vc + (size_t)g * a.C * HD;
    auto request_kv = [&]() {
        kcls = key_of(kk);
#pragma unroll
        for (int j = 0; j < 4; ++j) vcls[j] = key_of(4 * vg + j);
        const uint16_t* ks = src_of(kcls, kk, kown, kcg) + 32 * dq;
#pragma unroll
        for (int q = 0; q < 4; ++q) kv[q] = *(const u4v*)(ks + 8 * q);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            vv[j] = *(const u4v*)(src_of(vcls[j], 4 * vg + j, vown, vcg) + 8 * vd);
    };
    request_kv();
    // ---- vectors to finish (RMSNorm + RoPE): the block's queries (vector qv = r * gqa + j is
    // head g * gqa + j of row r) and the pass's own keys in this chunk (lanes ko0 .. ko1 - 1).
    // Job jb of a vector holds its parts pa and pa + X (8 dims each; X = half / 8 parts apart,
    // so a rotated pair of dims sits in one thread), 8 jobs a vector in 8 consecutive threads.
    constexpr int X = HALF >= 16 ? HALF / 8 : 8;
    // (nqj: queries among the jobs -- all of the block's with its first chunk, none later)
    int ko0 = 0, ko1 = 0, njobs = 0, nqj = nqv;
    u4v jxa[JR], jxb[JR];
    auto job_src = [&](int j, int& pa) -> const uint16_t* {
        const int vi = j >> 3, jb = j & 7;
        pa = (jb & (X - 1)) | ((jb & ~(X - 1)) << 1);
        const bool isq = vi < nqj;
        const int r2 = max(key_of(ko0 + vi - nqj), 0);
        const int qr = (qv0 + vi) / gqa, qh = g * gqa + (qv0 + vi) - qr * gqa;
        return a.qkv + (uint32_t)((isq ? qr : r2) * qkvN + (isq ? qh : a.nQ + g) * HD);
    };
    auto request_jobs = [&]() {
        ko0 = ko1 = 0;
        if (own_chunk) {
            ko0 = by_pos ? max(-crel, 0) : 0;
            ko1 = min(by_pos ? hi - crel + 1 : M - arow, AK);
        }
        njobs = 8 * (nqj + ko1 - ko0);
        if (CG > 1 && njobs == 0) return;
#pragma unroll
        for (int jj = 0; jj < JR; ++jj) {
            const int j = t + NT * jj;
            int pa;
            const uint16_t* src = job_src(j < njobs ? j : njobs - 1, pa);
            jxa[jj] = *(const u4v*)(src + 8 * pa);
            jxb[jj] = *(const u4v*)(src + 8 * (pa + X));
        }
    };
    u4v qf[4];  // WIDE: 16-byte parts of the block's finished queries
    if constexpr (WIDE) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = t + NT * j, v = qv0 + min(e >> 4, nqv - 1), r = v / gqa;
            qf[j] = *(const u4v*)(a.qkv + (uint32_t)((row0 + r) * qkvN +
                                                     (g * gqa + v - r * gqa) * HD + 8 * (e & 15)));
        }
    } else {
        request_jobs();
    }
    // the norm weights into LDS (16 lanes each of wave 0)
    if (!WIDE && wv == 0 && lane < HD / 8) {
        __builtin_amdgcn_global_load_lds(a.q_norm_w + 8 * lane,
                                         (__attribute__((address_space(3))) void*)qnw_s, 16, 0, 0);
        __builtin_amdgcn_global_load_lds(a.k_norm_w + 8 * lane,
                                         (__attribute__((address_space(3))) void*)knw_s, 16, 0, 0);
    }
    // ---- RoPE table rows (float4 = two angles), key and row metadata
    // the table goes straight into LDS (16 bytes a lane): pairs 2e, 2e + 1 of the [M][half]
    // angles, wave w taking pairs 64 w + lane, 64 (w + 4) + lane, ...
    const int ntab4 = WIDE ? 0 : M * half / 2, hd = half > 0 ? half : 1;
    for (int e0 = 64 * wv; e0 < ntab4; e0 += NT) {
        const int e = e0 + lane;
        if (e < ntab4)
            __builtin_amdgcn_global_load_lds(a.rope_cs + (2 * e / hd) * MJ_ROPE_F + 2 * e % hd,
                                             (__attribute__((address_space(3))) void*)(tab + 2 * e0),
                                             16, 0, 0);
    }
    const int rdep = sd->depth[t < M ? t : M - 1];
    const uint64_t ranc_t = sd->anc[t < M ? t : M - 1];
    const int abort_v = a.abort ? *a.abort : 0;  // thread 0's copy decides for the block

    // ---- LDS: K rows (own keys raw for now), V^T, the table, metadata; the padding query
    // rows of the last tile (read by the MFMAs, masked after) are cleared
    for (int i = nqv * 16 + t; i < nqt * 16 * 16; i += NT)
        *(u4v*)(Qs + (i >> 4) * QSTR + 8 * (i & 15)) = (u4v){0u, 0u, 0u, 0u};
    if (t < M) {
        rlo[t] = a.window > 0 ? rdep - a.window + 1 : INT32_MIN / 2;
        ranc[t] = ranc_t;
    }
    if (t == 0) *s_abort = abort_v;
    if constexpr (WIDE) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = t + NT * j;
            if (e < 16 * nqv) *(u4v*)(Qs + (e >> 4) * QSTR + 8 * (e & 15)) = qf[j];
        }
    }
    const float sc2 = a.scale * LOG2E;
    const int ln = lane & 15, lq = lane >> 4;
    // the group's partial so far (CG > 1): maximum and sum of query vector ln, outputs as O below
    float mg = -INFINITY, lg = 0.0f;
    f4 og[CG > 1 ? 8 : 1];
#pragma unroll
    for (int dt = 0; dt < (CG > 1 ? 8 : 1); ++dt) og[dt] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    // partial `part` of query vector tile qt: lane (d, lq) holds query vectors 16 qt + 4 lq + r,
    // dim 16 dt + d
    auto write_part = [&](int qt, const f4* O, float m, float l) {
        const size_t pbase =
            ((size_t)(z * a.nKV + g) * a.max_chunks + part) * (size_t)(nqt_part * 16) + qv0 + qt * 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float* op = a.opart + (pbase + 4 * lq + r) * HD;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) op[16 * dt + ln] = O[dt][r];
        }
        if (lq == 0) a.mlpart[pbase + ln] = make_float2(m, l);
    };

  for (;;) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *(u4v*)(Ks + kk * QSTR + 32 * dq + 8 * q) = kcls != -2 ? kv[q] : (u4v){0u, 0u, 0u, 0u};
    u4v w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = vcls[j] != -2 ? vv[j] : (u4v){0u, 0u, 0u, 0u};
    // dim 8 vd + i of keys 4 vg .. + 3: halves i of the four key vectors
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int sh = 16 * (i & 1);
        const uint32_t a0 = (w[0][i >> 1] >> sh) & 0xFFFFu, a1 = (w[1][i >> 1] >> sh) & 0xFFFFu;
        const uint32_t a2 = (w[2][i >> 1] >> sh) & 0xFFFFu, a3 = (w[3][i >> 1] >> sh) & 0xFFFFu;
        *(uint2*)(Vt + (8 * vd + i) * VSTR + 4 * vg) = make_uint2(a0 | (a1 << 16), a2 | (a3 << 16));
    }
    if (t < AK) {
        const int mcls = key_of(t);
        // position - L: p - L in chunks placed by position, depth[row] for a tree's own rows
        int rel = crel + t;
        if (!by_pos) rel = sd->depth[mcls >= 0 ? mcls : 0];
        kmeta[t] = mcls == -2 ? (int)0x80000000 : rel * 128 + (mcls + 2);
    }
    __syncthreads();
    if (*s_abort) return;  // block-uniform

    // ---- finish the vectors: RMSNorm over the vector's 8 jobs, RoPE of dims d < half against
    // d + half (maple_qk_norm_rope); queries into Qs, own keys into Ks and appended at slot
    // (L + r) % C with their V rows (maple_write_kv_pair).  No other block of this launch
    // reads those slots (the committed window never reaches them).
    if constexpr (!WIDE)
    for (int j0 = 0; j0 < njobs; j0 += NT * JR) {
#pragma unroll
        for (int jj = 0; jj < JR; ++jj) {
            const int j = j0 + t + NT * jj;
            if (j0 > 0) {
                int pa;
                const uint16_t* src = job_src(j < njobs ? j : njobs - 1, pa);
                jxa[jj] = *(const u4v*)(src + 8 * pa);
                jxb[jj] = *(const u4v*)(src + 8 * (pa + X));
            }
            const int vi = j >> 3, jb = j & 7;
            const int pa = (jb & (X - 1)) | ((jb & ~(X - 1)) << 1), pb = pa + X;
            const bool isq = vi < nqj;
            const int kl = ko0 + vi - nqj;  // own key lane
            const int kr2 = max(key_of(kl), 0);
            const int row = min(isq ? (qv0 + vi) / gqa : kr2, M - 1);
            float xa[8], xb[8], wa[8], wb[8];
            unpack8(jxa[jj], xa);
            unpack8(jxb[jj], xb);
            const uint16_t* nw = isq ? qnw_s : knw_s;
            unpack8(*(const u4v*)(nw + 8 * pa), wa);
            unpack8(*(const u4v*)(nw + 8 * pb), wb);
            finish_vec<HALF>(xa, xb, wa, wb, tab + row * half, pa, a.eps);
            const u4v oa = pack8(xa), ob = pack8(xb);
            if (j < njobs) {
                if (isq) {
                    *(u4v*)(Qs + vi * QSTR + 8 * pa) = oa;
                    *(u4v*)(Qs + vi * QSTR + 8 * pb) = ob;
                } else {
                    *(u4v*)(Ks + kl * QSTR + 8 * pa) = oa;
                    *(u4v*)(Ks + kl * QSTR + 8 * pb) = ob;
                    if (blockIdx.y == 0) {
                        const size_t dst = ((size_t)g * a.C + slot_of(kr2)) * HD;
                        *(u4v*)(a.kc + dst + 8 * pa) = oa;
                        *(u4v*)(a.kc + dst + 8 * pb) = ob;
                    }
                }
            }
        }
    }
    if (!WIDE && own_chunk && blockIdx.y == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (vcls[j] >= 0)
                *(u4v*)(a.vc + ((size_t)g * a.C + slot_of(vcls[j])) * HD + 8 * vd) = vv[j];
    }
    // LDS-only barrier: the K / V appends above are read by later launches, not by this block
    // (it holds the finished keys in LDS), so they complete behind the attention work instead of
    // before it (__syncthreads would wait for the stores too)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // the group's next chunk: its K and V (and own keys) requested ahead of this one's products
    const bool more = CG > 1 && c + 1 < ce;
    if (more) {
        ++c;
        set_chunk();
        nqj = 0;
        request_kv();
        request_jobs();
    }

    const int qt = wv;  // a tile a wave
    if (qt < nqt) {
        // S^T tiles: keys 16 kt + 4 lq + r against query vector 16 qt + ln
        u4v qb[4];
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) qb[s4] = *(const u4v*)(Qs + (qt * 16 + ln) * QSTR + 32 * s4 + 8 * lq);
        // all of the tile's K operands requested before its first product, and the V operands
        // before the mask and softmax (left to itself the compiler waits for each LDS read in
        // turn)
        f4 S[4];
        u4v av[4][4];
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
                av[kt][s4] = *(const u4v*)(Ks + (16 * kt + ln) * QSTR + 32 * s4 + 8 * lq);
        int4 km[4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) km[kt] = *(const int4*)(kmeta + 16 * kt + 4 * lq);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) S[kt] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
                S[kt] = mfma16x16x32(as_h8(av[kt][s4]), as_h8(qb[s4]), S[kt]);
        const int qv = qt * 16 + ln;
        const int row = qv < nqv ? (qv0 + qv) / gqa : 0;
        const int lo_r = rlo[row];
        const uint64_t anc = ranc[row];
        // B lane (d, lq) of the PV products = V^T[d][32 j + 4 lq .. + 3] and [32 j + 16 + 4 lq ..]
        uint2 bl[2][8], bh[2][8];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const uint16_t* vr = Vt + (16 * dt + ln) * VSTR + 32 * j + 4 * lq;
                bl[j][dt] = *(const uint2*)vr;
                bh[j][dt] = *(const uint2*)(vr + 16);
            }
        __builtin_amdgcn_sched_barrier(0);
        float m = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = r == 0 ? km[kt].x : r == 1 ? km[kt].y : r == 2 ? km[kt].z : km[kt].w;
                const int cls = (e & 127) - 2;  // -2 invalid, -1 committed, >= 0 own row
                const bool ok = (qv < nqv) & (e != (int)0x80000000) & ((e >> 7) >= lo_r) &
                                ((cls < 0) | (((anc >> (cls & 63)) & 1ull) != 0));
                const float sv = ok ? S[kt][r] * sc2 : -INFINITY;
                S[kt][r] = sv;
                m = fmaxf(m, sv);
            }
        }
        m = xrow_max(m);
        float l = 0.0f;
        u4v pa[2];  // A operands of the two PV products (fp16 pairs)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(S[kt][r] - m);
                l += p[r];
            }
            pa[kt >> 1][2 * (kt & 1)] = (uint32_t)f2h(p[0]) | ((uint32_t)f2h(p[1]) << 16);
            pa[kt >> 1][2 * (kt & 1) + 1] = (uint32_t)f2h(p[2]) | ((uint32_t)f2h(p[3]) << 16);
        }
        l = xrow_sum(l);
        // O = P V
        f4 O[8];
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) O[dt] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const u4v bv = {bl[j][dt].x, bl[j][dt].y, bh[j][dt].x, bh[j][dt].y};
                O[dt] = mfma16x16x32(as_h8(pa[j]), as_h8(bv), O[dt]);
            }
        }
        if constexpr (CG == 1) {
            write_part(qt, O, m, l);
        } else {
            float fa, fb;
            merge_part(mg, m, fa, fb);
            lg = fmaf(fb, l, lg * fa);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // weights of query vector 4 lq + r
                const float far = __shfl(fa, 4 * lq + r, MJ_WAVE);
                const float fbr = __shfl(fb, 4 * lq + r, MJ_WAVE);
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) og[dt][r] = fmaf(fbr, O[dt][r], og[dt][r] * far);
            }
        }
    }
    if (!more) break;
    // every wave is done with this chunk's K, V and metadata
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
    if constexpr (CG > 1) {
        if (wv < nqt) write_part(wv, og, mg, lg);
    }
}

// One 256-thread block per (row, query head): wave w merges, in increasing order, the groups
// whose absolute index is w mod 4 (lane = two dims), then the four wave sums are added in wave
// order and the row is written in qx order.  A group is merged from its chunks first (CG 1), or
// came merged (CG 4).  Every part of the pass is there (a fully masked one has max -inf, sum 0,
// output 0 and adds exact zeros), so a row's merge depends only on the chunks that hold its keys.
// WIDE: of all parts of a wide pass; the blocks past its rows append the pass's keys and values to
// the cache, two rows a block (of rows that share a slot, the last).
template <int CG, bool WIDE = false>
__global__ __launch_bounds__(256) void k_attn_combine(AttnArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if constexpr (WIDE) {
        if ((int)blockIdx.x >= a.M * a.nQ) {
            const int row = 2 * (blockIdx.x - a.M * a.nQ) + (tid >> 7);
            if (aborted(a.abort) || row >= a.M || row + a.C < a.M) return;
            const int64_t slot = (a.sd->L + row) % a.C;
            const uint16_t* src = a.qkv + (size_t)row * (a.nQ + 2 * a.nKV) * HD + a.nQ * HD;
            for (int p = tid & 127; p < 2 * a.nKV * 16; p += 128) {
                const int h = p >> 4;  // K heads, then V heads
                uint16_t* dst = (h < a.nKV ? a.kc : a.vc) +
                                ((size_t)(h < a.nKV ? h : h - a.nKV) * a.C + slot) * HD;
                *(u4v*)(dst + 8 * (p & 15)) = *(const u4v*)(src + 8 * p);
            }
            return;
        }
    }
    const int r = blockIdx.x / a.nQ, hq = blockIdx.x % a.nQ;  // row of the pass
    const int z = WIDE ? r / MJ_ROWS : 0;
    const StepDesc* sd = a.sd + z;
    const int M = WIDE ? sd->M : a.M;
    const int gqa = a.nQ / a.nKV;
    const int g = z * a.nKV + hq / gqa, qv = (r - MJ_ROWS * z) * gqa + (hq % gqa);
    const size_t nq16 = (size_t)(((WIDE ? MJ_ROWS : M) * gqa + 15) / 16) * 16;
    const ChunkGeom cg = chunk_geom(a.window, sd->L, M, sd->chain != 0);
    const int ng = group_count(cg), nparts = CG == 1 ? cg.nch : ng;
    const int gs = (int)(((int64_t)wv - cg.c0 / AG) & 3);  // this wave's first group
    const float2* ml = a.mlpart + (size_t)g * a.max_chunks * nq16 + qv;
    const float* op = a.opart + ((size_t)g * a.max_chunks * nq16 + qv) * HD + 2 * lane;
    // a round: four parts, requested at clamped indices (parts past the end are skipped below) --
    // the chunks of one group, or four of the wave's groups; two rounds at once
    constexpr int GR = CG == 1 ? 1 : 4;  // groups a round
    float2 m4[2][4], p4[2][4];
    const int plast = nparts > 0 ? nparts - 1 : 0;
    auto request = [&](int gb, float2* mm, float2* pp) {
        int cb = 0, ce = 0;
        if constexpr (CG == 1) group_chunks(cg, gb, cb, ce);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = min(CG == 1 ? cb + j : gb + 4 * j, plast);
            mm[j] = ml[(size_t)c * nq16];
            pp[j] = *(const float2*)(op + (size_t)c * nq16 * HD);
        }
    };
    // the first two rounds, together with the maxima (they do not need them)
    request(gs, m4[0], p4[0]);
    request(gs + 4 * GR, m4[1], p4[1]);
    // the maximum over the parts (clamped indices: a repeated part leaves it unchanged)
    float mx = ml[(size_t)min(lane, plast) * nq16].x;
    for (int c = lane + 64; c < nparts; c += 64) mx = fmaxf(mx, ml[(size_t)c * nq16].x);
    mx = wave_max(mx);
    float o0 = 0.0f, o1 = 0.0f, ls = 0.0f;
    auto add_group = [&](float m, float l, float v0, float v1) {
        const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mx);  // log2 units
        ls = fmaf(l, w, ls);
        o0 = fmaf(w, v0, o0);
        o1 = fmaf(w, v1, o1);
    };
    for (int gb = gs, rd = 0; gb < ng; gb += 4 * GR, ++rd) {
        if (rd >= 2) request(gb, m4[0], p4[0]);
        const float2* mm = rd == 1 ? m4[1] : m4[0];
        const float2* pp = rd == 1 ? p4[1] : p4[0];
        if constexpr (CG == 1) {
            int cb, ce;
            group_chunks(cg, gb, cb, ce);
            float mg = -INFINITY, lg = 0.0f, g0 = 0.0f, g1 = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (cb + j >= ce) break;
                float fa, fb;
                merge_part(mg, mm[j].x, fa, fb);
                lg = fmaf(fb, mm[j].y, lg * fa);
                g0 = fmaf(fb, pp[j].x, g0 * fa);
                g1 = fmaf(fb, pp[j].y, g1 * fa);
            }
            add_group(mg, lg, g0, g1);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (gb + 4 * j >= ng) break;
                add_group(mm[j].x, mm[j].y, pp[j].x, pp[j].y);
            }
        }
    }
    __shared__ float s_o[4][HD];
    __shared__ float s_l[4];
    __shared__ int s_abort;
    s_o[wv][2 * lane] = o0;
    s_o[wv][2 * lane + 1] = o1;
    if (lane == 0) s_l[wv] = ls;
    if (tid == 0) s_abort = a.abort ? *a.abort : 0;
    __syncthreads();
    if (s_abort) return;
    if (tid < 16) {
        const float lsum = ((s_l[0] + s_l[1]) + s_l[2]) + s_l[3];
        const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
        u4v ov;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d = 8 * tid + 2 * j;
            const float v0 = (((s_o[0][d] + s_o[1][d]) + s_o[2][d]) + s_o[3][d]) * inv;
            const float v1 =
                (((s_o[0][d + 1] + s_o[1][d + 1]) + s_o[2][d + 1]) + s_o[3][d + 1]) * inv;
            ov[j] = (uint32_t)f2h(v0) | ((uint32_t)f2h(v1) << 16);
        }
        const int K = a.nQ * HD;
        emit_qx(ov, tid, a.out_perm + (size_t)r * K, a.out_sum + (size_t)r * (K / 64),
                hq * HD + 8 * tid);
    }
}

hipError_t launch_attn(const AttnArgs& args, hipStream_t st) {
    AttnArgs a = args;
    if (a.M < 1 || a.M > MJ_ROWS) return hipErrorInvalidValue;  // row metadata is staged per row
    // RoPE partners are found by lane moves: half = rope_dim / 2 in {16, 32, 64}
    if (a.rope_dim != 0 && a.rope_dim != 32 && a.rope_dim != 64 && a.rope_dim != 128)
        return hipErrorInvalidValue;
    // key positions relative to L are packed as (p - L) * 128 + class in an int
    if (a.C < 1 || a.C >= ((int64_t)1 << 23)) return hipErrorInvalidValue;
    const int gqa = a.nQ / a.nKV;
    const int nqt = (a.M * gqa + 15) / 16;
    // Groups of chunks a block where the keys run deep: the partials are the launch's traffic (64
    // rows at 6000 keys write and read 51 MB of them, 13 MB in groups: block 56 -> 48 us), but a
    // further chunk in turn costs a block 2.4 us (64 rows: at 3000 keys 45 -> 43 us, at 1500 39 ->
    // 42; one row at 6000 29 -> 30).  Query tiles: two a block until the blocks pass 400, then four
    // (64 rows at 130 keys 40 -> 34 us, at 1024 43 -> 39, where two a block take 42; 17 rows at
    // 1024 28.1 -> 27.4; before, one block took all of the pass's tiles).
    const int nch = std::min(a.nch, a.max_chunks);
    const bool groups = nch >= MJ_ATTN_DEEP && nqt >= 3;
    a.parts = groups ? (nch + 1) / AG + 2 : nch;
    a.tpp = a.nKV * a.parts * ((nqt + 1) / 2) <= 400 ? 2 : 4;
    if (a.tpp > nqt) a.tpp = nqt;
    const int qparts = (nqt + a.tpp - 1) / a.tpp;
    const size_t lds = (size_t)(a.tpp * 16 * QSTR + AK * QSTR + HD * VSTR) * 2 +
                       (size_t)tab_floats2(a.M, a.rope_dim / 2) * 8 + AK * 4 + MJ_ROWS * (4 + 8) +
                       2 * HD * 2 + 16;
    // finishing jobs of a block that also holds the pass's own keys
    const int jobs = 8 * (std::min(a.M * gqa, 16 * a.tpp) + (a.M < AK ? a.M : AK));
    const bool jr3 = jobs > 256 * 2;
    const dim3 grid(a.nKV * a.parts, qparts);
    auto go = [&](auto k2, auto k3, auto kg) {
        launch_timed(groups ? kg : jr3 ? k3 : k2, grid, dim3(256), lds, st, a);
    };
#define MJ_AT(H) go(k_attn_chunk<H, 2, 1>, k_attn_chunk<H, 3, 1>, k_attn_chunk<H, 2, AG>)
    switch (a.rope_dim) {
        case 0: MJ_AT(0); break;
        case 32: MJ_AT(16); break;
        case 64: MJ_AT(32); break;
        default: MJ_AT(64); break;
    }
#undef MJ_AT
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 rows(a.M * a.nQ);
    if (groups)
        hipLaunchKernelGGL(k_attn_combine<AG>, rows, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(k_attn_combine<1>, rows, dim3(256), 0, st, a);
    return hipGetLastError();
}

// The queries and keys of a wide pass's projection rows finished in place (RMSNorm, RoPE), the
// arithmetic of k_attn_chunk's jobs: eight lanes a vector.
template <int HALF>
__global__ __launch_bounds__(256) void k_attn_finish(AttnArgs a) {
    constexpr int X = HALF >= 16 ? HALF / 8 : 8;
    const int heads = a.nQ + a.nKV, vi = (blockIdx.x * 256 + threadIdx.x) >> 3, jb = threadIdx.x & 7;
    const int row = vi / heads, head = vi - row * heads;
    if (row >= a.M || aborted(a.abort)) return;  // (whole groups of eight)
    const int pa = (jb & (X - 1)) | ((jb & ~(X - 1)) << 1), pb = pa + X;
    uint16_t* v = const_cast<uint16_t*>(a.qkv) + (size_t)row * (a.nQ + 2 * a.nKV) * HD + head * HD;
    const uint16_t* nw = head < a.nQ ? a.q_norm_w : a.k_norm_w;
    float xa[8], xb[8], wa[8], wb[8];
    unpack8(*(const u4v*)(v + 8 * pa), xa);
    unpack8(*(const u4v*)(v + 8 * pb), xb);
    unpack8(*(const u4v*)(nw + 8 * pa), wa);
    unpack8(*(const u4v*)(nw + 8 * pb), wb);
    finish_vec<HALF>(xa, xb, wa, wb, a.rope_cs + (size_t)row * MJ_ROPE_F, pa, a.eps);
    *(u4v*)(v + 8 * pa) = pack8(xa);
    *(u4v*)(v + 8 * pb) = pack8(xb);
}

// Attention of a wide pass (a.M rows, a descriptor for each 64 at a.sd) with at most MJ_ATTN_DEEP - 1
// chunks a part: three launches for all parts.  (A part after another, each with a launch for its
// partials, took 13.7 us a part: 200-token prefill of four layers 865 us, 735 so.)  The cases past that
// keep the parts in turn: there a part's launch fills the chip, and partials for all parts at once
// would take hundreds of MB.
hipError_t launch_attn_wide(const AttnArgs& args, hipStream_t st) {
    AttnArgs a = args;
    if (a.M <= MJ_ROWS || a.M > MJ_WIDE_ROWS || a.nch >= MJ_ATTN_DEEP || a.nch > a.max_chunks)
        return hipErrorInvalidValue;
    if (a.C < 1 || a.C >= ((int64_t)1 << 23)) return hipErrorInvalidValue;
    const int gqa = a.nQ / a.nKV, nz = (a.M + MJ_ROWS - 1) / MJ_ROWS;
    const int nqt = (MJ_ROWS * gqa + 15) / 16;
    a.max_chunks = a.parts = a.nch;
    a.tpp = std::min(4, nqt);
    const int jobs = a.M * (a.nQ + a.nKV) * 8;
    const dim3 fg((jobs + 255) / 256), blk(256);
    switch (a.rope_dim) {
        case 0: hipLaunchKernelGGL(k_attn_finish<0>, fg, blk, 0, st, a); break;
        case 32: hipLaunchKernelGGL(k_attn_finish<16>, fg, blk, 0, st, a); break;
        case 64: hipLaunchKernelGGL(k_attn_finish<32>, fg, blk, 0, st, a); break;
        case 128: hipLaunchKernelGGL(k_attn_finish<64>, fg, blk, 0, st, a); break;
        default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t lds = (size_t)(a.tpp * 16 * QSTR + AK * QSTR + HD * VSTR) * 2 + AK * 4 +
                       MJ_ROWS * (4 + 8) + 2 * HD * 2 + 16;
    launch_timed(k_attn_chunk<0, 1, 1, true>, dim3(a.nKV * a.parts, (nqt + a.tpp - 1) / a.tpp, nz), blk,
                 lds, st, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_attn_combine<1, true>), dim3(a.M * a.nQ + (a.M + 1) / 2), blk, 0, st, a);
    return hipGetLastError();
}

template <int HALF>
static hipError_t attn_attr() {
    hipError_t e = hipSuccess;
    const void* ks[] = {(const void*)k_attn_chunk<HALF, 2, 1>, (const void*)k_attn_chunk<HALF, 3, 1>,
                        (const void*)k_attn_chunk<HALF, 2, AG>};
    for (const void* k : ks)
        if (e == hipSuccess)
            e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e;
}

hipError_t set_attn_attributes() {
    hipError_t e = attn_attr<0>();
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void*)k_attn_chunk<0, 1, 1, true>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess) e = attn_attr<16>();
    if (e == hipSuccess) e = attn_attr<32>();
    if (e == hipSuccess) e = attn_attr<64>();
    return e;
}
