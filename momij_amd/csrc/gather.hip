// gather.hip -- 2-bit affine gather GEMM for verify passes on v_mfma_f32_16x16x32_f16.
//
// Semantics as k_qmv2 / k_gather (gqmm2_rows, SeedlessMetal.swift:2168-2221): per 64-input
// block, y += s * (sum q*x) + b * (sum x), fp32.
//
// Layout of the work: a block serves one expert (or the dense projection) and a strip of
// its output rows.  It stages the activation rows routed to that expert (qx order, up to 16
// per pass) in LDS once for all its waves; which rows those are it forms itself, from the router
// logits or the pairs' expert ids, or reads from a slot table.  Each wave owns
// a tile of 16 weight rows over one K-slice (KS slices per tile, summed through LDS at the
// end).  It issues every load of its weight tile (scales, biases, then the codes in 1 KB
// column groups, global -> LDS directly) before its first wait, and runs the MFMAs of a
// column group as soon as that group has landed.  Blocks of experts that no row picked exit
// at once, so only routed experts are read, each once per pass.
//
// Epilogues: STORE y = half(acc); ADD y = half(y + half(acc)) (o-proj residual,
// gqmm2_rows_fold_add 3488-3543); SWIGLU clamped SwiGLU of the up || gate row pair
// (maple_clamped_swiglu 2435-2450) written in qx order with its block sums.
#include <algorithm>
#include <type_traits>

#include "mj_device.h"
#include "mj_internal.h"
#include "moe_topk.h"

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// 16 bytes per lane from global memory straight into LDS at lds + 16 * lane (wave-uniform lds)
__device__ __forceinline__ void load_lds16(const void* g, void* lds) {
    __builtin_amdgcn_global_load_lds(g, (lds_ptr_t)lds, 16, 0, 0);
}

// the same with a cache policy (16: sc1, device-coherent: sees stores of other XCDs made with
// sc1 once they have completed)
template <int CPOL>
__device__ __forceinline__ void load_lds16c(const void* g, void* lds) {
    __builtin_amdgcn_global_load_lds(g, (lds_ptr_t)lds, 16, 0, CPOL);
}

// 4 bytes per lane, landing at lds + 4 * lane
__device__ __forceinline__ void load_lds4(const void* g, void* lds) {
    __builtin_amdgcn_global_load_lds(g, (lds_ptr_t)lds, 4, 0, 0);
}

// Launch shape: R = 16 activation rows at most per pass (the MFMA M dimension), RA <= R rows
// staged in LDS per pass (a bucket with more rows takes several passes; `multi` says whether
// any can), K = 256 * KPL.  A block has WPB waves = TPB tiles of 16
// weight rows x KS K-slices: wave w owns tile w % TPB and K-slice w / TPB.
template <int KPL, int GS, int EPI, int WPB, int KS, bool ROWA = false>
struct G5Shape {
    static constexpr int R = 16;
    static constexpr int K = KPL * 256;
    static constexpr int KB = K / 64;          // 64-blocks per row (= 16-byte code chunks per row)
    static constexpr int KBW = KB / KS;        // 64-blocks of one wave's K-slice
    static constexpr int TPB = WPB / KS;       // weight tiles per block
    static constexpr int XS = K + 8;           // LDS row stride of activations (halves)
    static constexpr int SCH = K / GS / 8;     // 16-byte scale chunks per weight row
    // K / GS == 4 (K = 512, group 128): a row's scales are 8 bytes, half a chunk; they are
    // staged 8 bytes a row and read as chunk 0 with its upper half zero
    static constexpr bool HSC = SCH == 0;
    static constexpr int SCW = HSC ? 1 : SCH / KS;  // ... per K-slice
    static constexpr int WCODE = 16 * KBW * 16;  // bytes of one wave's code tile
    // bytes of one wave's scales (and of its biases); row-alpha tiles hold one alpha a row
    static constexpr int WSB = ROWA ? 32 : 16 * SCW * 16;
    static constexpr int WAVE_BYTES = WCODE + 2 * WSB;
    static constexpr int SS = KB + 2;          // LDS row stride of block sums (float2)
    static_assert(WAVE_BYTES >= 64 * 16, "a K-slice partial fits in its wave's tile area");
    static_assert(!HSC || (K / GS == 4 && KS == 1), "half-chunk scales: one K-slice of 4 groups");
    // K-slice partials: in a wave's own tile area when every bucket is one pass, else in their
    // own region (later passes reuse the tiles)
    static constexpr int RED = (KS - 1) * TPB * 64 * 16;
    __host__ __device__ static size_t lds(int RA, bool multi) {
        return (size_t)WPB * WAVE_BYTES + (size_t)RA * XS * 2 + (size_t)RA * SS * 8 +
               (multi ? RED : 0);
    }
};

// Weight tile of one wave: 16 rows x K codes with their scales and biases, fetched straight
// into LDS.  Scales and biases go first, then the codes in column groups: load j brings
// 64-blocks 4j .. 4j+3 of all 16 rows (16 runs of 64 bytes), so the MFMAs of group j start as
// soon as that load has landed while later groups are still streaming.  The code chunk
// (row r, block B) sits at slot 64 * (B / 4) + 4r + ((B % 4) ^ (r / 4)): lane (n, q) then reads
// word q of block B of row n from bank 16 (n % 4) + 4 ((B % 4) ^ (n / 4)) + q -- one 64-lane
// read touches every bank once.
//
// MFMA: A = 16 activation rows x 32 k (qx order, from LDS), B = word q of one 64-block of the
// 16 weight rows (lane (n, q)), so every MFMA stays inside one group of the scale and the
// block's partial sums D[4q+r][n] are scaled once, in fp32.  The affine remainder
// sum_B (b_B X_B - s_B Bx_B) is an fp32 MFMA chain over (block, term) pairs.

// s_waitcnt that waits for the vector-memory counter only (gfx9 encoding: expcnt and lgkmcnt
// left at their maximum)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier for LDS data only: this wave's LDS writes done (lgkmcnt 0) and at most N
// vector-memory loads still in flight (its LDS-DMA staging is older than those N), then
// s_barrier.  __syncthreads() would also drain every outstanding global load (its fence waits
// for vmcnt 0), i.e. the whole weight stream.  The "memory" clobber keeps LDS accesses on
// their side of it.
// 8-byte LDS store issued as inline assembly: the compiler would otherwise wait for every
// in-flight LDS-DMA load (it cannot prove the store misses their destinations) before it.  The
// ranges are disjoint by construction here; lds_barrier's lgkmcnt(0) orders the store.
__device__ __forceinline__ void lds_store_f2(float2* p, float2 v) {
    const uint32_t addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)p;
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(bits) : "memory");
}

template <int N>
__device__ __forceinline__ void lds_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Workgroup barrier that leaves vector-memory loads in flight: for LDS written with ds_write
// only (the next item's weight stream keeps landing meanwhile, in LDS nobody reads here).
__device__ __forceinline__ void lds_only_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// static LDS of the routing words of a launch that ranks up to FR rows itself
constexpr size_t g5_fused_rec_bytes(int FR) { return 64 * (4 + 8 + (FR > 16 ? 8 : 0)); }

// Pair table of a persistent launch whose slots follow from the pairs' expert ids (REC_IDS),
// built by every block from a.inds: byte i of id[l] = expert of pair l + 64 i, bit i of on[l] = the
// pair has one; slot[s] = expert | part << 8, experts in increasing id, an expert with more than
// `ps` pairs taking several slots (parts) of ps pairs.  Kept small: with 2.6 KB of it the up
// product staged 7 rows a pass instead of 8 (64 rows over 64 experts: 41 -> 47 us).
#define MJ_IDS_PS_MIN 8
struct IdsLds {
    uint64_t id[64];
    uint8_t on[64];
    uint16_t slot[MJ_MAX_EXPERTS + MJ_MAX_PAIRS / MJ_IDS_PS_MIN];
    int nslot, ps;
};

// How one call of the tile-gather body fits into a launch.  MODE 0: the whole launch (the
// standalone kernels).  The fused MoE kernel calls the up || gate body (MODE 1) and then the down
// body (MODE 2) in every block; io carries the routing words from the first to the second.
struct FuseIO {
    uint32_t em = 0;   // lane t: rows that picked expert t (bit r)
    uint64_t er = 0;   // ... and expert t's rank in rows 0 .. 15 (3 bits at 3r)
    uint64_t er1 = 0;  // ... and in rows 16 .. 31 (3 bits at 3 (r - 16))
    IdsLds* ids = nullptr;  // the launch's pair table (REC_IDS)
};

// Where a persistent launch's slot records come from.  REC_RANK: the launch ranks the router
// logits itself (passes of at most FR rows over at most 64 experts).  REC_IDS: from the expert id
// of every (row, slot) pair in global memory (any rows and experts a pass may have).
// REC_TAB (wide passes): from a slot table in global memory; the next item's record is requested
// behind the current one's weights.
enum { REC_NONE = 0, REC_RANK = 1, REC_IDS = 2, REC_TAB = 3 };

// FR: rows the fused routing ranks at most (16: two a wave, ranks in er; 32: four a wave, rows
// 16 .. 31's ranks in er1)
template <int KPL, int GS, int EPI, int WPB, int KS, int REC, bool ROWA, int MODE,
          int FR = MJ_G5_FUSED_ROWS>
__device__ __forceinline__ void g5_body(GatherArgs a, int RA, int multi, FuseIO& io) {
    constexpr bool PER = REC != REC_NONE;
    constexpr bool FUS = REC == REC_RANK && MODE != 2;  // ranks the logits in its prologue
    static_assert(FR == 16 || FR == 32, "fused routing rows");
    using S = G5Shape<KPL, GS, EPI, WPB, KS, ROWA>;
    constexpr bool LIST = REC == REC_IDS || REC == REC_TAB;  // slots of any number
    constexpr int R = S::R, K = S::K, KB = S::KB, KBW = S::KBW, TPB = S::TPB, XS = S::XS;
    constexpr int SCW = S::SCW;
    constexpr int NT = WPB * 64;
    constexpr int PPR = K / 8;                 // 16-byte parts per activation row
    static_assert(PPR % 64 == 0 && R % WPB == 0 && SCW >= 1 && SCW <= 4 && KBW % 4 == 0, "shape");

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int q = lane >> 4, n = lane & 15;
    const int tt = wv % TPB, kh = wv / TPB;   // weight tile and K-slice of this wave
    const int ncb = (a.N + 16 * TPB - 1) / (16 * TPB);
    const int u = blockIdx.x / ncb;
    int cb = blockIdx.x % ncb;
    const bool own_sums = a.xsum == nullptr;  // block sums formed here from the staged rows

    // Persistent expert mode (PER): the work items are (slot i / ncb, column block i % ncb);
    // block b takes items b, b + gridDim.x, ... until the slots end.  A slot is a routed expert
    // with the pairs that picked it; its record (pair j in lane j, the expert id and the pair
    // count in the high halves of lanes 0 and 1) is formed from registers or LDS.  Dense: rows
    // 0 .. dense_rows-1 in groups of R, block u taking group u (the blocks of a group stream the
    // same weights, concurrently with the other groups' blocks).
    int lpair = 0;  // pair j of the item's record in lane j
    const int rbase = PER ? 0 : R * u;  // dense: first row of the block's group
    int e = 0, np = PER ? 0 : min(R, a.dense_rows - rbase);
    int item = blockIdx.x;
    int rec_n = 0;  // the next item's record (persistent mode)
    extern __shared__ __align__(16) char g5lds[];

    // Fused routing (persistent up || gate product, rlogits set): every block ranks the router
    // logits itself -- the same top-k as the route kernel (row_topk) -- and keeps, per expert
    // t in lane t, the rows that picked it (em: bit r) and t's rank in each of them (er: 3 bits
    // a row).  A slot's record follows from these in registers: slots number the routed experts
    // in increasing id (as the route kernel's), a record lists its pairs (row * k + rank) by
    // row.  The last block also writes inds / scores.
    struct FusedRoute {
        // per expert t, set by LDS atomics as the rows are ranked: the rows that picked t (bit
        // r) and t's rank in each (3 bits at 3r for rows 0 .. 15, at 3 (r - 16) in er1 beyond)
        uint32_t em[64];
        uint64_t er[64];
        uint64_t er1[FR > 16 ? 64 : 0];
    };
    // (an instantiation of its own, FUS: the routing code stays out of the other kernels)
    constexpr bool FUSABLE = FUS;
    static_assert(!FUS || EPI == EPI_SWIGLU, "fused routing: persistent up || gate");
    __shared__ __align__(16) std::conditional_t<FUSABLE, FusedRoute, char> s_fr;
    __shared__ int s_stop;
    constexpr bool fused = FUS;
    static_assert(MODE == 0 || (MODE == 1 && FUS) || (MODE == 2 && REC == REC_RANK && EPI == EPI_STORE),
                  "fused MoE phases: up || gate with routing, then down");
    uint32_t em = MODE == 2 ? io.em : 0u;
    uint64_t er = MODE == 2 ? io.er : 0ull;
    uint64_t er1 = MODE == 2 ? io.er1 : 0ull;
    // record of slot sl: pair j in lane j, expert id and pair count in the high halves of lanes 0
    // and 1 (count 0 past the last slot)
    auto slot_rec = [&](int sl) -> int {
      if constexpr (REC == REC_TAB) {
        return a.tab[16 * min(sl, a.tab_slots - 1) + (lane & 15)];
      } else if constexpr (REC == REC_IDS) {
        // lane l holds the ids of pairs l + 64 i; the pairs of the slot's expert are numbered
        // in increasing index by ballots and sent to the lane of their number in the part.
        // Lanes with nothing to send, in round i, send to the lane below the round's first
        // (63 in the first round: it is only taken when every lane sends)
        if (sl >= io.ids->nslot) return 0;
        const int se = __builtin_amdgcn_readfirstlane((int)io.ids->slot[sl]);
        const int ex = se & 255, ps = io.ids->ps, base = (se >> 8) * ps;
        const uint64_t iv = io.ids->id[lane];
        const uint32_t onv = io.ids->on[lane];
        int tot = -base, got = 0;  // pairs before round i, from the part's first
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (64 * i >= a.npairs) break;
            const uint64_t bal =
                __ballot((int)((uint32_t)(iv >> (8 * i)) & 255u) == ex && ((onv >> i) & 1u) != 0u);
            if (bal == 0ull) continue;  // wave-uniform
            const int pos = tot + (int)__builtin_amdgcn_mbcnt_hi(
                                      (uint32_t)(bal >> 32),
                                      __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
            const int next = tot + __popcll(bal);
            const bool send = ((bal >> lane) & 1ull) != 0ull && (unsigned)pos < (unsigned)ps;
            const int dst = send ? pos : tot > 0 ? tot - 1 : 63;
            const int v = __builtin_amdgcn_ds_permute(4 * dst, lane + 64 * i);
            if (lane >= tot && lane < next) got = v;
            tot = next;
        }
        const int cnt = min(ps, tot);
        return (lane < cnt ? got : 0) | (lane == 0 ? ex << 16 : lane == 1 ? cnt << 16 : 0);
      } else {
        const uint64_t on = __ballot(em != 0u);
        const int mys = __popcll(on & ((1ull << lane) - 1ull));
        const uint64_t hit = __ballot(em != 0u && mys == sl);
        if (hit == 0) return 0;
        const int ex = __builtin_ctzll(hit);
        const uint32_t rm = __builtin_amdgcn_readlane(em, ex);
        auto rl64 = [&](uint64_t w) {
            return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(w >> 32), ex) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)w, ex);
        };
        const uint64_t rx0 = rl64(er), rx1 = FR > 16 ? rl64(er1) : 0ull;
        // lane r < FR (row r) sends its pair to lane "rows of ex before r"; the lanes that
        // send nothing send to lane 63, which no record entry uses (at most FR pairs)
        const int rr = lane & (FR - 1);
        const bool mine = lane < FR && ((rm >> rr) & 1u);
        const int pos = __popc(rm & ((1u << rr) - 1u));
        const int pr = rr * a.rk + (int)(((rr < 16 ? rx0 : rx1) >> (3 * (rr & 15))) & 7u);
        const int got = __builtin_amdgcn_ds_permute((mine ? pos : 63) * 4, pr);
        return got | (lane == 0 ? ex << 16 : lane == 1 ? __popc(rm) << 16 : 0);
      }
    };
    // the pair table, once a launch
    if constexpr (REC == REC_IDS) {
        IdsLds& t = *io.ids;
        static_assert(NT >= MJ_MAX_PAIRS && MJ_MAX_EXPERTS == 256, "a pair and an expert a thread");
        const int idv = tid < a.npairs ? a.inds[tid] : -1;
        uint32_t* s_cnt = (uint32_t*)g5lds;  // pairs per expert, where the weight tiles go later
        if (tid < MJ_MAX_EXPERTS) s_cnt[tid] = 0u;
        // one reading of the abort word decides for the block (its waves meet at barriers)
        if (tid == 0) t.nslot = aborted(a.abort) ? -1 : 0;
        __syncthreads();
        if (t.nslot < 0) return;
        const bool ok = (unsigned)idv < (unsigned)(a.experts > 0 ? a.experts : MJ_MAX_EXPERTS);
        if (tid < MJ_MAX_PAIRS) ((uint8_t*)t.id)[8 * (tid & 63) + (tid >> 6)] = (uint8_t)idv;
        if (ok) atomicAdd(&s_cnt[idv], 1u);
        // (pairs without an expert: their bits of the lanes' bytes go through the scratch)
        uint8_t* s_ok = (uint8_t*)(s_cnt + MJ_MAX_EXPERTS);
        if (tid < MJ_MAX_PAIRS) s_ok[tid] = ok ? 1 : 0;
        __syncthreads();
        if (wv == 1) {
            uint32_t b = 0u;
#pragma unroll
            for (int i = 0; i < 8; ++i) b |= (uint32_t)s_ok[64 * i + lane] << i;
            t.on[lane] = (uint8_t)b;
        }
        if (wv == 0) {
            // lane l numbers the slots of experts l, l + 64, l + 128, l + 192.  Parts of the RA rows
            // one pass takes: an expert's parts are neighbours in the item order and read its
            // weights from L2, with the next item's requests in flight meanwhile, where a second
            // pass of one item waited for its rows (MoE of 64 rows over 64 experts 75.6 -> 68.3
            // us on one box; parts of 64 rows: 72)
            int c[4], first = 0;
            uint64_t on[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                c[i] = (int)s_cnt[lane + 64 * i];
                on[i] = __ballot(c[i] > 0);
            }
            const int ps = max(RA, MJ_IDS_PS_MIN);
            if (__ballot(max(max(c[0], c[1]), max(c[2], c[3])) > ps) == 0ull) {
                // no expert in parts: no sums across lanes
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (c[i] > 0)
                        t.slot[first + __popcll(on[i] & ((1ull << lane) - 1ull))] =
                            (uint16_t)(lane + 64 * i);
                    first += __popcll(on[i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int parts = (c[i] + ps - 1) / ps;
                    int incl = parts;
#pragma unroll
                    for (int o = 1; o < 64; o <<= 1) {
                        const int y = __shfl_up(incl, o, MJ_WAVE);
                        if (lane >= o) incl += y;
                    }
                    for (int p = 0; p < parts; ++p)
                        t.slot[first + incl - parts + p] = (uint16_t)((lane + 64 * i) | (p << 8));
                    first += __shfl(incl, 63, MJ_WAVE);
                }
            }
            if (lane == 0) {
                t.nslot = first;
                t.ps = ps;
            }
        }
        __syncthreads();
    }
    if constexpr (FUSABLE) {
        static_assert(sizeof(FusedRoute) == g5_fused_rec_bytes(FR), "record bytes");
        static_assert(FR <= 4 * WPB, "at most four rows a wave");
        constexpr int RPW = (FR + WPB - 1) / WPB;  // rows a wave ranks
        if (fused) {
            const int M = a.rM, E = a.rE, k = a.rk;
            // row scratch in the weight tile area, free until the first item's loads
            float* s_row = (float*)g5lds + 64 * wv;                  // [WPB][64]
            float* s_gate = (float*)(g5lds + 256 * WPB) + 8 * wv;    // [WPB][8]
            int* s_ind = (int*)(g5lds + 288 * WPB) + 8 * wv;         // [WPB][8]
            // the wave's rows' logits (clamped row and expert: no branch waits) and the abort
            // flag requested together
            float v[RPW];
#pragma unroll
            for (int sr = 0; sr < RPW; ++sr)
                v[sr] = a.rlogits[min(wv + WPB * sr, M - 1) * E + min(lane, E - 1)];
            const bool ab = aborted(a.abort);
            if (tid == 0) s_stop = ab ? 1 : 0;  // one reading decides for the block, as block_aborted
            if (wv == 0) {
                s_fr.em[lane] = 0u;
                s_fr.er[lane] = 0ull;
                if constexpr (FR > 16) s_fr.er1[lane] = 0ull;
            }
            __syncthreads();  // (LDS only: the logits stay in flight)
            if (s_stop) return;
            // expert t picked by row r at rank rk: its bits, ORed in from any wave
            auto mark = [&](int t, int r, int rk) {
                __hip_atomic_fetch_or(&s_fr.em[t], 1u << r, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
                uint64_t* w = &s_fr.er[t];
                if constexpr (FR > 16) w = r < 16 ? w : &s_fr.er1[t];
                __hip_atomic_fetch_or(w, (uint64_t)rk << (3 * (r & 15)), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
            };
            const bool wr = blockIdx.x == gridDim.x - 1;  // writes inds / scores
#pragma unroll
            for (int sr = 0; sr < RPW; ++sr) {
                const int r = wv + WPB * sr;
                if (r >= M) break;
                s_row[lane] = lane < E ? v[sr] + 0.0f : -INFINITY;
                __builtin_amdgcn_wave_barrier();
                if (wr) {  // the selection with its weights
                    int ind = 0;
                    float gate = 0.0f;
                    row_topk<1>(s_row, E, k, s_ind, s_gate, ind, gate);
                    if (lane < k) {
                        mark(ind, r, lane);
                        a.rinds[r * k + lane] = ind;
                        a.rscores[r * k + lane] = gate;
                    }
                } else {  // the selection only: the ranks of row_topk, no weights
                    const int rank = row_rank64(s_row, E);
                    if (lane < E && rank < k) mark(lane, r, rank);
                }
                __builtin_amdgcn_wave_barrier();
            }
            __syncthreads();
            // lane t: the rows that picked expert t, and its rank in each
            em = s_fr.em[lane];
            er = s_fr.er[lane];
            if constexpr (FR > 16) er1 = s_fr.er1[lane];
            io.em = em;
            io.er = er;
            io.er1 = er1;
            // the row scratch is free for the weight tiles: every wave is past the barrier above
        }
    }
    {
        // (persistent: decided with the routing, for the block; dense: a wave by itself, since the
        // rows it writes follow from the block's index alone)
        const int ab = !PER && a.abort ? *a.abort : 0;
        if constexpr (PER) {
            if constexpr (MODE == 2) {
                // blocks with one up item fewer come free first: they take the first down items
                // (slots in increasing order, the order the up items complete in)
                const int nS = __popcll(__ballot(em != 0u));
                const int G = (int)gridDim.x, rem = (nS * a.fup_ncb) % G;
                item = (int)blockIdx.x >= rem ? (int)blockIdx.x - rem : (int)blockIdx.x + (G - rem);
            }
            const int rec = slot_rec(LIST ? item / ncb : min(item / ncb, 63));
            if constexpr (REC == REC_TAB)
                if (block_aborted(a.abort)) return;
            e = __builtin_amdgcn_readlane(rec, 0) >> 16;
            np = LIST || item / ncb < 64 ? __builtin_amdgcn_readlane(rec, 1) >> 16 : 0;
            lpair = rec & 0xFFFF;
            cb = item % ncb;
        }
        if (ab || np <= 0) return;  // whole block
    }

    char* wreg = g5lds + (size_t)wv * S::WAVE_BYTES;      // this wave's weight tile
    char* wcode = wreg;
    uint16_t* wsc = (uint16_t*)(wreg + S::WCODE);          // [16][K/GS/KS] this K-slice
    uint16_t* wbi = (uint16_t*)(wreg + S::WCODE + S::WSB);
    // one set of staged rows; persistent mode keeps two pair lists (the next item's rows are staged once
    // every wave is done with the current ones, while the current epilogue still needs its pairs)
    constexpr int NBUF = PER ? 2 : 1;
    uint16_t* const xs = (uint16_t*)(g5lds + (size_t)WPB * S::WAVE_BYTES);  // [RA][XS] qx rows
    float2* const xsl = (float2*)(xs + RA * XS);  // [RA][SS] {sum x, sum base*x}
    char* red = (char*)(xsl + RA * S::SS);  // [KS-1][TPB][64] f4
    __shared__ int s_pair[NBUF][R];
    int buf = 0;
    // pair of row i of the pass from pb
    auto pair_of = [&](int pb, int i) { return PER ? s_pair[buf][i] : rbase + pb + i; };

    // ---- activation rows of a pass, straight into LDS: rows < npass only (the rest feed
    // MFMA output rows that are discarded).  Wave w stages rows w, w + WPB, ...
    // residual add over dense rows: the first pass's residual values (rows 4q .. 4q + 3 of
    // output column n) are requested with the first rows, ahead of the weight stream, so the
    // epilogue does not wait on a dependent load (older than the weights, they change no wait
    // count)
    constexpr bool RES_PF = EPI == EPI_ADD && !PER;
    const bool res_pf = RES_PF && kh == 0;
    uint32_t resv[4] = {0u, 0u, 0u, 0u};
    auto stage_load = [&](int pb, int npass, int b, int lp, int npp, bool first = false) {
        const int myr = min(pb + (lane < R ? lane : 0), npp - 1);
        const int prl = PER ? __shfl(lp, myr, MJ_WAVE) : rbase + myr;
        if constexpr (RES_PF) {
            // (after the pair list: the wait for a list load would cover these too)
            if (first && res_pf) {
                // rows of the lane's outputs: q (a pass of at most 4 rows), else 4q .. 4q+3
                const int col = min((cb * TPB + tt) * 16, a.N - 16) + n;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = npass <= 4 ? q : 4 * q + r;
                    resv[r] = a.y[(size_t)(rbase + min(i, npass - 1)) * a.N + col];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < R / WPB; ++j) {
            const int r = wv + WPB * j;
            const int pr = __builtin_amdgcn_readlane(prl, r);
            if (PER && lane == 0) s_pair[b][r] = pr;
            if (r < npass) {
                const char* src = (const char*)(a.xperm + (size_t)(pr / a.x_div) * K);
#pragma unroll
                for (int i = 0; i < PPR / 64; ++i)
                    load_lds16c<MODE == 2 ? 16 : 0>(src + 1024 * i + 16 * lane,
                                                    (char*)(xs + r * XS) + 1024 * i);
                if (!own_sums && lane < KB / 2)
                    load_lds16((const char*)(a.xsum + (size_t)(pr / a.x_div) * KB) + 16 * lane,
                               xsl + r * S::SS);
            }
        }
    };
    // {sum x, sum base*x} of each (row, 64-block) from the staged rows: a block over eight lanes
    // (block_sum8).  With a block a lane, 64 elements in turn by one wave while the others waited, the
    // down product of 17 rows over 256 experts took 16.4 us (14.3 so), the fused launch of 9 rows
    // 31.2 (30.4).  Row and block by constants: with a division by the pass's rows, blocks of 9 rows
    // over 64 experts of 512 took 26.6 us (25.9 so; 25.5 before the slots came from ids), of 16 over 8
    // of 1024 25.4 (25.1; 24.6)
    auto own_block_sums = [&](int npass) {
        for (int idx = tid; idx < npass * KB * 8; idx += NT) {
            const int rb = idx >> 3, c = idx & 7, r = rb / KB, b = rb % KB;
            const float2 sums = block_sum8(*(const u4v*)(xs + r * XS + 64 * b + 8 * c));
            if (c == 0) lds_store_f2(xsl + r * S::SS + b, sums);
        }
    };

    // ---- a wave's weight tile, coalesced into LDS: scales and biases, then the code groups
    const int I = a.N / 2;
    // scales (when `scales`) and code column groups j0 .. j1-1 of the tile
    auto issue_weights = [&](int ee, int cbb, bool scales = true, int j0 = 0, int j1 = S::KBW / 4) {
        auto tile_row = [&](int r) -> size_t {  // global row of tile row r
            if constexpr (EPI == EPI_SWIGLU) {
                const int j0 = (cbb * TPB + tt) * 8;
                return (size_t)ee * a.N + (r < 8 ? j0 + r : I + j0 + r - 8);
            } else {
                // (a last column block may have fewer tiles: its other waves repeat the last)
                return (size_t)ee * a.N + min((cbb * TPB + tt) * 16, a.N - 16) + r;
            }
        };
        __builtin_amdgcn_sched_barrier(0);  // loads issued before stay ahead in the vmcnt queue
        if (!scales) {
        } else if constexpr (ROWA) {
            // row-alpha weights: one alpha per row (scale alpha, bias -alpha in every group);
            // tile rows 0..7 and 8..15 are each 8 consecutive rows, 16 bytes
            if (lane < 2) load_lds16((const char*)a.alpha + tile_row(8 * lane) * 2, wsc);
        } else if constexpr (S::HSC) {
            // 8 bytes of scales (and of biases) a row: lane l brings half l % 2 of row l / 2
            const char* sg = (const char*)a.s;
            const char* bg = (const char*)a.b;
            if (lane < 32) {
                load_lds4(sg + tile_row(lane >> 1) * 8 + 4 * (lane & 1), wsc);
                load_lds4(bg + tile_row(lane >> 1) * 8 + 4 * (lane & 1), wbi);
            }
        } else {
            const char* sg = (const char*)a.s;
            const char* bg = (const char*)a.b;
            if (lane < 16 * SCW) {
                const int r = lane / SCW, c = kh * SCW + lane % SCW;
                load_lds16(sg + tile_row(r) * (K / GS) * 2 + 16 * c, wsc);
                load_lds16(bg + tile_row(r) * (K / GS) * 2 + 16 * c, wbi);
            }
        }
        const char* wg = (const char*)a.w;
        const int r = lane >> 2, B4 = (lane & 3) ^ (r >> 2);
#pragma unroll
        for (int j = 0; j < KBW / 4; ++j)  // column group j: blocks kh*KBW + 4j .. +3
            if (j >= j0 && j < j1)
            load_lds16(wg + tile_row(r) * (K / 4) + 16 * (kh * KBW + 4 * j + B4),
                       wcode + 1024 * j);
        __builtin_amdgcn_sched_barrier(0);
    };
    // persistent mode: from the second item on, a wave's weights were issued as soon as its
    // MFMAs of the previous item were done (its tile is private to it), ahead of that item's
    // reduction and epilogue; the item's rows are staged after the block is done with the old
    // ones, so the item starts once everything it issued has landed
    bool early = false;
    // Fused MoE launch.  Up phase: an item's act values are stored device-coherent (sc1) into
    // act rows that the router launch filled with the marker 0xFFFF (a NaN, which the clamped
    // SwiGLU never produces: both its inputs are clamped to [-7, 7] first).  Down phase: an
    // item stages its rows at once and, once they have landed, checks them for the marker; rows
    // still marked are staged again.  The wait is bounded: the launch is sized so that every
    // block is resident, two a CU, and then every up item completes; a wait that runs out its
    // bound sets the fault word, which the host reports, and goes on, so the launch always ends.
    __shared__ int s_mark[WPB];
    // bit 0: a half of the pass's staged rows still holds the marker; bit 1, where it is looked at:
    // the abort word is set (thread 0's reading).  The same answer in every thread
    auto rows_marked = [&](int npass, bool look) -> int {
        bool bad = false;
        for (int idx = tid; idx < npass * (K / 8); idx += NT) {
            const int r = idx / (K / 8), c = idx - r * (K / 8);
            const u4v v = *(const u4v*)(xs + r * XS + 8 * c);
#pragma unroll
            for (int w = 0; w < 4; ++w)
                bad |= (v[w] & 0xFFFFu) == 0xFFFFu || (v[w] >> 16) == 0xFFFFu;
        }
        const bool wbad = __ballot(bad) != 0ull;
        int mine = wbad ? 1 : 0;
        if (look && wv == 0) mine |= aborted(a.abort) ? 2 : 0;
        if (lane == 0) s_mark[wv] = mine;
        lds_only_barrier();
        int any = 0;
#pragma unroll
        for (int w = 0; w < WPB; ++w) any |= s_mark[w];
        return any;
    };

  for (;;) {
    const int npass0 = min(RA, np);
    if (!early) {
        if constexpr (MODE == 2) {
            // the weights do not depend on the up phase: requested first, then the rows, checked
            // for the marker once they have landed
            issue_weights(e, cb);
            stage_load(0, npass0, buf, lpair, np, true);
            early = true;  // everything issued lands before the first pass
        } else {
            stage_load(0, npass0, buf, lpair, np, true);  // ahead of the weights (loads return in order)
            issue_weights(e, cb);
        }
    }
    const UnpackK uk = unpack_consts();
    const int xrow = min(n, RA - 1);
    const uint32_t* wq = (const uint32_t*)wcode + 16 * n + q;  // B: word q of row n's chunks

    // NR activation rows a lane's MFMA outputs hold.  A pass of at most 4 rows (NR = 1) places
    // staged row i at MFMA rows 4i .. 4i+3 (lane n reads row n / 4), so lane (n, q) holds row q
    // in each of its four outputs and scales and finishes one of them; more rows (NR = 4) sit at
    // MFMA rows 0 .. 15, lane (n, q) holding rows 4q .. 4q+3.  Each output is the same sum of the
    // same products either way.
    auto run_pass = [&](auto nr_t, int pb, int npass) {
        constexpr int NR = decltype(nr_t)::value;
        static_assert(NR == 1 || NR == 4, "rows a lane");
        const int xr = NR == 1 ? min(n >> 2, RA - 1) : xrow;
        constexpr int G = KBW / 4;  // code column groups, issued after the scale loads
        constexpr int NSB = ROWA ? 1 : 2;  // scale / bias loads of a tile
        // every wave's staged rows visible (this wave's were issued before its weights)
        if (pb == 0 && !early)
            lds_barrier<G + NSB>();
        else
            lds_barrier<0>();
        if constexpr (MODE == 2) {
            // act rows an up item has not finished yet: staged again until they have
            for (int it = 0;; ++it) {
                const int marks = rows_marked(npass, (it & 63) == 63);
                if (marks != 1) break;
                if (it >= a.fpolls) {
                    if (a.ffault != nullptr && tid == 0)
                        __hip_atomic_store(a.ffault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    break;
                }
                lds_only_barrier();  // every wave has read the marks before they are rewritten
                __builtin_amdgcn_s_sleep(8);
                stage_load(pb, npass, buf, lpair, np);
                lds_barrier<0>();
            }
        }
        if (own_sums) {
            own_block_sums(npass);
            lds_barrier<G + NSB>();
        }
        // ranked routing's up product: a stand-in load behind this item's weights (PF: one vector
        // load younger than them), whose value is consumed (times zero) so that it stays
        // a slot table's next record: requested there for good
        constexpr int PF = FUS || REC == REC_TAB ? 1 : 0;
        if constexpr (FUS) {
            if (pb == 0) rec_n = *(const int*)a.rlogits;
        } else if constexpr (REC == REC_TAB) {
            rec_n = slot_rec((item + (int)gridDim.x) / ncb);
        }
        wait_vmcnt<G + PF>();      // scales and biases have landed
        u4v sv[SCW], bv[SCW];
        float alpha_n = 0.0f;  // row-alpha weights: alpha of weight row n
        if constexpr (ROWA) {
            alpha_n = h2f(wsc[n]);
        } else if constexpr (S::HSC) {
            const uint2 ts = *(const uint2*)(wsc + 4 * n), tb = *(const uint2*)(wbi + 4 * n);
            sv[0] = (u4v){ts.x, ts.y, 0u, 0u};
            bv[0] = (u4v){tb.x, tb.y, 0u, 0u};
        } else {
#pragma unroll
            for (int c = 0; c < SCW; ++c) {
                sv[c] = *(const u4v*)(wsc + (n * SCW + c) * 8);
                bv[c] = *(const u4v*)(wbi + (n * SCW + c) * 8);
            }
        }
        // + sum_B (b_B X_B - s_B Bx_B): fp32 MFMA chains over k = (block, term) pairs, issued
        // while the codes are still arriving (scales, biases and activation sums are in);
        // A = activation sums of block 2i + q/2 (term q & 1), B = bias / -scale of row n
        f4 corr[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) corr[c] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
        const float* xcs =
            (const float*)(xsl + xr * S::SS + kh * KBW + (q >> 1)) + (q & 1);
        // this lane's B values: the biases (term 0) or the negated scales (term 1), taken from
        // the fp16 half of block 2i + q/2's group (the sign flipped in the fp16 bits)
        const uint32_t sgn = (q & 1) ? 0x8000u : 0u;
        const uint32_t hsh = 16u * (uint32_t)(q >> 1);
        if constexpr (ROWA) {
            // bias -alpha and scale alpha: B = -alpha for both terms
#pragma unroll
            for (int i = 0; i < KBW / 2; ++i)
                corr[i & 3] = mfma16x16x4f32(xcs[4 * i], -alpha_n, corr[i & 3]);
        } else {
            u4v mv[SCW];
#pragma unroll
            for (int c = 0; c < SCW; ++c)
#pragma unroll
                for (int w = 0; w < 4; ++w) mv[c][w] = (q & 1) ? sv[c][w] : bv[c][w];
#pragma unroll
            for (int i = 0; i < KBW / 2; ++i) {
                const float xa_k = xcs[4 * i];  // block 2i + q/2
                uint32_t h;
                if constexpr (GS == 64) {  // group 2i + q/2: word i % 4 of chunk 2i / 8, half q/2
                    h = mv[(2 * i) / 8][i % 4] >> hsh;
                } else {  // group i
                    h = mv[i / 8][(i % 8) / 2] >> (16 * (i & 1));
                }
                const float wk = h2f((uint16_t)(h ^ sgn));
                corr[i & 3] = mfma16x16x4f32(xa_k, wk, corr[i & 3]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // A: activation row xr, quarter q, of this K-slice
        const uint16_t* xak = xs + xr * XS + 16 * q + 64 * kh * KBW;
        // the correction chain's sum starts the accumulator (its four partial chains are
        // then free); outputs r >= NR stay unused
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[r] = (corr[0][r] + corr[1][r]) + (corr[2][r] + corr[3][r]);
        // row-alpha weights: every block has scale alpha, so the MFMA sums chain over the whole
        // slice and alpha scales them once
        f4 dacc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};  // even / odd blocks
        // persistent mode, last pass of the item: the next item (its record, and whether there
        // is one) and its weights.  In the fused launch (records formed from registers) the
        // scales and first half of the code groups are requested once this item's first half
        // is done (its scales are in registers, its first half's codes read), the rest after
        // its MFMAs; the item waits for its own groups first, so later waits count nothing new
        constexpr bool SPLIT = PER && (MODE != 0 || LIST) && G >= 2;
        constexpr int GP = G / 2;  // code groups a part (four parts measured slower)
        bool stage_next = false;
        int np_next = 0;
        auto next_item = [&]() {
            if constexpr (PER) {
                const int nx = item + (int)gridDim.x;
                if constexpr (REC == REC_TAB) {
                } else if constexpr (REC == REC_IDS) {
                    rec_n = slot_rec(nx / ncb);
                } else if constexpr (MODE == 2) {
                    rec_n = slot_rec(min(nx / ncb, 63));
                } else {
                    rec_n = slot_rec(min(nx / ncb, 63)) | (rec_n & (int)opaque(0u));
                }
                np_next = __builtin_amdgcn_readlane(rec_n, 1) >> 16;
                stage_next = pb + RA >= np && (LIST || nx / ncb < 64) && np_next > 0;
            }
        };
        // sum_B s_B * (sum q x)_B: per 64-block f16 MFMA sums, scaled in fp32, one column group
        // at a time as its codes arrive
        // fused launch: the wave computes at raised priority (s_setprio, the issue arbiter's
        // order among the CU's ready waves), so a wave whose tile has landed gets through its
        // groups, and to its next item's requests, ahead of waves still on the unpack of
        // theirs (launch 31.2 -> 30.1 us; through the epilogue as well: 30.4 us; a second
        // level for the second half: step 1.552 -> 1.548 ms)
        if constexpr (SPLIT) __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < G; ++j) {
          if (!(SPLIT && j >= GP && stage_next)) {
            if (j == 0) wait_vmcnt<G - 1 + PF>();
            if (j == 1) wait_vmcnt<(G >= 2 ? G - 2 : 0) + PF>();
            if (j == 2) wait_vmcnt<(G >= 3 ? G - 3 : 0) + PF>();
            if (j == 3) wait_vmcnt<(G >= 4 ? G - 4 : 0) + PF>();
            if (j == 4) wait_vmcnt<(G >= 5 ? G - 5 : 0) + PF>();
            if (j == 5) wait_vmcnt<(G >= 6 ? G - 6 : 0) + PF>();
            if (j == 6) wait_vmcnt<(G >= 7 ? G - 7 : 0) + PF>();
            if (j == 7) wait_vmcnt<PF>();
          }
            __builtin_amdgcn_sched_barrier(0);
            // LDS operands two blocks at a time (2 code words, 4 activation fragments), both
            // blocks' requested before the first is used
#pragma unroll
            for (int B2 = 4 * j; B2 < 4 * j + 4; B2 += 2) {
                uint32_t wd[2];
                u4v xv[2][2];
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    // word q of chunk slot 64 j + 4n + ((B % 4) ^ (n / 4)), B = B2 + b
                    wd[b] = wq[256 * j + 4 * (((B2 + b) & 3) ^ (n >> 2))];
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        xv[b][h] = *(const u4v*)(xak + 64 * (B2 + b) + 8 * h);
                }
#pragma unroll
              for (int b = 0; b < 2; ++b) {  // block kh * KBW + B
                const int B = B2 + b;
                uint32_t v[8];
                unpack16k(wd[b], v, uk);
                if constexpr (ROWA) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const u4v bq = {v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
                        dacc[b] = mfma16x16x32(as_h8(xv[b][h]), as_h8(bq), dacc[b]);
                    }
                } else {
                    f4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const u4v bq = {v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
                        d = mfma16x16x32(as_h8(xv[b][h]), as_h8(bq), d);
                    }
                    const int g = B * 64 / GS;
                    const uint32_t sw = opaque(sv[g / 8][(g % 8) / 2]);
                    const float sc = h2f((uint16_t)(sw >> (16 * (g & 1))));
#pragma unroll
                    for (int r = 0; r < NR; ++r) acc[r] += sc * d[r];
                }
              }
            }
#pragma unroll
            for (int r = 0; r < NR; ++r) pin(acc[r]);
            if constexpr (SPLIT) {
                if ((j + 1) % GP == 0) {
                    if (j + 1 == GP) {
                        next_item();
                        if (stage_next) wait_vmcnt<0>();  // this item's remaining groups have landed
                    }
                    if (stage_next)
                        issue_weights(__builtin_amdgcn_readlane(rec_n, 0) >> 16,
                                      (item + (int)gridDim.x) % ncb, j + 1 == GP, j + 1 - GP, j + 1);
                    // priority 2 once the next item's first part is out (those waves are
                    // nearest their last requests), 0 after the last group
                    if (j + 1 == G)
                        __builtin_amdgcn_s_setprio(0);
                    else
                        __builtin_amdgcn_s_setprio(2);
                }
            }
        }
        if constexpr (ROWA) {
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[r] += alpha_n * (dacc[0][r] + dacc[1][r]);
        }
        // persistent mode, last pass of the item: this wave's tile is free, start the next
        // item's weights (the rest of them, split); its rows follow once every wave is done
        // with the current ones
        if constexpr (PER) {
            if constexpr (!SPLIT) {
                next_item();
                if (stage_next)
                    issue_weights(__builtin_amdgcn_readlane(rec_n, 0) >> 16, (item + (int)gridDim.x) % ncb);
            }
        }
        if constexpr (KS > 1) {
            // K-slices of a tile meet in LDS (a slice's partial goes into its own wave's tile
            // area, free once its MFMAs are done); slice 0 adds them in slice order
            auto slot = [&](int k2) -> f4* {
                return (f4*)((multi || PER) ? red + ((k2 - 1) * TPB + tt) * 1024
                                            : g5lds + (size_t)(k2 * TPB + tt) * S::WAVE_BYTES) +
                       lane;
            };
            if (kh > 0) *slot(kh) = (f4){acc[0], acc[1], acc[2], acc[3]};
            if (PER)
                lds_only_barrier();
            else
                lds_barrier<0>();
            if (kh == 0) {
#pragma unroll
                for (int k2 = 1; k2 < KS; ++k2) {
                    const f4 o = *slot(k2);
#pragma unroll
                    for (int r = 0; r < NR; ++r) acc[r] += o[r];
                }
            }
        }
        if constexpr (PER) {
            if (stage_next) {
                // every wave has read its rows (the K-slice barrier, or this one)
                if constexpr (KS == 1) lds_only_barrier();
                stage_load(0, min(RA, np_next), buf ^ 1, rec_n & 0xFFFF, np_next);
            }
        }
        // lane (n, q) now holds the outputs of activation rows 4q .. 4q+3 (NR = 4) or row q
        // (NR = 1) for weight row n
        if constexpr (EPI == EPI_SWIGLU) {
            // up row n < 8 pairs with gate row n + 8.  NR = 4: lanes n < 8 finish rows 4q, 4q + 1
            // and lanes n + 8 rows 4q + 2, 4q + 3, each taking the other half of its pair by a
            // swap; NR = 1: lanes n < 8 finish row q
            auto finish = [&](float up, float g, int i) {
                up = hround(up);
                g = hround(g);
                g = fminf(g, 7.0f);
                up = fminf(fmaxf(up, -7.0f), 7.0f);
                const float act = hround(g / (1.0f + expf(-g)) * up);
                const int j = (cb * TPB + tt) * 8 + (n & 7);
                uint16_t* dst = a.y + (size_t)pair_of(pb, i) * I + (j & ~15) + perm_pos(j & 15);
                if constexpr (MODE == 1)
                    __hip_atomic_store(dst, f2h(act), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else
                    *dst = f2h(act);
            };
            if constexpr (NR == 1) {
                const float recv = __shfl_xor(acc[0], 8, MJ_WAVE);
                if (kh == 0 && n < 8 && q < npass) finish(acc[0], recv, q);
            } else {
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) {
                    const bool lo = n < 8;
                    const float recv = __shfl_xor(lo ? acc[rr + 2] : acc[rr], 8, MJ_WAVE);
                    const int r = lo ? rr : rr + 2;
                    const int i = 4 * q + r;
                    if (kh == 0 && i < npass) finish(lo ? acc[rr] : recv, lo ? recv : acc[rr + 2], i);
                }
            }
        } else {
            const int col = (cb * TPB + tt) * 16 + n;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int i = NR == 1 ? q : 4 * q + r;
                if (kh == 0 && i < npass && col < a.N) {
                    uint16_t* yp = a.y + (size_t)pair_of(pb, i) * a.N + col;
                    if constexpr (EPI == EPI_ADD) {
                        const uint16_t res = res_pf && pb == 0 ? (uint16_t)resv[r] : *yp;
                        *yp = f2h(h2f(res) + hround(acc[r]));
                    } else {
                        *yp = f2h(acc[r]);
                    }
                }
            }
        }
    };
    // a first pass of at most 4 rows (nearly every expert of a verify pass) takes the
    // one-row-a-lane form; later passes of a bucket with more rows than fit the general one
    if (npass0 <= 4)
        run_pass(std::integral_constant<int, 1>{}, 0, npass0);
    else
        run_pass(std::integral_constant<int, 4>{}, 0, npass0);
    for (int pb = RA; pb < np; pb += RA) {
        __syncthreads();  // the previous pass is done with LDS
        const int npass = min(RA, np - pb);
        stage_load(pb, npass, buf, lpair, np);
        run_pass(std::integral_constant<int, 4>{}, pb, npass);
    }
    if constexpr (!PER) break;
    item += gridDim.x;
    if (!LIST && item / ncb >= 64) break;
    np = __builtin_amdgcn_readlane(rec_n, 1) >> 16;
    if (np <= 0) break;
    e = __builtin_amdgcn_readlane(rec_n, 0) >> 16;
    cb = item % ncb;
    lpair = rec_n & 0xFFFF;
    buf ^= 1;
    early = true;
  }
}

template <int KPL, int GS, int EPI, int WPB, int KS, int REC = REC_NONE, bool ROWA = false>
// four waves per SIMD: two 8-wave blocks per CU
__global__ __launch_bounds__(WPB * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_gather5(
    GatherArgs a, int RA, int multi) {
    FuseIO io;
    __shared__ __align__(16) std::conditional_t<REC == REC_IDS, IdsLds, char> s_ids;
    if constexpr (REC == REC_IDS) io.ids = &s_ids;
    g5_body<KPL, GS, EPI, WPB, KS, REC, ROWA, 0>(a, RA, multi, io);
}

// Fused MoE launch (H = 2048, I = 1024): the up || gate product with its routing, then the down
// product, in the same persistent blocks.  A block that has finished its up items takes down
// items (blocks with fewer up items first, slots in increasing order) and stages an item's act
// rows once every up item of its slot has completed, so the up product's last round overlaps
// the down product, which needs no launch or record read of its own.
// FR: rows the launch ranks at most, 16 or 32 (the 32-row form ranks four rows a wave and
// carries a second rank word, which costs a 9-row pass about 1 us).
template <int GS, bool ROWA, int FR>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_moe_fused(
    GatherArgs up, GatherArgs dn, int ra_up, int ra_dn, int multi_up, int multi_dn) {
    FuseIO io;
    g5_body<8, GS, EPI_SWIGLU, 8, 2, REC_RANK, ROWA, 1, FR>(up, ra_up, multi_up, io);
    __syncthreads();  // every wave is done with the up phase's LDS
    g5_body<4, GS, EPI_STORE, 8, 1, REC_RANK, ROWA, 2, FR>(dn, ra_dn, multi_dn, io);
}

// static LDS of a persistent kernel: its pair lists and what its records are formed from
constexpr size_t g5_stat(int rec, int FR) {
    return 256 + (rec == REC_IDS ? sizeof(IdsLds) : rec == REC_TAB ? 0 : g5_fused_rec_bytes(FR));
}

// dynamic LDS a tile-gather launch may take (the device has 160 KB per workgroup)
constexpr size_t G5_LDS_MAX = 160 * 1024 - 256;

// blocks of a persistent launch: two per CU (the LDS footprint allows two)
static int persistent_blocks() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            cus = 256;
    }
    return 2 * cus;
}

// staged rows per pass: for the persistent products as many as keep two blocks per CU, or one of
// 16 waves (more rows on one expert take extra passes, or slots); dense projections take up to 16
template <int KPL, int GS, int EPI, int WPB, int KS, int REC = REC_NONE, bool ROWA = false>
static int g5_rows(int want) {
    using S = G5Shape<KPL, GS, EPI, WPB, KS, ROWA>;
    constexpr bool PER = REC != REC_NONE;
    int RA = want < S::R ? want : S::R;
    const size_t limit =
        PER ? (WPB == 16 ? 160 : 80) * 1024 - g5_stat(REC, MJ_G5_FUSED_ROWS) : G5_LDS_MAX;
    while (RA > 1 && S::lds(RA, want > RA || PER) > limit) --RA;
    return RA;
}

template <int KPL, int GS, int EPI, int WPB, int KS, int REC = REC_NONE, bool ROWA = false>
static hipError_t launch_g5(const GatherArgs& a, int rows, int slots, hipStream_t st) {
    using S = G5Shape<KPL, GS, EPI, WPB, KS, ROWA>;
    constexpr bool PER = REC != REC_NONE;
    const int ncb = (a.N + 16 * S::TPB - 1) / (16 * S::TPB);
    const int want = rows < 1 ? 1 : rows;
    const int RA = g5_rows<KPL, GS, EPI, WPB, KS, REC, ROWA>(want);
    const bool multi = want > RA;
    int grid = slots * ncb;
    const int most = WPB == 16 ? persistent_blocks() / 2 : persistent_blocks();
    if (PER && grid > most) grid = most;
    launch_timed(k_gather5<KPL, GS, EPI, WPB, KS, REC, ROWA>, dim3(grid), dim3(WPB * 64),
                 S::lds(RA, multi || PER), st, a, RA, (int)multi);
    return hipGetLastError();
}

// Shapes the tile kernel covers: SWIGLU at K = 2048, STORE / ADD at K = 512, 1024 or 2048; N a
// multiple of a tile's 16 rows (of a block's 64 for SWIGLU); group size 64 or 128.
bool gather3_supported(int epi, int K, int N, int gs) {
    if (gs != 64 && gs != 128) return false;
    switch (epi) {
        case EPI_SWIGLU: return K == 2048 && N % 64 == 0;
        case EPI_ADD:
        case EPI_STORE: return (K == 512 || K == 1024 || K == 2048) && N % 16 == 0;
    }
    return false;
}

// The tile kernel fetches codes, scales and biases in 16-byte parts straight into LDS, the general
// kernel a scale at a time.  Arrays that start off a 16-byte line (views into a larger buffer) stay
// with the general kernel in the shapes it is made for: N in steps of 16, and residual products of
// K = 512 or 1024.  (Steps of 64 otherwise are the tile kernel's whatever the arrays' start.)
bool gather3_takes(int epi, int K, int N, int gs, const void* w, const void* s, const void* b) {
    const bool whole = N % 64 == 0 && (epi != EPI_ADD || K == 2048);
    return gather3_supported(epi, K, N, gs) &&
           (whole || (((uintptr_t)w | (uintptr_t)s | (uintptr_t)b) & 15) == 0);
}

// Whether an up || gate product over listed slots takes 16-wave blocks, one a CU, rather than two of
// eight waves: a block then stages 16 rows, not 8, so an expert with 9 to 16 rows is unpacked once
// (the unpacking is what bounds such passes: two thirds of the VALU's time), and each staged row
// serves twice the columns.  Where most experts have fewer rows the barriers over 16 waves only
// cost.  MoE of 64 rows over 64 experts (8 an expert) 64.9 -> 56.5 us, 40 rows (5) 54.8 -> 53.7, 20
// rows over 128 (1.25) 62.8 -> 66.4; 200-token prefill of two layers, 64 experts 604 -> 554, 256
// experts (6) 485 -> 464.
static bool g5_many(int npairs, int experts, int N) {
    return experts > 0 && npairs >= 5 * experts && N % 128 == 0;
}

hipError_t launch_gather3(const GatherArgs& a, int epi, int rows, hipStream_t st) {
    if (!gather3_supported(epi, a.K, a.N, a.gs)) return hipErrorInvalidValue;
    const bool rank = a.rlogits != nullptr, per = rank || a.inds != nullptr || a.tab != nullptr;
    if (a.tab != nullptr) {
        // wide passes: the experts' two products, their slots listed in the table
        const bool al = a.alpha != nullptr;
        const int slots = a.tab_slots;
        if (slots < 1) return hipErrorInvalidValue;
#define MJ_G5T(KPL, E, W, KS)                                                              \
    return a.gs == 64 ? (al ? launch_g5<KPL, 64, E, W, KS, REC_TAB, true>(a, 16, slots, st)   \
                            : launch_g5<KPL, 64, E, W, KS, REC_TAB, false>(a, 16, slots, st)) \
                      : (al ? launch_g5<KPL, 128, E, W, KS, REC_TAB, true>(a, 16, slots, st)  \
                            : launch_g5<KPL, 128, E, W, KS, REC_TAB, false>(a, 16, slots, st));
        if (epi == EPI_SWIGLU && g5_many(a.npairs, a.experts, a.N)) {
            MJ_G5T(8, EPI_SWIGLU, 16, 2)
        }
        if (epi == EPI_SWIGLU) { MJ_G5T(8, EPI_SWIGLU, 8, 2) }
        if (epi != EPI_STORE || a.K > 1024) return hipErrorInvalidValue;
        if (a.K == 512) { MJ_G5T(2, EPI_STORE, 8, 1) }
        MJ_G5T(4, EPI_STORE, 8, 1)
#undef MJ_G5T
    }
    // ranked routing: the up || gate product ranks the router logits itself
    if (rank && (epi != EPI_SWIGLU || a.rM < 1 || a.rM > MJ_G5_FUSED_ROWS || a.rE < 1 ||
                 a.rE > 64 || a.rk < 1 || a.rk > 8 || a.rk > a.rE || a.x_div != a.rk ||
                 a.rinds == nullptr || a.rscores == nullptr))
        return hipErrorInvalidValue;
    if (per && !rank && (a.npairs < 1 || a.npairs > MJ_MAX_PAIRS)) return hipErrorInvalidValue;
    if (!per && epi == EPI_SWIGLU) return hipErrorInvalidValue;
    // slots the launch may have: each a routed expert, or a part of one's pairs
    const int slots = rank ? 64 : a.npairs;
#define MJ_G5(KPL, E, W, KS64, KS128, REC, A)                                               \
    return a.gs == 64 ? launch_g5<KPL, 64, E, W, KS64, REC, A>(a, rows, slots, st)          \
                      : launch_g5<KPL, 128, E, W, KS128, REC, A>(a, rows, slots, st);
    // row-alpha expert weights (scale alpha, bias -alpha in every group of a row): the
    // fold kernels read one alpha per row instead of the group scales and biases
    const bool al = a.alpha != nullptr && per && epi != EPI_ADD;
    if (epi == EPI_SWIGLU) {
        if (rank && al) { MJ_G5(8, EPI_SWIGLU, 8, 2, 2, REC_RANK, true) }
        if (rank) { MJ_G5(8, EPI_SWIGLU, 8, 2, 2, REC_RANK, false) }
        if (g5_many(a.npairs, a.experts, a.N)) {
            if (al) { MJ_G5(8, EPI_SWIGLU, 16, 2, 2, REC_IDS, true) }
            MJ_G5(8, EPI_SWIGLU, 16, 2, 2, REC_IDS, false)
        }
        if (al) { MJ_G5(8, EPI_SWIGLU, 8, 2, 2, REC_IDS, true) }
        MJ_G5(8, EPI_SWIGLU, 8, 2, 2, REC_IDS, false)
    }
    if (per && epi == EPI_STORE && al) {
        if (a.K == 512) { MJ_G5(2, EPI_STORE, 8, 1, 1, REC_IDS, true) }
        if (a.K == 1024) { MJ_G5(4, EPI_STORE, 8, 1, 1, REC_IDS, true) }
        MJ_G5(8, EPI_STORE, 8, 2, 2, REC_IDS, true)
    }
    if (per && epi == EPI_STORE) {
        if (a.K == 512) { MJ_G5(2, EPI_STORE, 8, 1, 1, REC_IDS, false) }
        if (a.K == 1024) { MJ_G5(4, EPI_STORE, 8, 1, 1, REC_IDS, false) }
        MJ_G5(8, EPI_STORE, 8, 2, 2, REC_IDS, false)
    }
    if (per) {
        if (a.K == 512) { MJ_G5(2, EPI_ADD, 8, 1, 1, REC_IDS, false) }
        if (a.K == 1024) { MJ_G5(4, EPI_ADD, 8, 1, 1, REC_IDS, false) }
        MJ_G5(8, EPI_ADD, 8, 2, 2, REC_IDS, false)
    }
#undef MJ_G5
    // dense projections (qkv, o-proj: a few MB at most) spread over many small blocks, four
    // waves of one 16-row tile (group 64) or two (group 128): the unpack work of a block is
    // then short, and the launch fills the chip.  More than 16 rows: one set of blocks per
    // 16-row group, running side by side (each re-reads the small weight matrix) instead of
    // one block unpacking its tile again for every further 16 rows.
    const int groups = (a.dense_rows + 15) / 16;
    rows = rows < 16 ? rows : 16;
    // Past 16 rows at group 128 (two K-slices): 16 staged rows leave LDS for one block a CU, of four
    // waves or of eight; eight: qkv of 64 rows 9.4 -> 6.3 us, of 200 19.6 -> 13.7, o-proj of 200
    // 16.6 -> 11.3.  (Group 64's four slices of a tile fit two blocks.)
    if (a.K == 2048 && a.gs == 128 && a.dense_rows > 16)
        return epi == EPI_ADD ? launch_g5<8, 128, EPI_ADD, 8, 2>(a, rows, groups, st)
                              : launch_g5<8, 128, EPI_STORE, 8, 2>(a, rows, groups, st);
#define MJ_G5D(KPL, E, W, KS64, KS128)                                                    \
    return a.gs == 64 ? launch_g5<KPL, 64, E, W, KS64>(a, rows, groups, st)               \
                      : launch_g5<KPL, 128, E, W, KS128>(a, rows, groups, st);
    if (epi == EPI_ADD) {
        if (a.K == 512) { MJ_G5D(2, EPI_ADD, 8, 1, 1) }
        if (a.K == 1024) { MJ_G5D(4, EPI_ADD, 8, 1, 1) }
        MJ_G5D(8, EPI_ADD, 4, 4, 2)
    }
    if (a.K == 512) { MJ_G5D(2, EPI_STORE, 8, 1, 1) }
    if (a.K == 1024) { MJ_G5D(4, EPI_STORE, 8, 1, 1) }
    MJ_G5D(8, EPI_STORE, 4, 4, 2)
#undef MJ_G5D
}

int gather3_part_rows(int epi, int K, int N, int gs, bool alpha, int npairs, int experts) {
#define MJ_R(KPL, E, W, KS)                                                                  \
    return gs == 64 ? (alpha ? g5_rows<KPL, 64, E, W, KS, REC_TAB, true>(16)                    \
                             : g5_rows<KPL, 64, E, W, KS, REC_TAB, false>(16))                  \
                    : (alpha ? g5_rows<KPL, 128, E, W, KS, REC_TAB, true>(16)                   \
                             : g5_rows<KPL, 128, E, W, KS, REC_TAB, false>(16));
    if (epi == EPI_SWIGLU && g5_many(npairs, experts, N)) { MJ_R(8, EPI_SWIGLU, 16, 2) }
    if (epi == EPI_SWIGLU) { MJ_R(8, EPI_SWIGLU, 8, 2) }
    if (K == 512) { MJ_R(2, EPI_STORE, 8, 1) }
    MJ_R(4, EPI_STORE, 8, 1)
#undef MJ_R
}

// static LDS of the fused MoE kernel: both phases' pair lists and the routing words
constexpr size_t g5_fused_moe_stat(int FR) { return 256 + 256 + g5_fused_rec_bytes(FR); }

// rows staged a pass by the two phases, and the dynamic LDS of the launch (the form for `rows`)
template <int GS>
static size_t moe_fused_lds(int rows, int& ra_up, int& ra_dn) {
    using SU = G5Shape<8, GS, EPI_SWIGLU, 8, 2>;
    using SD = G5Shape<4, GS, EPI_STORE, 8, 1>;
    const int want = rows < 1 ? 1 : rows;
    const size_t limit = 80 * 1024 - g5_fused_moe_stat(want <= 16 ? 16 : 32);  // two blocks a CU
    ra_up = want < 16 ? want : 16;
    ra_dn = ra_up;
    while (ra_up > 1 && SU::lds(ra_up, true) > limit) --ra_up;
    while (ra_dn > 1 && SD::lds(ra_dn, true) > limit) --ra_dn;
    return std::max(SU::lds(ra_up, true), SD::lds(ra_dn, true));
}

// every block of the launch resident at once: two a CU at the largest footprint (32 rows),
// for both forms
template <int GS, bool ROWA>
static bool moe_fused_resident() {
    static int ok = -1;
    if (ok < 0) {
        int ra_up = 0, ra_dn = 0, n16 = 0, n32 = 0;
        const size_t lds16 = moe_fused_lds<GS>(16, ra_up, ra_dn);
        const size_t lds32 = moe_fused_lds<GS>(MJ_MOE_FUSED_ROWS, ra_up, ra_dn);
        ok = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n16, k_moe_fused<GS, ROWA, 16>, 512,
                                                          lds16) == hipSuccess &&
             hipOccupancyMaxActiveBlocksPerMultiprocessor(&n32, k_moe_fused<GS, ROWA, 32>, 512,
                                                          lds32) == hipSuccess &&
             n16 >= 2 && n32 >= 2;
    }
    return ok == 1;
}

template <int GS, bool ROWA>
static hipError_t launch_moe_fused_t(GatherArgs up, GatherArgs dn, int rows, hipStream_t st) {
    using SU = G5Shape<8, GS, EPI_SWIGLU, 8, 2>;
    const int want = rows < 1 ? 1 : rows;
    int ra_up = 0, ra_dn = 0;
    const size_t lds = moe_fused_lds<GS>(rows, ra_up, ra_dn);
    up.fup_ncb = up.N / (16 * SU::TPB);
    dn.fup_ncb = up.fup_ncb;
    if (want <= 16)
        launch_timed(k_moe_fused<GS, ROWA, 16>, dim3(persistent_blocks()), dim3(512), lds, st, up,
                     dn, ra_up, ra_dn, (int)(want > ra_up), (int)(want > ra_dn));
    else
        launch_timed(k_moe_fused<GS, ROWA, 32>, dim3(persistent_blocks()), dim3(512), lds, st, up,
                     dn, ra_up, ra_dn, (int)(want > ra_up), (int)(want > ra_dn));
    return hipGetLastError();
}

bool moe_fused_supported(int H, int I, int E, int gs, int M, bool rowa) {
    if (!(H == 2048 && I == 1024 && E <= 64 && (gs == 64 || gs == 128) && M >= 1 &&
          M <= MJ_MOE_FUSED_ROWS))
        return false;
    if (gs == 64) return rowa ? moe_fused_resident<64, true>() : moe_fused_resident<64, false>();
    return rowa ? moe_fused_resident<128, true>() : moe_fused_resident<128, false>();
}

hipError_t launch_moe_fused(const GatherArgs& up, const GatherArgs& dn, int rows, hipStream_t st) {
    const bool rowa = up.alpha != nullptr;
    if (!moe_fused_supported(up.K, dn.K, up.rE, up.gs, up.rM, rowa) || up.N != 2 * dn.K ||
        dn.N != up.K || up.rlogits == nullptr)
        return hipErrorInvalidValue;
    if (up.gs == 64)
        return rowa ? launch_moe_fused_t<64, true>(up, dn, rows, st)
                    : launch_moe_fused_t<64, false>(up, dn, rows, st);
    return rowa ? launch_moe_fused_t<128, true>(up, dn, rows, st)
                : launch_moe_fused_t<128, false>(up, dn, rows, st);
}

template <int KPL, int GS, int EPI, int WPB, int KS, int REC = REC_NONE, bool ROWA = false>
static hipError_t g5_attr() {
    return hipFuncSetAttribute((const void*)k_gather5<KPL, GS, EPI, WPB, KS, REC, ROWA>,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)std::min(G5Shape<KPL, GS, EPI, WPB, KS, ROWA>::lds(16, true),
                                             G5_LDS_MAX));
}

hipError_t set_gather3_attributes() {
    hipError_t e = hipSuccess;
#define MJ_A(KPL, E, W, KS64, KS128, REC, A)                                  \
    if (e == hipSuccess) e = g5_attr<KPL, 64, E, W, KS64, REC, A>();          \
    if (e == hipSuccess) e = g5_attr<KPL, 128, E, W, KS128, REC, A>();
    MJ_A(8, EPI_ADD, 4, 4, 2, REC_NONE, false)
    MJ_A(2, EPI_ADD, 8, 1, 1, REC_NONE, false)
    MJ_A(4, EPI_ADD, 8, 1, 1, REC_NONE, false)
    MJ_A(2, EPI_STORE, 8, 1, 1, REC_NONE, false)
    MJ_A(4, EPI_STORE, 8, 1, 1, REC_NONE, false)
    MJ_A(8, EPI_STORE, 4, 4, 2, REC_NONE, false)
    // (past 16 rows, group 128 alone)
    if (e == hipSuccess) e = g5_attr<8, 128, EPI_STORE, 8, 2>();
    if (e == hipSuccess) e = g5_attr<8, 128, EPI_ADD, 8, 2>();
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_RANK, false)
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_RANK, true)
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_IDS, false)
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_IDS, true)
    MJ_A(2, EPI_STORE, 8, 1, 1, REC_IDS, false)
    MJ_A(4, EPI_STORE, 8, 1, 1, REC_IDS, false)
    MJ_A(8, EPI_STORE, 8, 2, 2, REC_IDS, false)
    MJ_A(2, EPI_STORE, 8, 1, 1, REC_IDS, true)
    MJ_A(4, EPI_STORE, 8, 1, 1, REC_IDS, true)
    MJ_A(8, EPI_STORE, 8, 2, 2, REC_IDS, true)
    MJ_A(2, EPI_ADD, 8, 1, 1, REC_IDS, false)
    MJ_A(4, EPI_ADD, 8, 1, 1, REC_IDS, false)
    MJ_A(8, EPI_ADD, 8, 2, 2, REC_IDS, false)
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_TAB, false)
    MJ_A(8, EPI_SWIGLU, 8, 2, 2, REC_TAB, true)
    MJ_A(8, EPI_SWIGLU, 16, 2, 2, REC_TAB, false)
    MJ_A(8, EPI_SWIGLU, 16, 2, 2, REC_TAB, true)
    MJ_A(8, EPI_SWIGLU, 16, 2, 2, REC_IDS, false)
    MJ_A(8, EPI_SWIGLU, 16, 2, 2, REC_IDS, true)
    MJ_A(2, EPI_STORE, 8, 1, 1, REC_TAB, false)
    MJ_A(2, EPI_STORE, 8, 1, 1, REC_TAB, true)
    MJ_A(4, EPI_STORE, 8, 1, 1, REC_TAB, false)
    MJ_A(4, EPI_STORE, 8, 1, 1, REC_TAB, true)
#undef MJ_A
    // the fused MoE kernels
    {
        int ra_up = 0, ra_dn = 0;
        size_t most = 0;
        for (int rows : {16, MJ_MOE_FUSED_ROWS})
            most = std::max({most, moe_fused_lds<64>(rows, ra_up, ra_dn),
                             moe_fused_lds<128>(rows, ra_up, ra_dn)});
        const int lds = (int)std::min(most, G5_LDS_MAX);
        const void* ks[] = {(const void*)k_moe_fused<64, false, 16>, (const void*)k_moe_fused<64, true, 16>,
                            (const void*)k_moe_fused<128, false, 16>, (const void*)k_moe_fused<128, true, 16>,
                            (const void*)k_moe_fused<64, false, 32>, (const void*)k_moe_fused<64, true, 32>,
                            (const void*)k_moe_fused<128, false, 32>, (const void*)k_moe_fused<128, true, 32>};
        for (const void* k : ks)
            if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    }
    return e;
}
