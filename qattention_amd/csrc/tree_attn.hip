// tree_attn.hip -- ancestor-sparse tree-verify attention kernels for gfx950.
//
// These kernels compute the same function (the ancestor walk + softmax of
// src/ragged_attn.py:262-497); dispatch_tree picks one:
//
//  * tree_gather_kernel   one row group (D/8 lanes, 16 B per lane) per
//                         (token, q head); the d+1 ancestor rows of a chunk of
//                         steps are gathered from global memory with all loads
//                         issued before the first score is formed.  Handles the
//                         heap walk, the explicit-parent walk and the paged
//                         K/V layout, and merges split-K prefix partial states.
//
//  * tree_group_kernel    the same walk for 2 or 4 q heads of a kv head at
//                         once, or for one with more lanes per query.
//
//  * tree_merge_kernel    merges split-K prefix states and walks, one wave per
//                         (token, q head), for few queries.
//
//  * tree_stream_kernel   heap trees only (subtree_stream.hip).  Persistent
//                         workgroups walk subtree tiles (a band of BFS levels
//                         under G adjacent roots) of each (sequence, kv head),
//                         staging the tile's K/V rows, the few ancestor rows
//                         above it and its Q rows in LDS while the previous
//                         tile is computed, so each K/V row leaves HBM once per
//                         kv head.  All q heads of a GQA group share the rows.
//                         This file holds its tiling plan (make_subtree_plan).
//
// Scores are kept in the log2 domain (scale * log2(e) folded into one multiply)
// and exponentiated with v_exp_f32.  Dot products use v_dot2_f32_{f16,bf16};
// the D/8-lane reduction uses DPP.
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <vector>

#include "qattn_common.h"
#include "qattn_device.h"
#include "tree_walk.h"

namespace qattn {

constexpr int kThreads = 256;

static thread_local char g_err[512];

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

void clear_error() { g_err[0] = 0; }

// The calling thread's walk-export table (qattn_debug_walk), or null.
static thread_local int32_t* g_dbg_walk = nullptr;
// The calling thread's last launch (qattn_debug_last_kernel).
static thread_local const char* g_last_kernel = "";

// ---------------------------------------------------------------------------
// Gather kernel: 4 lanes per (token, q head), 64 pairs per workgroup with the
// head index fastest, so a workgroup reads 2 tokens' contiguous head rows.
// ---------------------------------------------------------------------------
// DBG: the walk-export instantiation (qattn_debug_walk): every query's walk
// steps are also written to p.dbg_walk.
// TPB: threads per workgroup.  A split merge that would occupy under half
// the CUs takes one wave per workgroup instead, so four times the CUs share
// its loads (each CU's vector memory path, not latency, bounds such a launch:
// 4 x 60 nodes x 32 heads over 2048 tokens, D = 64 19.5 -> 19.2 us, 500 nodes x
// 8 heads 14.4 -> 13.8).
template <typename T, int D, int WALK, int LAYOUT, bool LSE, bool PSTATE, bool BATCH, bool DBG = false,
          int TPB = kThreads>
__global__ __launch_bounds__(kThreads) void tree_gather_kernel(TreeParams p) {
    constexpr int NCH = D / 32;
    constexpr int SLOTS = TPB / 4;
    const int j = threadIdx.x & 3;
    // Without split states: XCD-contiguous block order.  The dispatcher
    // places block i on XCD i % 8, so XCD x takes the x-th eighth of the
    // logical blocks and neighbouring tokens, whose ancestors coincide, share
    // one L2 (gen1024 -5.3%, cfg2 and cfg3 through this kernel -2% and -5%
    // in A/B runs on one box; with split states the EAGLE-3 step ran 5.6%
    // slower, so that order stays).
    uint32_t lbk = blockIdx.x;
    if constexpr (!PSTATE) {
        const uint32_t nb = gridDim.x, bx = blockIdx.x, per = nb >> 3, rem = nb & 7, x = bx & 7;
        lbk = x * per + min(x, rem) + (bx >> 3);
    }
    const int64_t slot = (int64_t)lbk * SLOTS + (threadIdx.x >> 2);
    int h, tok, seq;
    slot_coords(p, slot, (int64_t)gridDim.x * SLOTS, h, tok, seq);
    if (seq >= p.B) return;
    int32_t start, n;
    if (!seq_bounds<BATCH>(p, seq, start, n)) return;
    if (tok >= n) return;
    const int64_t qrow = (int64_t)start + tok;
    Vec16 qf[NCH];
    load_q4<D, BATCH>(p, seq, qrow, h, j, qf);
    float m = -INFINITY, l = 0.f, acc[8 * NCH];
    // the first chunk of the walk's K/V loads is in flight while the prefix
    // splits are merged (the walk does not depend on them)
    int32_t* dbg = nullptr;
    if constexpr (DBG) {
        if (j == 0) {
            dbg = p.dbg_walk + (qrow * p.Hq + h) * (p.max_depth + 1);
            for (int i = 0; i <= p.max_depth; ++i) dbg[i] = -1;
        }
    }
    Walk4<T, D, WALK, LAYOUT, 8 / (D / 32), BATCH, DBG> w(p, seq, start, n, tok, h / p.group, j, dbg);
    w.issue();
    if constexpr (PSTATE) {
        load_partial_state4<T, D>(p, qrow, h, j, m, l, acc);
    } else {
#pragma unroll
        for (int e = 0; e < 8 * NCH; ++e) acc[e] = 0.f;
    }
    w.fold(qf, m, l, acc);
    while (w.more()) {
        w.issue();
        w.fold(qf, m, l, acc);
    }
    write_out4<T, D, LSE, BATCH>(p, seq, qrow, h, j, m, l, acc);
}

// ---------------------------------------------------------------------------
// Group kernel: the gather walk of GS (1, 2 or 4) q heads of one kv head at
// once, LPR lanes per (token, head group).  The gather kernel loads every
// ancestor row once per q head, and with grouped heads those loads, not HBM,
// are its bound (512 bytes per step and query at D = 128 against the row's
// 512 / (GS x children) from memory); here a loaded row serves GS queries.
// Few loads in flight per wave and many waves beat the reverse: at D = 128 one
// step per chunk (K and V: 16 VGPRs) against 2 or 4 steps ran 87.5 / 95 / 105
// us on 4 x 4681 nodes b=8 32/8 heads, at D = 64 two steps against 4 and 8 ran
// 64 / 71 / 75 us on 24 ragged trees of up to 1365 nodes 32/8 heads (the
// gather kernel: 116 and 91 us, the subtree kernel: 126 and 112).
//
// GS = 1 is the same walk with more lanes per query than the gather kernel's 4,
// for calls too small to fill the chip with 4.
// ---------------------------------------------------------------------------
constexpr int group_lanes(int head_dim) { return head_dim == 32 ? 4 : 8; }

// DBG: the walk-export instantiation, as for the gather kernel.
// hg: Hq / GS, the head groups of a token; pg: GS-head groups per kv head.
template <typename T, int D, int WALK, int LAYOUT, int GS, int LPR, bool DBG = false>
__global__ __launch_bounds__(kThreads) void tree_group_kernel(TreeParams p, Divider hg, Divider pg) {
    constexpr int NCH = D / (8 * LPR);
    constexpr int SLOTS = kThreads / LPR;
    constexpr int CH = 2 / NCH;  // walk steps per chunk
    const int j = threadIdx.x % LPR;
    const uint32_t nb = gridDim.x, bx = blockIdx.x, per = nb >> 3, rem = nb & 7, x = bx & 7;
    const uint32_t lbk = x * per + min(x, rem) + (bx >> 3);
    const int32_t slot = (int32_t)(lbk * SLOTS + threadIdx.x / LPR);  // (the host keeps the grid's slots below 2^31)
    const int32_t r = divide(slot, hg);
    const int g = slot - r * hg.d, seq = divide(r, p.msdiv), tok = r - seq * p.max_seqlen;
    if (seq >= p.B) return;
    int32_t start, n;
    if (!seq_bounds(p, seq, start, n)) return;
    if (tok >= n) return;
    const int64_t qrow = (int64_t)start + tok;
    const int h0 = g * GS;
    Vec16 qf[GS][NCH];
#pragma unroll
    for (int u = 0; u < GS; ++u) load_q4<D, false, LPR>(p, seq, qrow, h0 + u, j, qf[u]);
    float m[GS], l[GS], acc[GS][8 * NCH];
#pragma unroll
    for (int u = 0; u < GS; ++u) {
        m[u] = -INFINITY;
        l[u] = 0.f;
#pragma unroll
        for (int e = 0; e < 8 * NCH; ++e) acc[u][e] = 0.f;
    }
    int32_t* dbg = nullptr;
    if constexpr (DBG) {
        if (j == 0) {
            dbg = p.dbg_walk + (qrow * p.Hq + h0) * (p.max_depth + 1);
            for (int i = 0; i <= p.max_depth; ++i) dbg[i] = -1;
        }
    }
    Walk4<T, D, WALK, LAYOUT, CH, false, DBG, LPR> w(p, seq, start, n, tok, divide(g, pg), j, dbg);
    do {
        w.issue();
        // (more tokens share a wave than in the gather kernel, so shorter walks wait for longer ones)
        if constexpr (GS > 1 && LAYOUT == KV_PACKED) w.drop_invalid();
#pragma unroll
        for (int u = 0; u < GS; ++u) w.fold_query(qf[u], m[u], l[u], acc[u]);
        w.s0 += CH;
    } while (w.more());
#pragma unroll
    for (int u = 0; u < GS; ++u) {
        if (p.lse)
            write_out4<T, D, true, false, LPR>(p, seq, qrow, h0 + u, j, m[u], l[u], acc[u]);
        else
            write_out4<T, D, false, false, LPR>(p, seq, qrow, h0 + u, j, m[u], l[u], acc[u]);
    }
    if constexpr (DBG) {  // the heads of a group share their walk
        if (j == 0)
            for (int u = 1; u < GS; ++u)
                for (int i = 0; i <= p.max_depth; ++i) dbg[u * (p.max_depth + 1) + i] = dbg[i];
    }
}

// ---------------------------------------------------------------------------
// Split merge and walk of few queries (a decode step of a small tree): one
// wave per (token, q head), D/8 lanes per row, so the wave's 64 * 8 / D lane
// groups each take a share of the split states and of the walk's steps and
// are merged at the end.
// ---------------------------------------------------------------------------
// Latency is its bound: the queries are too few to fill the chip, and a query
// given to 4 lanes runs its 8 states and 8 steps as a chain of round trips.
// Here the states, the parents (in registers, read by readlane) and then all
// K/V rows are one round trip each.  One step of a 60-node depth-7 draft tree
// over 2048 tokens, 32/8 heads, D = 128, 8 splits, both kernels: 4 lanes per
// query (one-wave workgroups) 16.0 us fp16, 19.0 bf16; 8 lanes 15.2; 16 lanes
// 13.7; this 13.2 and 14.2 (13.8 and 14.6 with the V rows of steps without a key
// cleared).
constexpr int kMergeParents = 256;
template <typename T, int D, int WALK, bool BATCH, bool DBG = false>
__global__ __launch_bounds__(kThreads) void tree_merge_kernel(TreeParams p) {
    constexpr int LPR = D / 8, NG = 64 / LPR;
    constexpr bool H = kPartHalf<T>;
    const int lane = threadIdx.x & 63, j = lane % LPR, g = lane / LPR;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int h, tok, seq;
    slot_coords(p, (int64_t)blockIdx.x * (kThreads / 64) + wave, (int64_t)gridDim.x * (kThreads / 64), h, tok, seq);
    if (seq >= p.B) return;
    int32_t start, n;
    if (!seq_bounds<BATCH>(p, seq, start, n)) return;
    if (tok >= n) return;
    const int64_t qrow = (int64_t)start + tok;
    const int kvh = h / p.group;
    // parents 64 i + lane of the sequence
    const bool regs = WALK == WALK_PARENTS && n <= kMergeParents;
    const int32_t pb = parents_base<BATCH>(p, seq, start);
    int32_t pr[kMergeParents / 64] = {};
    if (regs) {
#pragma unroll
        for (int i = 0; i < kMergeParents / 64; ++i)
            if (64 * i + lane < n) pr[i] = p.parents[pb + 64 * i + lane];
    }
    auto next = [&](int32_t cur) {
        if constexpr (WALK == WALK_HEAP) {
            return heap_parent(cur, p.bdiv);
        } else {
            int32_t par;
            if (regs) {
                par = rl(pr[0], cur & 63);
#pragma unroll
                for (int i = 1; i < kMergeParents / 64; ++i)
                    if ((cur >> 6) == i) par = rl(pr[i], cur & 63);
            } else {
                par = __builtin_amdgcn_readfirstlane(p.parents[pb + cur]);
            }
            return (par >= 0 && par < n) ? par : cur;
        }
    };
    const Vec16 qf = ld16((const uint16_t*)p.q + qrow * p.sq_t + (BATCH ? (int64_t)seq * p.sq_b : 0) +
                          (int64_t)h * p.sq_h + 8 * j);
    int32_t* dbg = nullptr;
    if constexpr (DBG) {
        if (j == 0) {
            dbg = p.dbg_walk + (qrow * p.Hq + h) * (p.max_depth + 1);
            for (int t = g; t <= p.max_depth; t += NG) dbg[t] = -1;
        }
    }
    // ---- this group's split states (numerator / l as stored), two in flight ----
    float m = -INFINITY, l = 0.f, acc[8] = {};
    const int64_t plane = p.total_tokens * (int64_t)p.Hq, idx = qrow * p.Hq + h;
    struct State {
        float m, l;
        Vec16 a[H ? 1 : 2];
    };
    auto load_state = [&](int s) {
        State x{};
        x.m = -INFINITY;
        if (s < p.n_split) {
            const int64_t k = s * plane + idx;
            x.m = p.part_m[k];
            x.l = p.part_l[k];
            if constexpr (H) {
                x.a[0] = ld16((const uint16_t*)p.part_acc + k * D + 8 * j);
            } else {
                x.a[0] = ld16((const float*)p.part_acc + k * D + 8 * j);
                x.a[1] = ld16((const float*)p.part_acc + k * D + 8 * j + 4);
            }
        }
        return x;
    };
    auto fold_state = [&](const State& x) {
        // (a split of nothing but NaN scores has m = -inf and l = NaN: its
        // weight 0 * l carries the NaN on)
        const float mb = fmaxf(m, x.m);
        const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - mb);
        const float w = (x.m == -INFINITY ? 0.f : fast_exp2(x.m - mb)) * x.l;
        l = l * alpha + w;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float v;
            if constexpr (H)
                v = elem<F16>(x.a[0], e);
            else
                v = __builtin_bit_cast(float, x.a[e >> 2].w[e & 3]);
            acc[e] = __builtin_fmaf(w, v, acc[e] * alpha);
        }
        m = mb;
    };
    State st0 = load_state(g), st1 = load_state(NG + g);
    // ---- the walk: steps t0 + g and t0 + NG + g of each 2 NG are this group's ----
    const int64_t kvb = kv_base(p, seq, start);
    const uint16_t* kb = (const uint16_t*)p.k + (int64_t)kvh * p.sk_h + 8 * j;
    const uint16_t* vb = (const uint16_t*)p.v + (int64_t)kvh * p.sv_h + 8 * j;
    int32_t cur = tok, prev = -1;
    for (int t0 = 0; t0 <= p.max_depth && cur != prev; t0 += 2 * NG) {
        int32_t node[2] = {tok, tok};  // (a step without a key reads the query's own row, score -inf)
        bool ok[2] = {false, false};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            for (int i = 0; i < NG && t0 + u * NG + i <= p.max_depth && cur != prev; ++i) {
                if (i == g) {
                    node[u] = cur;
                    ok[u] = true;
                }
                prev = cur;
                cur = next(cur);
            }
        }
        Vec16 kf[2], vf[2][1];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            kf[u] = ld16(kb + (kvb + node[u]) * p.sk_t);
            vf[u][0] = ld16(vb + (kvb + node[u]) * p.sv_t);
            if constexpr (DBG) {
                if (j == 0 && ok[u]) dbg[t0 + u * NG + g] = node[u];
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // every row is requested before the first wait
        if (t0 == 0) {
            fold_state(st0);
            fold_state(st1);
        }
        float sc[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float d = qk4<T, 1, LPR>(&qf, &kf[u]) * p.scale_log2;
            sc[u] = ok[u] ? d : -INFINITY;
        }
        // fold_scores without its early return (under a branch the compiler
        // sinks the V loads behind the scores, one more round trip); a lane
        // group without a step adds zeros
        const float m_new = __builtin_elementwise_maximum(m, __builtin_elementwise_maximum(sc[0], sc[1]));
        const float ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = fast_exp2(m - ref);
        float p0 = fast_exp2(sc[0] - ref), p1 = fast_exp2(sc[1] - ref);
        l = __builtin_fmaf(l, alpha, p0 + p1);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            // (weight 0 times an infinity in the own row would be NaN; the
            // empty statement keeps these first uses of V behind the scores)
            uint32_t(&w)[4] = vf[u][0].w;
            asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(u ? p1 : p0));
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = ok[u] ? w[e] : 0u;
        }
        axpy8<T>(acc, p0, vf[0][0]);
        axpy8<T>(acc, p1, vf[1][0]);
        m = m_new;
    }
    for (int s = 2 * NG + g; s < p.n_split; s += NG) fold_state(load_state(s));
    // ---- merge the groups ----
#pragma unroll
    for (int off = LPR; off < 64; off *= 2) {
        const float mo = __shfl_xor(m, off), lo = __shfl_xor(l, off);
        const float mb = fmaxf(m, mo);
        const float a = m == -INFINITY ? 0.f : fast_exp2(m - mb), b = mo == -INFINITY ? 0.f : fast_exp2(mo - mb);
        l = l * a + lo * b;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = acc[e] * a + __shfl_xor(acc[e], off) * b;
        m = mb;
    }
    if (g == 0) {
        if (p.lse)
            write_out4<T, D, true, BATCH, LPR>(p, seq, qrow, h, j, m, l, acc);
        else
            write_out4<T, D, false, BATCH, LPR>(p, seq, qrow, h, j, m, l, acc);
    }
}

// ---------------------------------------------------------------------------
// Ancestor table kernel (debug export of the walk)
// ---------------------------------------------------------------------------
template <int WALK>
__global__ __launch_bounds__(kThreads) void ancestors_kernel(TreeParams p, int32_t* out) {
    const int64_t idx = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int seq = (int)(idx / p.max_seqlen);
    const int tok = (int)(idx % p.max_seqlen);
    if (seq >= p.B) return;
    int32_t start, n;
    if (!seq_bounds(p, seq, start, n)) return;
    if (tok >= n) return;
    int32_t* row = out + ((int64_t)start + tok) * (p.max_depth + 1);
    const int32_t pb = parents_base(p, seq, start);
    int32_t cur = tok, prev = -1;
    for (int s = 0; s <= p.max_depth; ++s) {
        row[s] = (cur != prev) ? cur : -1;
        prev = cur;
        cur = walk_next<WALK>(p, pb, n, cur);
    }
}

// ---------------------------------------------------------------------------
// LSE merge kernel
// ---------------------------------------------------------------------------
struct MergeParams {
    const float* lse_p;
    const float* lse_t;
    const void* o_p;
    const void* o_t;
    void* out;
    int64_t sl_p[3], sl_t[3], so_p[4], so_t[4], so[4];
    int32_t B, H, Nq;
};

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void lse_merge_kernel(MergeParams mp) {
    constexpr int LPR = D / 8;
    constexpr int SLOTS = kThreads / LPR;
    const int lane = threadIdx.x % LPR;
    const int64_t pos = (int64_t)blockIdx.x * SLOTS + threadIdx.x / LPR;
    if (pos >= (int64_t)mp.B * mp.H * mp.Nq) return;
    const int i = (int)(pos % mp.Nq);
    const int h = (int)((pos / mp.Nq) % mp.H);
    const int bb = (int)(pos / ((int64_t)mp.Nq * mp.H));
    const float lp = mp.lse_p[bb * mp.sl_p[0] + h * mp.sl_p[1] + i * mp.sl_p[2]];
    const float lt = mp.lse_t[bb * mp.sl_t[0] + h * mp.sl_t[1] + i * mp.sl_t[2]];
    const float mx = fmaxf(lp, lt);
    const float wp = fast_exp2((lp - mx) * kLog2e);
    const float wt = fast_exp2((lt - mx) * kLog2e);
    const float ws = fmaxf(wp + wt, 1e-8f);
    const Vec16 a = ld16((const uint16_t*)mp.o_p + bb * mp.so_p[0] + h * mp.so_p[1] + i * mp.so_p[2] + lane * 8);
    const Vec16 c = ld16((const uint16_t*)mp.o_t + bb * mp.so_t[0] + h * mp.so_t[1] + i * mp.so_t[2] + lane * 8);
    float r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = (wp * elem<T>(a, j) + wt * elem<T>(c, j)) / ws;
    st16((uint16_t*)mp.out + bb * mp.so[0] + h * mp.so[1] + i * mp.so[2] + lane * 8, pack8<T>(r));
}

// ---------------------------------------------------------------------------
// Host side: validation, planning, dispatch
// ---------------------------------------------------------------------------
bool row_aligned(const void* ptr, const int64_t* st, int n_outer) {
    if (((uintptr_t)ptr & 15u) != 0) return false;
    for (int i = 0; i < n_outer; ++i)
        if (st[i] % 8 != 0) return false;
    return st[n_outer] == 1;
}

int check_common(int32_t dtype, int32_t head_dim, int32_t batch, int32_t max_seqlen,
                        int64_t total_tokens, int32_t hq, int32_t hkv, int32_t max_depth) {
    if (dtype != QATTN_DTYPE_F16 && dtype != QATTN_DTYPE_BF16) {
        set_error("dtype %d is not fp16 (0) or bf16 (1)", dtype);
        return QATTN_ERR_DTYPE;
    }
    if (head_dim != 32 && head_dim != 64 && head_dim != 128) {
        set_error("head_dim %d not in {32, 64, 128}", head_dim);
        return QATTN_ERR_HEAD_DIM;
    }
    if (batch < 0 || max_seqlen < 0 || total_tokens < 0 || hq < 1 || hkv < 1 || hq % hkv != 0 ||
        max_depth < 0) {
        set_error("bad sizes: batch=%d max_seqlen=%d total_tokens=%lld hq=%d hkv=%d max_depth=%d", batch,
                  max_seqlen, (long long)total_tokens, hq, hkv, max_depth);
        return QATTN_ERR_ARG;
    }
    if (total_tokens >= (int64_t(1) << 31) || (int64_t)max_seqlen * batch >= (int64_t(1) << 40)) {
        set_error("sizes too large: total_tokens=%lld", (long long)total_tokens);
        return QATTN_ERR_ARG;
    }
    return QATTN_OK;
}

int launch_status(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return QATTN_ERR_HIP;
    }
    g_last_kernel = what;
    return QATTN_OK;
}

// Subtree tiling plan for a heap tree of n nodes.  Level l of the heap holds
// b^l nodes; a band of levels [lo, hi) is cut into tiles of G roots at level
// lo whose subtrees (down to hi) plus one ancestor row per level above lo fit
// the LDS budget.  Bands are chosen bottom-up, each the tallest that fits a
// single-root subtree.  Returns false when no plan fits the LDS budget.
static bool make_subtree_plan(int b, int64_t n, int max_depth, int rcap, int ncap, SubtreePlan& plan) {
    plan = SubtreePlan{};
    for (int i = 0; i < kMaxBands; ++i) plan.tile_base[i] = INT32_MAX;
    if (n <= 0 || b < 1) return false;
    {
        int64_t st = 0, pw = 1;
        for (int l = 0; l < 64; ++l) {
            plan.lvl_start[l] = (int32_t)std::min<int64_t>(st, INT32_MAX);
            plan.lvl_pow[l] = (uint32_t)std::min<int64_t>(pw, UINT32_MAX);
            if (st < INT32_MAX) st += pw;
            if (pw < UINT32_MAX && b > 1) pw = std::min<int64_t>(pw * b, UINT32_MAX);
        }
    }
    if (b == 1) {
        const int extra = (int)std::min<int64_t>(max_depth, n - 1);
        int h = std::min(rcap - extra, ncap);
        h = std::min(h, 64 - extra);
        if (h < 1) return false;
        h = (int)std::min<int64_t>(h, n);
        plan.nbands = 1;
        plan.chain_h = h;
        plan.tile_base[0] = 0;
        plan.band[0] = 1u << 16;  // lo, hi come from chain_h for b == 1
        const int64_t tiles = (n + h - 1) / h;
        if (tiles >= (int64_t(1) << 30)) return false;
        plan.total_tiles = (int32_t)tiles;
        plan.max_rows = h + extra;
        return true;
    }
    // level starts s[l] and full widths w[l]
    std::vector<int64_t> s, w;
    int64_t sl = 0, wl = 1;
    while (sl < n) {
        s.push_back(sl);
        w.push_back(wl);
        sl += wl;
        if (wl > n) wl = n + 1; else wl *= b;
    }
    const int Lmax = (int)s.size() - 1;
    auto width = [&](int l) -> int64_t { return std::min<int64_t>(w[l], n - s[l]); };
    auto subtree = [&](int h) -> int64_t {  // nodes of one complete root subtree, h levels
        int64_t tot = 0, bj = 1;
        for (int j = 0; j < h; ++j) {
            tot += bj;
            if (tot > rcap) return int64_t(rcap) + 1;
            bj *= b;
        }
        return tot;
    };
    auto extra_rows = [&](int64_t G, int lo) -> int64_t {  // ancestors above G adjacent roots
        int64_t tot = 0, bj = 1;
        const int J = std::min(lo, max_depth);
        for (int j = 1; j <= J; ++j) {
            if (bj <= n) bj *= b;
            const int64_t span = (G - 1 + bj - 1) / bj + 1;
            tot += std::min<int64_t>(span, width(lo - j));
        }
        return tot;
    };
    std::vector<Band> bands;
    int hi = Lmax;
    while (hi >= 0) {
        int best = 0;
        for (int h = 1; h <= hi + 1; ++h) {
            const int lo = hi - h + 1;
            const int nlev = hi - std::max(0, lo - max_depth) + 1;
            if (subtree(h) + extra_rows(1, lo) > rcap || subtree(h) > ncap || nlev > 64) break;
            best = h;
        }
        if (best == 0) return false;
        const int lo = hi - best + 1;
        const int64_t size = subtree(best);
        const int64_t wlo = width(lo);
        int64_t G = 1;
        while (G < wlo && (G + 1) * size + extra_rows(G + 1, lo) <= rcap && (G + 1) * size <= ncap) ++G;
        bands.push_back(Band{lo, hi, (int32_t)G, 0});
        if ((int)bands.size() > kMaxBands) return false;
        hi = lo - 1;
    }
    std::reverse(bands.begin(), bands.end());  // top band first
    int64_t tiles = 0, rows = 0;
    for (size_t i = 0; i < bands.size(); ++i) {
        Band& bd = bands[i];
        bd.tile_base = (int32_t)tiles;
        const int64_t wlo = width(bd.lo);
        tiles += (wlo + bd.G - 1) / bd.G;
        rows = std::max<int64_t>(rows, bd.G * subtree(bd.hi - bd.lo + 1) + extra_rows(bd.G, bd.lo));
        if (bd.hi > 255 || bd.G > 65535) return false;
        plan.tile_base[i] = bd.tile_base;
        plan.band[i] = (uint32_t)bd.lo | ((uint32_t)bd.hi << 8) | ((uint32_t)bd.G << 16);
    }
    if (tiles >= (int64_t(1) << 30)) return false;
    plan.nbands = (int32_t)bands.size();
    plan.total_tiles = (int32_t)tiles;
    plan.max_rows = (int32_t)rows;
    plan.chain_h = 0;
    return rows <= rcap;
}

// Queries up to which a split merge takes one wave each (tree_merge_kernel).
// The fewer bytes a state and a row hold, the sooner a whole wave per query
// costs more issue slots than the shorter chain of loads saves; and one small
// tree finds its states in the L2 that wrote them.  Whole steps over 2048
// tokens, us, gather / merge kernel, fp16 unless noted:
//  D = 128: one tree of 16-250 nodes x 32 heads 1.2-1.3 times as fast (128 nodes
//    20.0 / 16.1, 250 29.5 / 25.0); 500 x 8 heads 19.6 / 18.5, 2 x 60 x 32 20.5 /
//    20.4, 4 x 60 x 32 28.0 / 28.8, 1000 x 8 29.4 / 30.1
//  D = 64: one tree of 128 x 32 13.9 / 12.5, 250 x 32 19.8 / 18.7, bf16 24.1 /
//    19.9; 300 x 8 12.6 / 12.1, 2 x 60 x 32 13.8 / 14.6, 4 x 60 x 32 19.2 / 22.6
//  D = 32: 1024 queries 9.2 / 9.2, 2400 10.6 / 11.1, 8000 13.2 / 16.5; bf16 3072
//    12.0 / 11.2, 4000 12.3 / 13.1
template <typename T, int D>
static int64_t merge_limit(const TreeParams& p) {
    if (D == 32) return kPartHalf<T> ? 1024 : 3072;
    if (p.B == 1 && p.max_seqlen <= kMergeParents) return 8192;
    return D == 64 ? 3072 : 6144;
}

template <typename T, int D, int WALK, int LAYOUT, bool LSE, bool PSTATE, bool BATCH = false, bool DBG = false>
static int launch_gather(const TreeParams& p, hipStream_t st) {
    constexpr int SLOTS = kThreads / 4;  // 4 lanes per (token, q head)
    const int64_t slots = (int64_t)p.B * p.max_seqlen * p.Hq;
    const int64_t blocks = (slots + SLOTS - 1) / SLOTS;
    if (blocks >= (int64_t(1) << 31)) {
        set_error("grid too large (%lld blocks)", (long long)blocks);
        return QATTN_ERR_ARG;
    }
    if constexpr (PSTATE && LAYOUT == KV_PACKED) {
        if (slots <= merge_limit<T, D>(p)) {
            constexpr int WAVES = kThreads / 64;
            hipLaunchKernelGGL((tree_merge_kernel<T, D, WALK, BATCH, DBG>),
                               dim3((unsigned)((slots + WAVES - 1) / WAVES)), dim3(kThreads), 0, st, p);
            return launch_status("tree_merge_kernel");
        }
        if (blocks < 128) {
            constexpr int S1 = 64 / 4;
            hipLaunchKernelGGL((tree_gather_kernel<T, D, WALK, LAYOUT, LSE, PSTATE, BATCH, DBG, 64>),
                               dim3((unsigned)((slots + S1 - 1) / S1)), dim3(64), 0, st, p);
            return launch_status("tree_gather_kernel");
        }
    }
    hipLaunchKernelGGL((tree_gather_kernel<T, D, WALK, LAYOUT, LSE, PSTATE, BATCH, DBG>), dim3((unsigned)blocks),
                       dim3(kThreads), 0, st, p);
    return launch_status("tree_gather_kernel");
}

template <typename T, int D, int WALK, bool BATCH>
static int gather_packed(const TreeParams& p, bool lse, bool pstate, hipStream_t st) {
    if (pstate) {
        return lse ? launch_gather<T, D, WALK, KV_PACKED, true, true, BATCH>(p, st)
                   : launch_gather<T, D, WALK, KV_PACKED, false, true, BATCH>(p, st);
    }
    return lse ? launch_gather<T, D, WALK, KV_PACKED, true, false, BATCH>(p, st)
               : launch_gather<T, D, WALK, KV_PACKED, false, false, BATCH>(p, st);
}

// Walk export (qattn_debug_walk): the walk-export instantiation of the gather
// kernel that serves the same call (dtype, LSE, walk, layout, prefix state).
template <typename T, int D, bool LSE>
static int gather_dbg(const TreeParams& p, int walk, int layout, bool pstate, hipStream_t st) {
    if (layout == KV_PAGED) return launch_gather<T, D, WALK_HEAP, KV_PAGED, LSE, false, false, true>(p, st);
    if (walk == WALK_HEAP)
        return pstate ? launch_gather<T, D, WALK_HEAP, KV_PACKED, LSE, true, false, true>(p, st)
                      : launch_gather<T, D, WALK_HEAP, KV_PACKED, LSE, false, false, true>(p, st);
    return pstate ? launch_gather<T, D, WALK_PARENTS, KV_PACKED, LSE, true, false, true>(p, st)
                  : launch_gather<T, D, WALK_PARENTS, KV_PACKED, LSE, false, false, true>(p, st);
}

template <typename T, int D, int WALK, int LAYOUT, int GS, int LPR>
static int launch_group_gs(const TreeParams& p, hipStream_t st) {
    constexpr int SLOTS = kThreads / LPR;
    const int64_t blocks = ((int64_t)p.B * p.max_seqlen * (p.Hq / GS) + SLOTS - 1) / SLOTS;
    const Divider hg = make_divider(p.Hq / GS), pg = make_divider(p.group / GS);
    if (p.dbg_walk)
        hipLaunchKernelGGL((tree_group_kernel<T, D, WALK, LAYOUT, GS, LPR, true>), dim3((unsigned)blocks),
                           dim3(kThreads), 0, st, p, hg, pg);
    else
        hipLaunchKernelGGL((tree_group_kernel<T, D, WALK, LAYOUT, GS, LPR>), dim3((unsigned)blocks), dim3(kThreads), 0,
                           st, p, hg, pg);
    return launch_status(GS > 1 ? (GS == 4 ? "tree_group_kernel, 4 heads" : "tree_group_kernel, 2 heads")
                                : (LPR == 16 ? "tree_group_kernel, 16 lanes" : "tree_group_kernel, 8 lanes"));
}

// q heads per slot and lanes per row of the group kernel for a call; gs 0: the
// gather kernel.
struct GroupPlan {
    int gs, lanes;
};

// Slots of 2 or 4 heads must fill the chip: fewer, longer-running waves lose to
// the gather kernel's one query per slot below about 8 waves per CU for GS = 4
// and 16 for GS = 2 (500-node trees b=3, 32/8 heads, D = 128: 1500 waves 13.9
// against 12.1 us, 2000 15.8 against 17.2, 8000 41.8 against 49.3; D = 64: 2000
// waves equal, 3000 12.2 against 13.9; 16/8 heads: 3000 13.5 against 13.0, 4000
// 16.0 against 17.4), and at D = 128, where a round is one step, four times that
// for walks of more than 32 steps (64 steps, 32/8 heads: 4000 waves 136 against
// 125 us, 8000 equal; 16/8 heads 8000 136 against 124; 32 steps no slower from
// 2000).  At the other end the gather kernel's 4 lanes per query
// leave the chip idle.  One 16-byte chunk per lane at D = 128 (16 lanes): 64 to
// 4096 queries b=2 1.25 times as fast, 8192 with explicit parents 4.5 against
// 5.7 us, paged 4.7 against 5.0; ungrouped heads 12288 5.5 against 6.4, b=8 3.9
// against 4.1, but 14400 b=8 5.0 against 4.8 and paged 9600 5.4 against 5.1.
// 8 lanes ran one 672-node b=28 tree (3 steps) in 7.5 against 8.8 us, three
// of them in 16.8 against 17.9, but 1000 nodes b=3 (7 steps) in 12.8 against
// 12.5.  At D = 64 (8 lanes) a round of loads covers 2 steps against 4, so it
// pays where it takes less than twice the rounds (5 steps 3.37 against 3.62
// us, paged 4.00 against 4.14; 4 steps 3.02 against 2.91, paged 3.44 against
// 3.13; 8 steps 3.97 against 3.72) and for the dependent loads of explicit
// parents (7 steps 3.95 against 4.09), up to 8192 queries (12288: 4.6 against
// 4.3).  Packed layouts (cu) without split states only.  steps: walk steps
// per query, at most.
static GroupPlan group_plan(const TreeParams& p, int head_dim, int walk, int layout, int steps, bool pstate) {
    const int64_t queries = (int64_t)p.B * p.max_seqlen * p.Hq;
    if (!p.cu || pstate || queries >= (int64_t(1) << 31)) return {0, 0};
    if (p.group % 2 == 0) {
        const int gs = p.group % 4 == 0 ? 4 : 2, lanes = group_lanes(head_dim);
        const int64_t waves = queries / gs * lanes / 64, need = 8192 / gs;
        if (waves >= (head_dim == 128 && steps > 32 ? 4 * need : need)) return {gs, lanes};
    }
    if (head_dim == 32) return {0, 0};
    if (head_dim == 64 && queries <= 8192) {
        // 8 lanes load 2 steps per round, the gather kernel's 4 lanes 4
        const bool rounds = steps % 4 == 1 || steps % 4 == 2;
        return rounds || (walk == WALK_PARENTS && steps > 4) ? GroupPlan{1, 8} : GroupPlan{0, 0};
    }
    if (head_dim == 128 && queries <= (p.group == 1 && layout != KV_PAGED ? 12288 : 8192)) return {1, 16};
    if (head_dim == 128 && p.group == 1 && queries <= 65536 && steps <= 4) return {1, 8};
    return {0, 0};
}

// Mean walk steps per node of a b-ary heap of n nodes.
static double heap_steps(int b, int64_t n, int max_depth) {
    double steps = 0;
    int64_t first = 0, width = 1;
    for (int level = 0; first < n; ++level) {
        steps += (double)std::min(width, n - first) * (std::min(level, max_depth) + 1);
        if (b == 1 && level >= max_depth) return (steps + (double)(n - first - 1) * (max_depth + 1)) / (double)n;
        first += width;
        width = std::min(width * b, n);
    }
    return steps / (double)n;
}

// Whether the subtree kernel is the faster one for a heap walk without split
// states, from two estimates in us.  A walk costs the bytes its lanes load
// (each query's Q, O and each slot's K/V row per step) at the rate the
// vector memory path was seen to reach: 7.2 TB/s for the group kernel, 12.5
// plus 4 us for the gather kernel.  The subtree kernel costs 5 us plus the
// larger of its compulsory bytes at 5 TB/s and its rounds of tiles (768
// workgroups), each 2 us plus 0.07 us per 256 bytes of query rows.  Measured /
// estimated, subtree against walk: b=4 d=5 x 4, 32 heads 40 / 41 against 48 / 52
// us; 672 nodes b=28, 32 heads 10.7 / 9.4 against 8.0 / 7.4; 1023 nodes b=2 x 8,
// 32/8 heads 47 / 54 against 57 / 59; 4681 nodes b=8 x 4, 32/8 heads 126 / 115
// against 88 / 94; 100 nodes b=4 x 32, 32/8 heads 40 / 33 against 20 / 15.  A
// gather walk must be clearly cheaper (its rate varies more with the tree).
static bool subtree_pays(const TreeParams& p, const SubtreePlan& plan, int head_dim, bool paged, int gs) {
    const double nodes = (double)p.B * p.max_seqlen, row = 2.0 * head_dim;
    const double steps = heap_steps(p.bdiv.d, p.max_seqlen, p.max_depth);
    double walk = nodes * (p.Hq / std::max(gs, 1)) * 2 * row * (std::max(gs, 1) + steps) * 1e-6;
    walk = gs > 1 ? walk / 7.2 : 4 + walk / 12.5;
    if (paged) walk *= 1.15;  // (a page-table round trip per chunk)
    const double rounds = (double)p.B * p.Hkv * plan.total_tiles / 768;
    const double qrows = (double)p.max_seqlen * p.group / plan.total_tiles;
    const double hbm = nodes * 2 * row * (p.Hq + p.Hkv) * 1e-6 / 5.0;
    const double sub = 5 + std::max(rounds * (2 + 0.07 * qrows * row / 256), hbm);
    return gs > 1 ? sub < walk : 0.85 * sub < walk;
}

template <typename T, int D, int GS, int LPR>
static int launch_group_walk(const TreeParams& p, int walk, int layout, hipStream_t st) {
    if (layout == KV_PAGED) return launch_group_gs<T, D, WALK_HEAP, KV_PAGED, GS, LPR>(p, st);
    return walk == WALK_HEAP ? launch_group_gs<T, D, WALK_HEAP, KV_PACKED, GS, LPR>(p, st)
                             : launch_group_gs<T, D, WALK_PARENTS, KV_PACKED, GS, LPR>(p, st);
}

template <typename T, int D>
static int launch_group(const TreeParams& p, const GroupPlan& gp, int walk, int layout, hipStream_t st) {
    if (gp.gs == 4) return launch_group_walk<T, D, 4, group_lanes(D)>(p, walk, layout, st);
    if (gp.gs == 2) return launch_group_walk<T, D, 2, group_lanes(D)>(p, walk, layout, st);
    if constexpr (D == 128) {
        if (gp.lanes == 16) return launch_group_walk<T, D, 1, 16>(p, walk, layout, st);
    }
    if constexpr (D > 32) return launch_group_walk<T, D, 1, 8>(p, walk, layout, st);
    set_error("no group kernel for head_dim %d with %d heads per slot", D, gp.gs);  // (not for group_plan's answers)
    return QATTN_ERR_ARG;
}

template <typename T, int D>
static int dispatch_tree(const TreeParams& p, int walk, int layout, bool lse, bool pstate, int algo,
                         hipStream_t st) {
    // walk steps of a query, at most (a heap of b >= 2: no more than its levels)
    int steps = p.max_depth < 64 ? p.max_depth + 1 : 64;
    if (walk == WALK_HEAP && p.bdiv.d > 1) {
        int levels = 0;
        for (int64_t first = 0, width = 1; first < p.max_seqlen; first += width, width *= p.bdiv.d) ++levels;
        steps = std::min(steps, levels);
    }
    const bool paged = layout == KV_PAGED;
    if (walk == WALK_HEAP && (!paged || !pstate) && algo != QATTN_ALGO_GATHER) {
        SubtreePlan plan;
        int rcap = 0, qcap = 0;
        stream_tile_caps(D, &rcap, &qcap);
        // (paged: the page table is copied to LDS, so it has a size limit, and
        // one 32-bit offset addresses K and V: equal strides below 2^31)
        const bool paged_ok = !paged || ((int64_t)p.B * p.pt_cols <= stream_max_page_entries() &&
                                         p.sk_page == p.sv_page && p.sk_t == p.sv_t && p.sk_h == p.sv_h &&
                                         p.sk_page >= 0 && p.sk_page < (int64_t(1) << 31) && p.sk_t >= 0 &&
                                         p.sk_t < (int64_t(1) << 31) && p.page_size <= 4096 &&
                                         (p.max_seqlen - 1) / p.page_size < (1 << 19));
        const bool ok = p.B <= stream_max_batch() && paged_ok &&
                        make_subtree_plan(p.bdiv.d, p.max_seqlen, p.max_depth, rcap, qcap / p.group, plan);
        const int64_t wgs = ok ? (int64_t)p.B * p.Hkv * plan.total_tiles : 0;
        // The subtree kernel needs enough tiles to fill 256 CUs; a merged
        // prefix state makes each query heavier, so it only pays off there
        // when tiles are plentiful.  Without one, the cheaper estimate wins
        // (uniform batches have no group kernel and keep the tile rule).
        const bool use = ok && (algo == QATTN_ALGO_SUBTREE ||
                                (wgs >= (pstate ? 2048 : 512) &&
                                 (pstate || !p.cu || subtree_pays(p, plan, D, paged, group_plan(p, D, walk, layout, steps, false).gs))));
        if (algo == QATTN_ALGO_SUBTREE && !ok) {
            if (!paged_ok)
                set_error("paged subtree kernel: page-table entries %lld (at most %d), page size %d (at most "
                          "4096), or K/V cache strides that differ or reach 2^31",
                          (long long)p.B * p.pt_cols, stream_max_page_entries(), p.page_size);
            else
                set_error("no subtree plan fits (b=%d, max_seqlen=%d, max_depth=%d, batch=%d)", p.bdiv.d,
                          p.max_seqlen, p.max_depth, p.B);
            return QATTN_ERR_ARG;
        }
        if (use) return launch_stream(p, plan, T::kCode, D, pstate, paged, st);
    } else if (algo == QATTN_ALGO_SUBTREE) {
        set_error("the subtree kernel supports the heap walk on packed or paged K/V only");
        return QATTN_ERR_ARG;
    }
    const GroupPlan gp = group_plan(p, D, walk, layout, steps, pstate);
    if (gp.gs) return launch_group<T, D>(p, gp, walk, layout, st);
    if (p.dbg_walk) {
        // walk export: calls over packed cu_seqlens, either dtype, with or without LSE
        if (!p.cu) {
            set_error("the walk export runs calls over packed cu_seqlens");
            return QATTN_ERR_ARG;
        }
        return lse ? gather_dbg<T, D, true>(p, walk, layout, pstate, st)
                   : gather_dbg<T, D, false>(p, walk, layout, pstate, st);
    }
    if (layout == KV_PACKED) {
        // (a null cu is a uniform batch: its addressing is compiled separately)
        if (!p.cu) {
            return walk == WALK_HEAP ? gather_packed<T, D, WALK_HEAP, true>(p, lse, pstate, st)
                                     : gather_packed<T, D, WALK_PARENTS, true>(p, lse, pstate, st);
        }
        return walk == WALK_HEAP ? gather_packed<T, D, WALK_HEAP, false>(p, lse, pstate, st)
                                 : gather_packed<T, D, WALK_PARENTS, false>(p, lse, pstate, st);
    }
    return lse ? launch_gather<T, D, WALK_HEAP, KV_PAGED, true, false>(p, st)
               : launch_gather<T, D, WALK_HEAP, KV_PAGED, false, false>(p, st);
}

int run_tree(const TreeParams& p, int dtype, int head_dim, int walk, int layout, bool pstate, int algo,
             hipStream_t st) {
    const bool lse = p.lse != nullptr;
    if (dtype == QATTN_DTYPE_F16) {
        switch (head_dim) {
            case 32: return dispatch_tree<F16, 32>(p, walk, layout, lse, pstate, algo, st);
            case 64: return dispatch_tree<F16, 64>(p, walk, layout, lse, pstate, algo, st);
            default: return dispatch_tree<F16, 128>(p, walk, layout, lse, pstate, algo, st);
        }
    }
    switch (head_dim) {
        case 32: return dispatch_tree<BF16, 32>(p, walk, layout, lse, pstate, algo, st);
        case 64: return dispatch_tree<BF16, 64>(p, walk, layout, lse, pstate, algo, st);
        default: return dispatch_tree<BF16, 128>(p, walk, layout, lse, pstate, algo, st);
    }
}

// Fill the fields shared by the tree entry points.  Returns an error code.
int fill_tree_params(TreeParams& p, const void* q, const int64_t* qs, const void* k, const int64_t* ks,
                     const void* v, const int64_t* vs, void* o, const int64_t* os, float* lse,
                     const int64_t* lss, const int32_t* cu, int32_t batch, int32_t max_seqlen,
                     int64_t total_tokens, int32_t hq, int32_t hkv, int32_t b, int32_t max_depth, float scale,
                     bool uniform) {
    p = TreeParams{};
    if (!q || !qs || !k || !ks || !v || !vs || !o || !os || (!cu && !uniform) || (lse && !lss)) {
        set_error("null pointer argument");
        return QATTN_ERR_ARG;
    }
    if (b < 1) {
        set_error("branching_factor %d < 1", b);
        return QATTN_ERR_ARG;
    }
    if (!row_aligned(q, qs, 2) || !row_aligned(o, os, 2)) {
        set_error("q/o rows must be 16-byte aligned with stride_dim 1");
        return QATTN_ERR_LAYOUT;
    }
    if (!(scale == scale)) {
        set_error("scale is NaN");
        return QATTN_ERR_ARG;
    }
    p.q = q;
    p.k = k;
    p.v = v;
    p.o = o;
    p.lse = lse;
    p.cu = cu;
    p.sq_t = qs[0];
    p.sq_h = qs[1];
    p.sk_t = ks[0];
    p.sk_h = ks[1];
    p.sv_t = vs[0];
    p.sv_h = vs[1];
    p.so_t = os[0];
    p.so_h = os[1];
    if (lse) {
        p.slse_t = lss[0];
        p.slse_h = lss[1];
    }
    p.total_tokens = total_tokens;
    p.kv_rows = total_tokens;
    p.B = batch;
    p.Hq = hq;
    p.Hkv = hkv;
    p.group = hq / hkv;
    p.max_seqlen = max_seqlen;
    p.max_depth = max_depth;
    p.bdiv = make_divider(b);
    p.hqdiv = make_divider(hq);
    p.msdiv = make_divider(max_seqlen > 0 ? max_seqlen : 1);
    p.scale_log2 = scale * kLog2e;
    p.dbg_walk = g_dbg_walk;
    return QATTN_OK;
}

}  // namespace qattn

using namespace qattn;

extern "C" {

const char* qattn_version(void) { return "qattention_amd 0.1.0 (gfx950)"; }

const char* qattn_last_error(void) { return g_err; }

int qattn_debug_walk(int32_t* out) {
    g_dbg_walk = out;
    return QATTN_OK;
}

const char* qattn_debug_last_kernel(void) { return g_last_kernel; }

int qattn_tree_fwd(const void* q, const int64_t q_stride[3], const void* k, const int64_t k_stride[3],
                   const void* v, const int64_t v_stride[3], void* o, const int64_t o_stride[3], float* lse,
                   const int64_t lse_stride[2], const int32_t* cu_seqlens, int32_t batch, int32_t max_seqlen,
                   int64_t total_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                   int32_t branching_factor, int32_t max_depth, float scale, int32_t dtype, int32_t algo,
                   void* stream) {
    clear_error();
    int rc = check_common(dtype, head_dim, batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, max_depth);
    if (rc) return rc;
    if (algo < QATTN_ALGO_AUTO || algo > QATTN_ALGO_SUBTREE) {
        set_error("unknown algo %d", algo);
        return QATTN_ERR_ARG;
    }
    if (batch == 0 || max_seqlen == 0 || total_tokens == 0) return QATTN_OK;  // nothing to compute
    TreeParams p;
    rc = fill_tree_params(p, q, q_stride, k, k_stride, v, v_stride, o, o_stride, lse, lse_stride, cu_seqlens,
                          batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, branching_factor, max_depth,
                          scale);
    if (rc) return rc;
    if (!row_aligned(k, k_stride, 2) || !row_aligned(v, v_stride, 2)) {
        set_error("k/v rows must be 16-byte aligned with stride_dim 1");
        return QATTN_ERR_LAYOUT;
    }
    return run_tree(p, dtype, head_dim, WALK_HEAP, KV_PACKED, false, algo, (hipStream_t)stream);
}

int qattn_tree_parents_fwd(const void* q, const int64_t q_stride[3], const void* k, const int64_t k_stride[3],
                           const void* v, const int64_t v_stride[3], void* o, const int64_t o_stride[3],
                           float* lse, const int64_t lse_stride[2], const int32_t* cu_seqlens,
                           const int32_t* parents, int32_t batch, int32_t max_seqlen, int64_t total_tokens,
                           int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t max_depth,
                           float scale, int32_t dtype, void* stream) {
    clear_error();
    int rc = check_common(dtype, head_dim, batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, max_depth);
    if (rc) return rc;
    if (batch == 0 || max_seqlen == 0 || total_tokens == 0) return QATTN_OK;  // nothing to compute
    if (!parents) {
        set_error("parents is null");
        return QATTN_ERR_ARG;
    }
    TreeParams p;
    rc = fill_tree_params(p, q, q_stride, k, k_stride, v, v_stride, o, o_stride, lse, lse_stride, cu_seqlens,
                          batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, 1, max_depth, scale);
    if (rc) return rc;
    if (!row_aligned(k, k_stride, 2) || !row_aligned(v, v_stride, 2)) {
        set_error("k/v rows must be 16-byte aligned with stride_dim 1");
        return QATTN_ERR_LAYOUT;
    }
    p.parents = parents;
    return run_tree(p, dtype, head_dim, WALK_PARENTS, KV_PACKED, false, QATTN_ALGO_GATHER, (hipStream_t)stream);
}

int qattn_tree_paged_fwd(const void* q, const int64_t q_stride[3], const void* k_cache, const int64_t k_stride[4],
                         const void* v_cache, const int64_t v_stride[4], void* o, const int64_t o_stride[3],
                         float* lse, const int64_t lse_stride[2], const int32_t* cu_seqlens,
                         const int32_t* page_table, int32_t pt_cols, int32_t num_pages, int32_t page_size,
                         int32_t batch, int32_t max_seqlen, int64_t total_tokens, int32_t num_q_heads,
                         int32_t num_kv_heads, int32_t head_dim, int32_t branching_factor, int32_t max_depth,
                         float scale, int32_t dtype, int32_t algo, void* stream) {
    clear_error();
    int rc = check_common(dtype, head_dim, batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, max_depth);
    if (rc) return rc;
    if (algo < QATTN_ALGO_AUTO || algo > QATTN_ALGO_SUBTREE) {
        set_error("unknown algo %d", algo);
        return QATTN_ERR_ARG;
    }
    if (batch == 0 || max_seqlen == 0 || total_tokens == 0) return QATTN_OK;  // nothing to compute
    if (!page_table || !k_stride || !v_stride || page_size < 1 || pt_cols < 0 || num_pages < 0) {
        set_error("bad paged arguments: page_size=%d pt_cols=%d num_pages=%d", page_size, pt_cols, num_pages);
        return QATTN_ERR_ARG;
    }
    // The walk's K/V access is page * stride_page + slot * stride_slot + head * stride_head.
    const int64_t ks3[3] = {k_stride[1], k_stride[2], k_stride[3]};
    const int64_t vs3[3] = {v_stride[1], v_stride[2], v_stride[3]};
    TreeParams p;
    rc = fill_tree_params(p, q, q_stride, k_cache, ks3, v_cache, vs3, o, o_stride, lse, lse_stride, cu_seqlens,
                          batch, max_seqlen, total_tokens, num_q_heads, num_kv_heads, branching_factor, max_depth,
                          scale);
    if (rc) return rc;
    if (!row_aligned(k_cache, ks3, 2) || !row_aligned(v_cache, vs3, 2) || k_stride[0] % 8 || v_stride[0] % 8) {
        set_error("k/v cache rows must be 16-byte aligned with stride_dim 1");
        return QATTN_ERR_LAYOUT;
    }
    p.page_table = page_table;
    p.pt_cols = pt_cols;
    p.num_pages = num_pages;
    p.page_size = page_size;
    p.pdiv = make_divider(page_size);
    p.sk_page = k_stride[0];
    p.sv_page = v_stride[0];
    return run_tree(p, dtype, head_dim, WALK_HEAP, KV_PAGED, false, algo, (hipStream_t)stream);
}

int qattn_ancestors(const int32_t* cu_seqlens, const int32_t* parents, int32_t batch, int32_t max_seqlen,
                    int64_t total_tokens, int32_t branching_factor, int32_t max_depth, int32_t* out,
                    void* stream) {
    clear_error();
    if (!cu_seqlens || !out || batch < 0 || max_seqlen < 0 || total_tokens < 0 || max_depth < 0 ||
        (!parents && branching_factor < 1) || total_tokens >= (int64_t(1) << 31)) {
        set_error("bad arguments to qattn_ancestors");
        return QATTN_ERR_ARG;
    }
    if (batch == 0 || max_seqlen == 0 || total_tokens == 0) return QATTN_OK;
    TreeParams p{};
    p.cu = cu_seqlens;
    p.parents = parents;
    p.B = batch;
    p.max_seqlen = max_seqlen;
    p.total_tokens = total_tokens;
    p.max_depth = max_depth;
    p.bdiv = make_divider(parents ? 1 : branching_factor);
    const int64_t n = (int64_t)batch * max_seqlen;
    const int64_t blocks = (n + kThreads - 1) / kThreads;
    if (parents)
        hipLaunchKernelGGL(ancestors_kernel<WALK_PARENTS>, dim3((unsigned)blocks), dim3(kThreads), 0,
                           (hipStream_t)stream, p, out);
    else
        hipLaunchKernelGGL(ancestors_kernel<WALK_HEAP>, dim3((unsigned)blocks), dim3(kThreads), 0,
                           (hipStream_t)stream, p, out);
    return launch_status("ancestors_kernel");
}

int qattn_lse_merge(const float* lse_pre, const int64_t lse_pre_stride[3], const float* lse_tree,
                    const int64_t lse_tree_stride[3], const void* o_pre, const int64_t o_pre_stride[4],
                    const void* o_tree, const int64_t o_tree_stride[4], void* out, const int64_t out_stride[4],
                    int32_t B, int32_t H, int32_t Nq, int32_t head_dim, int32_t dtype, void* stream) {
    clear_error();
    if (!lse_pre || !lse_tree || !o_pre || !o_tree || !out || !lse_pre_stride || !lse_tree_stride ||
        !o_pre_stride || !o_tree_stride || !out_stride || B < 0 || H < 0 || Nq < 0) {
        set_error("bad arguments to qattn_lse_merge");
        return QATTN_ERR_ARG;
    }
    if (dtype != QATTN_DTYPE_F16 && dtype != QATTN_DTYPE_BF16) {
        set_error("dtype %d is not fp16 (0) or bf16 (1)", dtype);
        return QATTN_ERR_DTYPE;
    }
    if (head_dim != 32 && head_dim != 64 && head_dim != 128) {
        set_error("head_dim %d not in {32, 64, 128}", head_dim);
        return QATTN_ERR_HEAD_DIM;
    }
    if (!row_aligned(o_pre, o_pre_stride, 3) || !row_aligned(o_tree, o_tree_stride, 3) ||
        !row_aligned(out, out_stride, 3)) {
        set_error("merge operands must have stride_dim 1 and 16-byte aligned rows");
        return QATTN_ERR_LAYOUT;
    }
    const int64_t npos = (int64_t)B * H * Nq;
    if (npos == 0) return QATTN_OK;
    MergeParams mp{};
    mp.lse_p = lse_pre;
    mp.lse_t = lse_tree;
    mp.o_p = o_pre;
    mp.o_t = o_tree;
    mp.out = out;
    for (int i = 0; i < 3; ++i) {
        mp.sl_p[i] = lse_pre_stride[i];
        mp.sl_t[i] = lse_tree_stride[i];
    }
    for (int i = 0; i < 4; ++i) {
        mp.so_p[i] = o_pre_stride[i];
        mp.so_t[i] = o_tree_stride[i];
        mp.so[i] = out_stride[i];
    }
    mp.B = B;
    mp.H = H;
    mp.Nq = Nq;
    const int slots = kThreads / (head_dim / 8);
    const int64_t blocks = (npos + slots - 1) / slots;
    if (blocks >= (int64_t(1) << 31)) {
        set_error("grid too large");
        return QATTN_ERR_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
#define QATTN_MERGE(T, D) \
    hipLaunchKernelGGL((lse_merge_kernel<T, D>), dim3((unsigned)blocks), dim3(kThreads), 0, st, mp)
    if (dtype == QATTN_DTYPE_F16) {
        if (head_dim == 32) QATTN_MERGE(F16, 32);
        else if (head_dim == 64) QATTN_MERGE(F16, 64);
        else QATTN_MERGE(F16, 128);
    } else {
        if (head_dim == 32) QATTN_MERGE(BF16, 32);
        else if (head_dim == 64) QATTN_MERGE(BF16, 64);
        else QATTN_MERGE(BF16, 128);
    }
#undef QATTN_MERGE
    return launch_status("lse_merge_kernel");
}

}  // extern "C"
