/*
 * bp_resident_diff.hip -- the unrolled forward and the adjoint of bp_diff.hip
 * as resident runs: networks that fit on the chip (bp_resident.hip) go
 * through all K iterations, or all K + 1 adjoint steps, in one launch.
 *
 * An adjoint step launched on its own moves 135 MB for a 200k-node 3-state
 * DAG: tables (26 MB), their gradients read and written (52), messages'
 * operands, w (23), beliefs.  Here each thread keeps its slots' tables and
 * their gradients in registers for all steps, the nodes' dL/dst stay in
 * registers too, messages and the nodes' dT in LDS; a step gathers the
 * combine buffers of the kept iterates, reads a row or two of beliefs per
 * node and exchanges w.
 *
 * w: each workgroup writes its slots' rows in the order in which they are
 * dealt to its threads, a stretch of its own per step, and a node gathers
 * the rows of its out-edges by their places (`out_at`).  The slots are dealt
 * in order of their sources, so what one workgroup needs of another's rows
 * lies together, no line has two writers, and a step's stretch is read by
 * ordinary loads, as the combine buffers are in bp_resident.hip.  (Rows
 * scattered to their place in the source-grouped list, as the launches have
 * it, are 8-byte stores through to memory and loads past the caches here.)
 * What a step needs of the kept iterates alone (messages, their products)
 * comes between arriving at the grid barrier and waiting there.
 * Measured, per step: 200k nodes of 3 states (725k slots) 25 us, against 30
 * with all of it behind the barrier, 38 with scattered rows and 35 as
 * launches; 2k nodes 6.9, 17 as launches.
 * Everything else that is read was written by an earlier launch.
 *
 * Both runs are enqueued on the caller's stream and not waited for.  The
 * kernels behind them make up for a run that was given up: one workgroup,
 * which needs no other, goes through the same steps with the launches' code
 * and leaves word for the host, whose later calls use launches.
 *
 * Every float operation is the launches', in their order: gradients are
 * bit-identical.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "bp_adjoint.h"
#include "bp_resident.h"

using namespace bpk;

namespace {

struct ResAdjArgs {
    const unsigned *in_off, *slot_src, *out_off;
    const unsigned *out_at; /* [E] by source: where the out-edge's row of w is */
    const float *J;
    const unsigned *wg_node;
    const unsigned short *wg_slots;
    const float *st, *buf; /* kept iterates */
    size_t stride;
    const float *st0, *gin;
    float *w;        /* step t's rows at w + t * w_stride */
    size_t w_stride;
    float *jbar, *dst0;
    unsigned K;
    Meeting meeting;
};

template <typename F> __device__ __forceinline__ F *row_at(F *p, unsigned bytes)
{
    return reinterpret_cast<F *>((uintptr_t)p + bytes);
}

/* T threads, NS slots for each: half the threads of the forward's workgroups,
 * with twice the registers, where a slot's table and gradient would not
 * leave 128 enough. */
template <int S, int T, int NS>
__global__ __launch_bounds__(T) void k_resident_adjoint(ResAdjArgs a)
{
    constexpr int SP = Stride<S>::value;
    constexpr int NN = T < RB ? (NS / 2 + 1) / 2 * 2 : (NS + 1) / 2; /* nodes per thread */
    constexpr int W = T * NS;
    /* What the registers have room for: sibling products before the wait,
     * rows of w through LDS, products without the tests for NaN, the next
     * step's gathers before the barrier.  A backward of 31 steps, us,
     * without the last three / with them: 2k nodes of 3 states 282 / 228, 60k
     * 395 / 331, 120k 602 / 525, 150k binary 539 / 471 (by the third alone),
     * 8k of 4 states 324 / 248; at three slots of 3 states they spill
     * (200k nodes 885 / 980). */
    constexpr bool EARLY = NS == 1, STAGED = NS <= 2, FAST = S != 3 || NS != 3, AHEAD = NS <= 2;
    __shared__ __align__(16) float lm[S * (W + PAD)]; /* messages by slot */
    __shared__ __align__(16) float ldt[S * T * NN];  /* the nodes' dT */
    __shared__ unsigned short lnode[W];               /* the slot's node */
    __shared__ unsigned lout[W];                      /* out_at of the workgroup's nodes, as much as fits */
    __shared__ __align__(16) float lw[STAGED ? S * (W + 4) : 1]; /* their rows of w */
    __shared__ unsigned ok, committed, suspect;
    const unsigned tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const unsigned G = gridDim.x, wg = xcd_block(blockIdx.x, G);
    if (called_off(a.meeting))
        return;
    const unsigned n0 = a.wg_node[wg], n1 = a.wg_node[wg + 1];
    const unsigned s0 = a.in_off[n0], ns = a.in_off[n1] - s0, ob = a.out_off[n0];
    const unsigned outs = min((unsigned)W, a.out_off[n1] - ob);
    for (unsigned o = tid; o < outs; o += T)
        lout[o] = a.out_at[ob + o];
    if (tid == 0)
        suspect = 0;

    /* the nodes: in-slots (first | count << 16) and out-edges */
    unsigned slots[NN], o0[NN], o1[NN];
    float g[NN][S];
#pragma unroll
    for (int r = 0; r < NN; ++r) {
        const unsigned l = r * T + tid, v = n0 + l;
        slots[r] = o0[r] = o1[r] = 0;
        if (v < n1) {
            const unsigned b = a.in_off[v] - s0, e = a.in_off[v + 1] - s0;
            slots[r] = b | (e - b) << 16;
            o0[r] = a.out_off[v] - ob;
            o1[r] = a.out_off[v + 1] - ob;
            load_rowp<S, SP>(a.gin + (size_t)v * SP, g[r]);
            for (unsigned q = b; q < e; ++q)
                lnode[q] = (unsigned short)l;
        }
    }
    /* the slots, in source order: place in LDS, source, node and siblings
     * (node: 11 bits, first sibling: 13, count: 8) */
    float J[NS][S * S], jb[NS][S * S];
    unsigned src[NS], at[(NS + 1) / 2], sib[NS];
    /* the rows of w from the nodes' out-edges, to LDS: a thread for each, all
     * in one round trip (a thread for each node, four at a time, took as
     * long as the node with the most: 2.6 us of 8.5 on 2k nodes) */
    auto fetch_w = [&](const float *w) {
        if constexpr (!STAGED)
            return;
        float x[NS][S];
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (k * T + tid < outs)
                load_rowp<S, SP>(w + (size_t)lout[k * T + tid] * SP, x[k]);
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (k * T + tid < outs)
                put_row<S>(lw + (k * T + tid) * S, x[k]);
        __syncthreads();
    };
    /* acc += the rows from [b, e), in order */
    auto add_w = [&](const float *w, unsigned b, unsigned e, float *acc) {
        for (unsigned o = b; o < e; o += 4) {
            float x[4][S];
            if (STAGED && o + 4 <= W) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    get_row<S>(lw + (o + u) * S, x[u]);
            } else {
                unsigned p[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const unsigned q = o + u < e ? o + u : o;
                    p[u] = q < (unsigned)W ? lout[q] : a.out_at[ob + q];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    load_rowp<S, SP>(w + (size_t)p[u] * SP, x[u]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (o + u < e)
#pragma unroll
                    for (int i = 0; i < S; ++i)
                        acc[i] = acc[i] + x[u][i];
        }
    };
    /* the product of the messages that a slot's node gets beside its own */
    auto siblings = [&](auto clean, int k, float *P) {
        const unsigned place = k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu;
        const unsigned q0 = sib[k] >> 11 & 0x1fffu, cnt = (sib[k] >> 24) + 1, own = place - q0;
#pragma unroll
        for (int i = 0; i < S; ++i)
            P[i] = 1.0f;
        for (unsigned q = 0; q < cnt; q += 4) {
            float f[4][S];
            factors<S, S, 4, !decltype(clean)::value>(lm + (q0 + q) * S, cnt - q, f);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < S; ++i)
                    P[i] = P[i] * (q + j == own ? 1.0f : f[j][i]);
        }
    };
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        src[k] = n0 * (SP * 4u);
        sib[k] = 0;
        if (k % 2 == 0)
            at[k / 2] = 0;
        if (k * T + wave * WAVE >= ns)
            continue; /* the wave has no slot in this turn */
        const unsigned l = k * T + tid, q = a.wg_slots[(size_t)wg * W + (l < ns ? l : ns - 1)];
        at[k / 2] = k % 2 ? (at[k / 2] & 0xffffu) | q << 16 : q;
        src[k] = a.slot_src[s0 + q] * (SP * 4u); /* byte offsets of rows: 32 bits do */
        const unsigned n = lnode[q], b = a.in_off[n0 + n] - s0, e = a.in_off[n0 + n + 1] - s0;
        sib[k] = n | b << 11 | (e - b - 1) << 24; /* one in-edge at least, 256 at most */
    }
    /* tables by way of LDS, a row of all slots at a time */
#pragma unroll
    for (int c = 0; c < S; ++c) {
        for (unsigned l = tid; l < ns; l += T) {
            float t[S];
            load_row<S>(a.J + ((size_t)(s0 + l) * S + c) * S, t);
            put_row<S>(lm + l * S, t);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (k * T + wave * WAVE < ns)
                get_row<S>(lm + (k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu) * S, J[k] + c * S);
        __syncthreads();
    }
    unsigned number = 1;
    grid_arrive(a.meeting, wg);

    /* the combine buffers that step t's messages are made of */
    auto sources = [&](unsigned t) { return t == 0 ? a.st0 : a.buf + (size_t)(t - 1) * a.stride; };
    float ahead[AHEAD ? NS : 1][S];
    auto gather = [&](unsigned t) {
        if constexpr (AHEAD)
#pragma unroll
            for (int k = 0; k < NS; ++k)
                load_rowp<S, SP>(row_at(sources(t), src[k]), ahead[k]);
    };
    gather(a.K);
    for (unsigned t = a.K + 1; t-- > 0;) {
        const bool last = t == 0; /* step 0: m_0 from st_0 */
        hold(at);
        hold(sib);
        hold(slots);
        float b[NS][S], sig[NS];
        bool odd = false; /* a message that may hold NaN */
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if constexpr (AHEAD) {
#pragma unroll
                for (int i = 0; i < S; ++i)
                    b[k][i] = ahead[k][i];
            } else {
                load_rowp<S, SP>(row_at(sources(t), src[k]), b[k]);
            }
        }
        /* slot phase 1: the messages and their sums (0: not positive) */
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (k * T + wave * WAVE >= ns)
                continue;
            float m[S], sum = 0.0f;
#pragma unroll
            for (int i = 0; i < S; ++i) {
                float acc = 0.0f;
#pragma unroll
                for (int j = 0; j < S; ++j)
                    acc = acc + J[k][i * S + j] * b[k][j];
                m[i] = acc;
                sum = sum + acc;
            }
            const bool positive = sum > 0.0f;
            odd = odd || !(fabsf(sum) < INFINITY);
            if (!positive)
                sum = 1.0f;
            sig[k] = positive ? sum : 0.0f;
#pragma unroll
            for (int i = 0; i < S; ++i)
                m[i] = m[i] / sum;
            if (k * T + tid < ns) {
                const unsigned place = k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu;
                put_row<S>(lm + place * S, m);
            }
        }
        if (FAST && __ballot(odd) != 0 && lane == 0)
            suspect = t + 1;
        __syncthreads();
        /* the products of the nodes' in-messages and, with a slot per
         * thread, of each slot's siblings; without the tests for NaN where
         * every message's sum was finite */
        float Tm[NN][S], P[EARLY ? NS : 1][S];
        const bool clean = FAST && __builtin_amdgcn_readfirstlane(suspect) != t + 1; /* uniform */
        auto products = [&](auto clean) {
#pragma unroll
            for (int r = 0; r < NN; ++r) {
                const unsigned cnt = slots[r] >> 16;
                const float *msgs = lm + (slots[r] & 0xffffu) * S;
#pragma unroll
                for (int i = 0; i < S; ++i)
                    Tm[r][i] = 1.0f;
                for (unsigned q = 0; q < cnt; q += 4) {
                    float f[4][S];
                    factors<S, S, 4, !decltype(clean)::value>(msgs + q * S, cnt - q, f);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        mul_all<S>(Tm[r], f[j]);
                }
            }
            if constexpr (EARLY)
#pragma unroll
                for (int k = 0; k < NS; ++k)
                    if (k * T + tid < ns)
                        siblings(clean, k, P[k]);
        };
        if (clean)
            products(std::true_type());
        else
            products(std::false_type());
        /* the other workgroups' w of the step before (the first time: all are here) */
        if (!grid_wait(a.meeting, G, number++, &ok))
            return;
        if (t < a.K)
            fetch_w(a.w + (size_t)(t + 1) * a.w_stride);
        /* node phase: dT, dL/dst_{t-1} */
#pragma unroll
        for (int r = 0; r < NN; ++r) {
            const unsigned l = r * T + tid, v = n0 + l;
            if (v < n1) {
                float gb[S], dT[S], stp[S], stc[S];
                load_rowp<S, SP>((last ? a.st0 : a.st + (size_t)t * a.stride) + (size_t)v * SP, stc);
                if (!last)
                    load_rowp<S, SP>((t > 1 ? a.st + (size_t)(t - 1) * a.stride : a.st0) + (size_t)v * SP, stp);
#pragma unroll
                for (int i = 0; i < S; ++i)
                    gb[i] = 0.0f;
                if (t < a.K)
                    add_w(a.w + (size_t)(t + 1) * a.w_stride, o0[r], o1[r], gb);
                if (last) {
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        dT[i] = gb[i] * stc[i];
                        g[r][i] = g[r][i] + gb[i] * Tm[r][i];
                    }
                } else {
                    const bool indeg = slots[r] >> 16;
                    float ds[S], sa = 0.0f, dot = 0.0f;
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        ds[i] = g[r][i] + gb[i] * Tm[r][i];
                        dT[i] = gb[i] * stc[i];
                        const float av = indeg ? stp[i] * Tm[r][i] : stp[i];
                        sa = sa + av;
                        dot = dot + ds[i] * stc[i];
                    }
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        const float da = (sa > 0.0f) ? (ds[i] - dot) / sa : ds[i];
                        g[r][i] = indeg ? da * Tm[r][i] : da;
                        if (indeg)
                            dT[i] = dT[i] + da * stp[i];
                    }
                }
                put_row<S>(ldt + l * S, dT);
            }
        }
        __syncthreads();
        if (!last)
            gather(t - 1);
        /* slot phase 2: dm, dz, dJ, w */
        float *wout = a.w + (size_t)t * a.w_stride + (size_t)wg * W * SP;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const unsigned l = k * T + tid;
            if (l < ns) {
                const unsigned place = k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu;
                float (&Pk)[S] = P[EARLY ? k : 0];
                float m[S], dT[S], dm[S], dz[S], dot = 0.0f;
                if constexpr (!EARLY) {
                    if (clean)
                        siblings(std::true_type(), k, Pk);
                    else
                        siblings(std::false_type(), k, Pk);
                }
                get_row<S>(lm + place * S, m);
                get_row<S>(ldt + (sib[k] & 0x7ffu) * S, dT);
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    dm[i] = (m[i] == m[i]) ? dT[i] * Pk[i] : 0.0f;
                    dot = dot + dm[i] * m[i];
                }
#pragma unroll
                for (int i = 0; i < S; ++i)
                    dz[i] = sig[k] > 0.0f ? (dm[i] - dot) / sig[k] : dm[i];
#pragma unroll
                for (int i = 0; i < S; ++i)
#pragma unroll
                    for (int j = 0; j < S; ++j)
                        jb[k][i * S + j] = t == a.K ? dz[i] * b[k][j] : jb[k][i * S + j] + dz[i] * b[k][j];
                float wv[SP];
#pragma unroll
                for (int j = 0; j < SP; ++j) {
                    float acc = 0.0f;
                    if (j < S)
#pragma unroll
                        for (int i = 0; i < S; ++i)
                            acc = acc + J[k][i * S + j] * dz[i];
                    wv[j] = acc;
                }
                store_row_agent<SP>(wout + l * SP, wv);
            }
        }
        grid_arrive(a.meeting, wg);
    }
    if (!grid_wait(a.meeting, G, number, &ok))
        return;
    if (tid == 0)
        committed = settle(a.meeting.decision, a.meeting.run, COMMIT);
    __syncthreads();
    if (!committed)
        return;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const unsigned l = k * T + tid;
        if (l < ns) {
            float *to = a.jbar + (size_t)(s0 + (k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu)) * S * S;
#pragma unroll
            for (int i = 0; i < S * S; ++i)
                to[i] = jb[k][i];
        }
    }
    fetch_w(a.w);
#pragma unroll
    for (int r = 0; r < NN; ++r) {
        const unsigned v = n0 + r * T + tid;
        if (v < n1) {
            /* dL/dst_0 = what step 0 left + w_0 of the out-edges */
            add_w(a.w, o0[r], o1[r], g[r]);
            float row[SP];
#pragma unroll
            for (int i = 0; i < SP; ++i)
                row[i] = i < S ? g[r][i] : 0.0f;
            store_row_nt<SP>(a.dst0 + (size_t)v * SP, row);
        }
    }
}

/* out_at: the place of each slot's row of w, by the slot's position in the
 * source-grouped list */
__global__ void k_places(const unsigned *in_off, const unsigned *wg_node, const unsigned short *wg_slots, unsigned W,
                         const unsigned *slot_pos, unsigned *out_at)
{
    const unsigned wg = blockIdx.x, s0 = in_off[wg_node[wg]], ns = in_off[wg_node[wg + 1]] - s0;
    for (unsigned l = threadIdx.x; l < ns; l += blockDim.x)
        out_at[slot_pos[s0 + wg_slots[(size_t)wg * W + l]]] = wg * W + l;
}

/* ---- one workgroup's way through the same steps --------------------------- */

__device__ __forceinline__ bool went_through(const Meeting &m)
{
    return __hip_atomic_load(m.decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (m.run << 1 | COMMIT);
}

/* what the workgroup's waves wrote is there for all of them */
__device__ __forceinline__ void group_step()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}

template <int S>
__global__ __launch_bounds__(BLOCK) void k_forward_rescue(LoopyArgs a, float *st, float *buf, size_t stride, unsigned K,
                                                          Meeting m, unsigned *gave_up)
{
    if (went_through(m))
        return;
    constexpr int R = SlotsPerLane<S>::value;
    __shared__ float lds[WAVES_PER_BLOCK][S * WAVE * R];
    unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    double none = 0.0;
    for (unsigned t = 1; t <= K; ++t) {
        a.states = st + (size_t)(t - 1) * stride;
        a.states_out = st + (size_t)t * stride;
        a.buf_in = buf + (size_t)(t - 1) * stride;
        a.buf_out = buf + (size_t)t * stride;
        for (unsigned c = wave; c < a.nchunks; c += WAVES_PER_BLOCK)
            run_chunk<S, false, FWD, R, false, 1, false>(a, c, lds[wave], nullptr, nullptr, lane, none);
        group_step();
    }
    if (threadIdx.x == 0)
        __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int S>
__global__ __launch_bounds__(BLOCK) void k_adjoint_rescue(AdjArgs a, const float *st, const float *buf, size_t stride,
                                                          const float *st0, const float *gin, float *gst0, float *gst1,
                                                          float *w0, float *w1, float *dst0p, float *dst0, unsigned V,
                                                          unsigned K, Meeting m, unsigned *gave_up)
{
    constexpr int SP = Stride<S>::value;
    if (went_through(m))
        return;
    constexpr int R = S <= 4 ? BP_ADJ_SLOTS_SMALL : 1, W = WAVE * R;
    __shared__ float lm[WAVES_PER_BLOCK][S * W];
    __shared__ float ldt[WAVES_PER_BLOCK][S * W];
    __shared__ unsigned short lnode[WAVES_PER_BLOCK][W];
    __shared__ unsigned short lq[WAVES_PER_BLOCK][2 * W];
    unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const float *g = gin;
    for (unsigned t = K; t > 0; --t) {
        a.st_prev = t > 1 ? st + (size_t)(t - 1) * stride : st0;
        a.st_cur = st + (size_t)t * stride;
        a.bsrc = buf + (size_t)(t - 1) * stride;
        a.gst_in = g;
        a.gst_out = t & 1 ? gst0 : gst1;
        a.w_in = t < K ? ((t + 1) & 1 ? w1 : w0) : nullptr;
        a.w_out = t & 1 ? w1 : w0;
        a.jbar_first = t == K;
        for (unsigned c = wave; c < a.nchunks; c += WAVES_PER_BLOCK)
            adjoint_chunk<S, 0, R>(a, c, lm[wave], ldt[wave], lnode[wave], lq[wave], lane);
        g = a.gst_out;
        group_step();
    }
    a.st_prev = nullptr;
    a.st_cur = a.bsrc = st0;
    a.gst_in = g;
    a.gst_out = dst0p;
    a.w_in = K ? w1 : nullptr;
    a.w_out = w0;
    a.jbar_first = K == 0;
    for (unsigned c = wave; c < a.nchunks; c += WAVES_PER_BLOCK)
        adjoint_chunk<S, 1, R>(a, c, lm[wave], ldt[wave], lnode[wave], lq[wave], lane);
    group_step();
    for (unsigned v = threadIdx.x; v < V; v += blockDim.x) {
        float acc[S];
        load_rowp<S, SP>(dst0p + (size_t)v * SP, acc);
        sum_out_w<S, SP>(w0, a.out_slot, a.out_off[v], a.out_off[v + 1], acc);
#pragma unroll
        for (int i = 0; i < SP; ++i)
            dst0[(size_t)v * SP + i] = i < S ? acc[i] : 0.0f;
    }
    if (threadIdx.x == 0)
        __hip_atomic_store(gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* Slots per thread of the plan (of 1024) that the adjoint's registers hold
 * with their gradients. */
constexpr unsigned adjoint_slots(unsigned S) { return S == 2 ? 4 : S == 3 ? 3 : 2; }

template <int S, int NS> void launch_ns(const ResAdjArgs &a, unsigned G, hipStream_t st)
{
    /* table and gradient of a slot: 2 S S registers */
    constexpr bool HALF = 2 * S * S * NS > 54;
    constexpr int T = HALF ? RB / 2 : RB;
    hipLaunchKernelGGL((k_resident_adjoint<S, T, HALF ? 2 * NS : NS>), dim3(G), dim3(T), 0, st, a);
}

template <int S> void launch_adjoint(const ResAdjArgs &a, unsigned ns, unsigned G, hipStream_t st)
{
    if (ns == 1)
        launch_ns<S, 1>(a, G, st);
    else if (ns == 2)
        launch_ns<S, 2>(a, G, st);
    else if constexpr (adjoint_slots(S) > 2)
        if (ns == adjoint_slots(S))
            launch_ns<S, (int)adjoint_slots(S)>(a, G, st);
}

} // namespace

/* 2 to 4 states, slots per thread within the adjoint's registers and
 * in-degrees within its packed fields. */
bool bp_resident_diff_fits(const bp_dev *d, unsigned max_in_degree)
{
    const bp_resident &r = d->res;
    return r.on && !d->mixed && d->S >= 2 && d->S <= 4 && r.ns <= adjoint_slots(d->S) && max_in_degree <= 256 &&
           !d->status()->gave_up;
}

size_t bp_resident_diff_rows(const bp_dev *d) { return (size_t)d->res.G * d->res.ns * RB * d->SP; }

int bp_resident_diff_places(bp_dev *d, const unsigned *slot_pos, unsigned *out_at)
{
    const bp_resident &r = d->res;
    hipLaunchKernelGGL(k_places, dim3(r.G), dim3(256), 0, d->stream, d->in_off, r.wg_node, r.wg_slots, r.ns * RB,
                       slot_pos, out_at);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(d->stream));
    return 0;
}

int bp_resident_diff_forward(bp_dev *d, unsigned K, float *st, float *buf, size_t stride, hipStream_t stream)
{
    std::lock_guard<std::mutex> lock(bp_resident_mutex());
    Meeting m;
    if (bp_resident_turn(d->device, stream) || bp_resident_forward(d, K, st, buf, stride, stream, &m))
        return -1;
    if (!d->res.single) {
        LoopyArgs a = bp_make_args(d);
        a.J = d->J;
        a.slot_tab = nullptr;
        unsigned *word = &d->status()->gave_up;
        if (d->S == 2)
            hipLaunchKernelGGL(k_forward_rescue<2>, dim3(1), dim3(BLOCK), 0, stream, a, st, buf, stride, K, m, word);
        else if (d->S == 3)
            hipLaunchKernelGGL(k_forward_rescue<3>, dim3(1), dim3(BLOCK), 0, stream, a, st, buf, stride, K, m, word);
        else
            hipLaunchKernelGGL(k_forward_rescue<4>, dim3(1), dim3(BLOCK), 0, stream, a, st, buf, stride, K, m, word);
        HIP_TRY(hipGetLastError());
    }
    return bp_resident_turn_taken(d->device, stream, true);
}

int bp_resident_diff_backward(bp_dev *d, unsigned K, const float *st, const float *buf, size_t stride,
                              const bp_adjoint_arrays &x, hipStream_t stream)
{
    bp_resident &r = d->res;
    std::lock_guard<std::mutex> lock(bp_resident_mutex());
    if (bp_resident_turn(d->device, stream))
        return -1;
    ResAdjArgs a;
    a.in_off = d->in_off;
    a.slot_src = d->slot_src;
    a.out_off = x.out_off;
    a.out_at = x.out_at;
    a.J = d->J;
    a.wg_node = r.wg_node;
    a.wg_slots = r.wg_slots;
    a.st = st;
    a.buf = buf;
    a.stride = stride;
    a.st0 = x.st0;
    a.gin = x.gin;
    a.w = x.rows;
    a.w_stride = bp_resident_diff_rows(d);
    a.jbar = x.jbar;
    a.dst0 = x.dst0;
    a.K = K;
    a.meeting = bp_resident_meeting(d, K + 2, r.settled);
    r.settled = r.run;
    AdjArgs s = {};
    s.in_off = d->in_off;
    s.slot_src = d->slot_src;
    s.out_off = x.out_off;
    s.out_slot = x.out_slot;
    s.slot_pos = x.slot_pos;
    s.J = d->J;
    s.chunk = x.chunk;
    s.nchunks = x.nchunks;
    s.jbar = x.jbar;
    unsigned *word = &d->status()->gave_up;
    auto go = [&](auto states) {
        constexpr int S = decltype(states)::value;
        launch_adjoint<S>(a, r.ns, r.G, stream);
        hipLaunchKernelGGL(k_adjoint_rescue<S>, dim3(1), dim3(BLOCK), 0, stream, s, st, buf, stride, x.st0, x.gin,
                           x.gst[0], x.gst[1], x.w[0], x.w[1], x.dst0p, x.dst0, d->V, K, a.meeting, word);
    };
    if (d->S == 2)
        go(std::integral_constant<int, 2>());
    else if (d->S == 3)
        go(std::integral_constant<int, 3>());
    else
        go(std::integral_constant<int, 4>());
    HIP_TRY(hipGetLastError());
    return bp_resident_turn_taken(d->device, stream, true);
}
