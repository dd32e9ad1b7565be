/*
 * bp_resident.hip -- loopy iterations of networks that fit on the chip.
 *
 * k_resident runs many iterations of src/graph/graph.c:1121-1183 in one
 * launch.  Each workgroup (one per CU, 1024 threads) owns a contiguous range
 * of device nodes with their in-slots and keeps what does not change between
 * iterations -- tables, source indices, slot ranges -- in registers, the
 * nodes' beliefs in registers and the last two iterations' messages in LDS.
 * Only the combine buffers travel: 8 or 16 bytes per node and iteration.
 *
 * What bounds a launch per iteration is not the arithmetic: a small network
 * spends its time on launches (5.5 us for 2,600 message edges that take
 * under 1 us of work, and twice that with the stop test's own launch), and a
 * million-arc binary one re-reads its tables, indices and messages from the
 * Infinity Cache every iteration.  The register files hold 128 MB in all,
 * enough for the tables of 2M binary, 0.75M four-state or 0.25M eight-state
 * message edges.
 *
 * Exchange between workgroups.  An iteration writes its combine buffers to a
 * place of its own (`ring`, one per iteration of the launch) with
 * agent-scope stores, which go through to memory, waits for them, and meets
 * the other workgroups at a grid barrier.  The next iteration gathers with
 * ordinary loads: no L2 can hold a stale copy of those lines, because the
 * launch reads no ring address before the barrier that follows its writes,
 * and because workgroup ranges are cut at 128-byte lines, so no line has two
 * writers.  No cache is flushed or invalidated.  (Reading two alternating
 * buffers past the L2s instead was slower.)
 *
 * Gathers.  A lane that gathers alone costs the L2 a request of its own, and
 * a 500k-node iteration made 1.8M of them: 5.8 of its 14.5 us.  Which thread
 * takes which slot is free -- the messages meet in LDS -- so each workgroup's
 * slots are dealt out in order of their source, and lanes that share a line
 * share the request (half as many on random DAGs).
 *
 * The barrier: workgroup w adds 1 to counter w mod 16 (one per 256 bytes) and
 * the first wave polls all 16.  200 barriers of 256 workgroups, per barrier:
 * 1.4 us; one flag per workgroup and 64 bytes 2.5 us, flags in a row 3.8, one
 * counter 3.8.  Up to 64 workgroups every form takes about 1.25 us.
 *
 * Workgroups wait for each other, so all must be on the chip at once.  The
 * grid is at most one workgroup per CU, and the host lets one such launch
 * run on a device at a time (bp_resident_turn).  If other work keeps part of the
 * chip nevertheless, waits end after `timeout` and the run gives up: nothing
 * has been written that a later step reads, the first workgroup to give up
 * (or, past the last barrier, to go on) settles it for all in one word, and
 * the host then runs the same iterations with a launch each.
 *
 * A network whose slots fit one workgroup needs none of this: its combine
 * buffers stay in LDS as well and it can always run (SINGLE).
 *
 * Measured, per iteration, us (a launch each / plain / with deltas / with the
 * stop test): 500k binary nodes 18.8 (with deltas) / 10.6 / 11.6 / 13.3, 5k
 * - / 2.9 / 3.2 / 3.4, 700 in one workgroup 5.5 / 1.7 / 2.2 / 2.3, 200k of 3
 * states 12.5 (plain) / 9.2 / 9.6 / 10.9.
 *
 * Every float operation is the one k_loopy performs, in its order, so
 * beliefs and messages are bit-identical to it; the FP64 deltas add the same
 * terms grouped by workgroup.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "bp_parallel.h"
#include "bp_resident.h"

using namespace bpk;

namespace {

struct ResArgs {
    const unsigned *in_off, *slot_src;
    const unsigned char *slot_xy, *nvars;
    const float *J;
    const unsigned *slot_tab;
    const unsigned *wg_node;        /* [G + 1] first node of each workgroup */
    const unsigned short *wg_slots; /* [G][NS * 1024] the slot (within the workgroup's) of each thread and turn */
    float *states;
    const float *buf_in; /* combine buffers of the first iteration */
    float *buf_out;      /* ... of the iteration after the last */
    float *msg0, *msg1;  /* messages before the run; the other array */
    float *ring;         /* iteration t's combine buffers at ring + t * ring_stride */
    size_t ring_stride;
    float *keep;      /* non-null: every iteration's beliefs go to keep + t * ring_stride, and nothing else is left */
    unsigned S;       /* the network's largest state count */
    unsigned n;       /* iterations, at most */
    int until;        /* stop test of graph.c:1313 after each */
    float conv;
    double previous;  /* the delta before the run, for the test */
    double *partials; /* DELTA: [n][G] delta partials */
    double *parts;    /* [2][MAX_G] the running iteration's, for the test */
    Meeting meeting;
    bp_resident_status *status; /* host memory */
};

/* Lanes per node in the node phase, and rounds of the workgroup over its
 * nodes: a message edge belongs to one node, and the networks' nodes have
 * two to four of them.  Eight states take four lanes of two: a workgroup of
 * 1,024 slots has some 290 nodes, work for five of its 16 waves otherwise. */
template <int S> struct LanesPerNode {
    static constexpr int value = S == 8 ? 4 : 1;
};
template <int S, int NS> struct NodeRounds {
    static constexpr int value = S == 8 ? 2 : (NS + 1) / 2;
};

/* normalise() over four lanes of two entries each: the sum runs through the
 * lanes in entry order, from 0.0 left to right as with one lane. */
__device__ __forceinline__ void normalise_quad(float *v, unsigned h, unsigned n)
{
    float sum = 0.0f;
#pragma unroll
    for (unsigned step = 0; step < 4; ++step) {
        if (step > 0) {
            /* quad_perm (0, 0, 1, 2): each lane gets its left neighbour's */
            const float left = __int_as_float(
                __builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x90, 0xF, 0xF, false));
            sum = h == step ? left : sum;
        }
        if (h == step) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (2 * h + i < n)
                    sum = sum + v[i];
        }
    }
    /* quad_perm (3, 3, 3, 3) */
    sum = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xFF, 0xF, 0xF, false));
    if (sum <= 0.0f)
        sum = 1.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (2 * h + i < n)
            v[i] = v[i] / sum;
}

/* The node phase of k_loopy: st = N(st * t), t = the product of the
 * in-messages in slot order, and the combine buffer b = st * the same
 * factors one by one (graph.c:985-1024, 851-882).  H entries of the node,
 * from h * H on. */
template <int S, bool MIXED, int NS, bool CLEAN, int H>
__device__ __forceinline__ void resident_node(const float *msgs, unsigned cnt, unsigned n, unsigned h, float *st,
                                              float *b)
{
    /* K messages are kept for both products and the rest read D at a time:
     * as many as the tables leave registers for */
    constexpr int HELD = S * S * NS;
    constexpr int K = H == 2 && HELD <= 16 ? 8 : HELD > 36 && S < 8 ? 2 : 4, D = HELD > 32 && S < 8 ? 2 : 4;
    float f[K][H], t[H];
    factors<S, H, K, CLEAN>(msgs, cnt, f);
#pragma unroll
    for (int i = 0; i < H; ++i)
        t[i] = 1.0f;
#pragma unroll
    for (int j = 0; j < K; ++j)
        mul_all<H>(t, f[j]);
    for (unsigned q = K; q < cnt; q += D) {
        float g[D][H];
        factors<S, H, D, CLEAN>(msgs + q * S, cnt - q, g);
#pragma unroll
        for (int j = 0; j < D; ++j)
            mul_all<H>(t, g[j]);
    }
    mul_all<H>(st, t);
    if constexpr (H < S)
        normalise_quad(st, h, n);
    else
        normalise<S, MIXED>(st, n);
#pragma unroll
    for (int i = 0; i < H; ++i)
        b[i] = st[i];
#pragma unroll
    for (int j = 0; j < K; ++j)
        mul_all<H>(b, f[j]);
    for (unsigned q = K; q < cnt; q += D) {
        float g[D][H];
        factors<S, H, D, CLEAN>(msgs + q * S, cnt - q, g);
#pragma unroll
        for (int j = 0; j < D; ++j)
            mul_all<H>(b, g[j]);
    }
}

/* NS slots per thread. */
template <int S, bool MIXED, int NS, bool SINGLE, bool DELTA>
__global__ __launch_bounds__(RB) void k_resident(ResArgs a)
{
    constexpr int SP = Stride<S>::value;
    constexpr int LN = LanesPerNode<S>::value, NN = NodeRounds<S, NS>::value;
    constexpr int H = S / LN, HP = LN > 1 ? H : SP; /* a lane's entries of a node, and of its row */
    constexpr int RN = RB / LN;                     /* nodes of a round */
    constexpr int W = RB * NS;
    /* messages by slot: iteration t's in lm[t & 1] (while the tables are
     * loaded, a staging area) */
    __shared__ __align__(16) float lm[2][S * (W + PAD)];
    __shared__ __align__(16) float lbuf[SINGLE ? SP * RN * NN : 4];
    __shared__ double red[2][RW];
    __shared__ double total;
    __shared__ unsigned ok, committed, suspect;
    const unsigned tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const unsigned G = gridDim.x, wg = SINGLE ? 0u : xcd_block(blockIdx.x, G);
    if (!SINGLE && called_off(a.meeting))
        return;
    const unsigned n0 = a.wg_node[wg], n1 = a.wg_node[wg + 1];
    const unsigned s0 = a.in_off[n0], ns = a.in_off[n1] - s0;
    if (tid == 0)
        suspect = 0;

    /* what stays: tables, sources (with the state counts in the top byte:
     * node numbers are at most 2^20 here), places in LDS.  Threads past the
     * last slot repeat it and put its message into the padding. */
    float J[NS][S * S];
    unsigned src[NS], at[(NS + 1) / 2]; /* two places to a register */
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        src[k] = n0;
        if (k % 2 == 0)
            at[k / 2] = 0;
        if (k * RB + wave * WAVE >= ns)
            continue; /* the wave has no slot in this turn */
        const unsigned l = k * RB + tid, q = a.wg_slots[(size_t)wg * W + (l < ns ? l : ns - 1)];
        const unsigned s = s0 + q;
        at[k / 2] = k % 2 ? (at[k / 2] & 0xffffu) | q << 16 : q;
        src[k] = a.slot_src[s];
        if constexpr (MIXED)
            src[k] |= (unsigned)a.slot_xy[s] << 24;
    }
    /* tables by way of LDS, a row (S = 2: both rows) of all slots at a time:
     * read in slot order, handed out in source order */
    constexpr int CH = S == 2 ? 4 : S; /* floats of a slot's table at a time */
#pragma unroll
    for (int c = 0; c < S * S / CH; ++c) {
        float *stage = lm[0];
        for (unsigned l = tid; l < ns; l += RB) {
            const unsigned s = s0 + l;
            float t[CH];
            if (MIXED && (S < 8 || a.slot_tab)) {
                load_row<CH>(a.J + a.slot_tab[s] + c * (int)mixed_row_stride(S), t);
            } else if (MIXED) { /* one state count of 5 to 8 on the 8-state kernel */
                const unsigned n = a.S;
                const float *T = a.J + ((size_t)s * n + c) * n;
#pragma unroll
                for (int j = 0; j < CH; ++j)
                    t[j] = (unsigned)c < n && (unsigned)j < n ? T[j] : 0.0f;
            } else {
                load_row<CH>(a.J + (size_t)s * S * S + c * CH, t);
            }
            put_row<CH>(stage + l * CH, t);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (k * RB + wave * WAVE < ns)
                get_row<CH>(stage + (k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu) * CH, J[k] + c * CH);
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NS; ++k) /* threads past the last slot */
        if (k * RB + tid >= ns)
            at[k / 2] = k % 2 ? (at[k / 2] & 0xffffu) | (unsigned)W << 16 : (at[k / 2] & 0xffff0000u) | W;
    if (DELTA) /* the old messages, to their own slots' places */
        for (unsigned l = tid; l < ns; l += RB) {
            float old[S];
            load_rowp<S, SP>(a.msg0 + (size_t)(s0 + l) * SP, old);
            put_row<S>(lm[0] + l * S, old);
        }
    const unsigned h = tid % LN; /* which entries of its nodes the lane has: from h * H on */
    float st[NN][H];
    unsigned slots[NN], nn[NN]; /* first in-slot | in-degree << 16 (both below 2^16) */
#pragma unroll
    for (int r = 0; r < NN; ++r) {
        const unsigned v = n0 + r * RN + tid / LN;
        slots[r] = 0;
        nn[r] = S;
#pragma unroll
        for (int i = 0; i < H; ++i)
            st[r][i] = 1.0f;
        if (v < n1) {
            const unsigned b = a.in_off[v], e = a.in_off[v + 1];
            slots[r] = (b - s0) | (e - b) << 16;
            if (MIXED)
                nn[r] = a.nvars[v];
            load_rowp<H, HP>(a.states + (size_t)v * SP + h * H, st[r]);
            if constexpr (SINGLE) {
                float b0[H];
                load_rowp<H, HP>(a.buf_in + (size_t)v * SP + h * H, b0);
#pragma unroll
                for (int i = 0; i < H; ++i)
                    lbuf[v * SP + h * H + i] = b0[i];
            }
        }
    }
    if constexpr (SINGLE) {
        __syncthreads();
    } else {
        if (!grid_step(a.meeting, wg, G, 1, &ok)) /* everybody is here */
            return;
    }

    double previous = a.previous, before = a.previous;
    unsigned ran = 0, stopped = 0;
    for (;;) {
        hold(at);
        hold(slots);
        if (MIXED)
            hold(src);
        const float *in = SINGLE ? lbuf : ran == 0 ? a.buf_in : a.ring + (size_t)(ran - 1) * a.ring_stride;
        float bsrc[NS][S];
        if (ran < a.n) {
#pragma unroll
            for (int k = 0; k < NS; ++k)
                load_rowp<S, SP>(in + (size_t)(MIXED ? src[k] & 0xffffffu : src[k]) * SP, bsrc[k]);
        }
        if (DELTA && a.until && ran > 0) {
            /* the stop test on the iteration just done, while the gathers
             * are under way; every workgroup adds the same partials in the
             * same order */
            double sum = 0.0;
            if constexpr (SINGLE) {
#pragma unroll
                for (int w = 0; w < RW; ++w)
                    sum += red[(ran - 1) & 1][w];
            } else {
                if (wave == 0) {
                    for (unsigned i = lane; i < G; i += WAVE)
                        sum += __hip_atomic_load(a.parts + ((ran - 1) & 1) * MAX_G + i, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
                    sum = wave_sum(sum);
                    if (lane == 0)
                        total = sum;
                }
                __syncthreads();
                sum = total;
            }
            before = previous;
            previous = sum;
            double change = sum - before;
            if (change < 0.0)
                change = -change;
            if (sum < (double)a.conv || change < (double)a.conv) {
                stopped = 1;
                break;
            }
        }
        if (ran == a.n)
            break;
        const float *lold = lm[ran & 1];
        float *lnew = lm[(ran & 1) ^ 1];
        double dacc = 0.0;
        bool odd = false; /* a message that may hold NaN */
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (k * RB + wave * WAVE >= ns)
                continue;
            const unsigned x = MIXED ? src[k] >> 24 & 15u : (unsigned)S, y = MIXED ? src[k] >> 28 : (unsigned)S;
            const unsigned place = k % 2 ? at[k / 2] >> 16 : at[k / 2] & 0xffffu;
            float m[S], sum;
            if constexpr (MIXED)
                sum = send_padded<S>(J[k], bsrc[k], x, y, m);
            else
                sum = send<S, false>(J[k], bsrc[k], S, S, m);
            odd = odd || !(fabsf(sum) < INFINITY);
            if (DELTA) {
                float old[S];
                get_row<S>(lold + place * S, old);
                double d = 0.0;
#pragma unroll
                for (int i = 0; i < S; ++i)
                    if (!MIXED || (unsigned)i < x) {
                        float q = old[i] - m[i];
                        if (q != q)
                            q = 0.0f;
                        d += (double)fabsf(q);
                    }
                dacc += k * RB + tid < ns ? d : 0.0;
            }
            put_row<S>(lnew + place * S, m);
        }
        if (__ballot(odd) != 0 && lane == 0)
            suspect = ran + 1;
        if (DELTA) {
            dacc = wave_sum(dacc);
            if (lane == 0)
                red[ran & 1][wave] = dacc;
        }
        __syncthreads();
        const bool clean = __builtin_amdgcn_readfirstlane(suspect) == ran + 1;
        if (DELTA && wave == RW - 1 && (!SINGLE || !a.until)) {
            /* the wave with the fewest nodes adds up the workgroup's delta */
            static_assert(RW == 16, "a row of lanes");
            const double sum = row_sum(red[ran & 1][lane % RW]);
            if (lane == 0) {
                if (!a.until)
                    a.partials[(size_t)ran * G + wg] = sum;
                else
                    __hip_atomic_store(a.parts + (ran & 1) * MAX_G + wg, sum, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int r = 0; r < NN; ++r) {
            if (r * RN + wave * (WAVE / LN) >= n1 - n0)
                continue;
            const unsigned v = n0 + r * RN + tid / LN;
            if (v < n1) { /* all lanes of a node or none */
                const float *msgs = lnew + (slots[r] & 0xffffu) * S + h * H;
                const unsigned cnt = slots[r] >> 16, n = nn[r];
                float b[H];
                if (clean)
                    resident_node<S, MIXED, NS, true, H>(msgs, cnt, n, h, st[r], b);
                else
                    resident_node<S, MIXED, NS, false, H>(msgs, cnt, n, h, st[r], b);
                float row[HP];
#pragma unroll
                for (int i = 0; i < HP; ++i)
                    row[i] = (i < H && (!MIXED || h * H + i < n)) ? b[i] : 0.0f;
                const size_t to = (size_t)ran * a.ring_stride + (size_t)v * SP + h * H;
                if constexpr (SINGLE) {
#pragma unroll
                    for (int i = 0; i < H; ++i)
                        lbuf[v * SP + h * H + i] = row[i];
                    if (a.keep)
                        store_row_nt<HP>(a.ring + to, row);
                } else {
                    store_row_agent<HP>(a.ring + to, row);
                }
                if (a.keep) {
#pragma unroll
                    for (int i = 0; i < HP; ++i)
                        row[i] = (i < H && (!MIXED || h * H + i < n)) ? st[r][i] : 0.0f;
                    store_row_nt<HP>(a.keep + to, row);
                }
            }
        }
        ++ran;
        if constexpr (SINGLE) {
            __syncthreads();
        } else {
            if (!grid_step(a.meeting, wg, G, ran + 1, &ok))
                return;
        }
    }

    if constexpr (!SINGLE) {
        if (tid == 0)
            committed = settle(a.meeting.decision, a.meeting.run, COMMIT);
        __syncthreads();
        if (!committed)
            return;
    }
    if (a.keep)
        return;
    /* results: beliefs, the combine buffers of the next iteration, the last
     * two iterations' messages */
    float *newest = ran & 1 ? a.msg1 : a.msg0, *older = ran & 1 ? a.msg0 : a.msg1;
    for (unsigned l = tid; l < ns; l += RB) {
        float m[S], row[SP];
        get_row<S>(lm[ran & 1] + l * S, m);
#pragma unroll
        for (int i = 0; i < SP; ++i)
            row[i] = i < S ? m[i] : 0.0f;
        store_row_nt<SP>(newest + (size_t)(s0 + l) * SP, row);
        if (ran > 1) { /* after one iteration they are in place */
            get_row<S>(lm[(ran & 1) ^ 1] + l * S, m);
#pragma unroll
            for (int i = 0; i < SP; ++i)
                row[i] = i < S ? m[i] : 0.0f;
            store_row_nt<SP>(older + (size_t)(s0 + l) * SP, row);
        }
    }
#pragma unroll
    for (int r = 0; r < NN; ++r) {
        const unsigned v = n0 + r * RN + tid / LN;
        if (v < n1) {
            const size_t at_row = (size_t)v * SP + h * H;
            float row[HP];
#pragma unroll
            for (int i = 0; i < HP; ++i)
                row[i] = (i < H && (!MIXED || h * H + i < nn[r])) ? st[r][i] : 0.0f;
            store_row_nt<HP>(a.states + at_row, row);
            if constexpr (SINGLE) {
#pragma unroll
                for (int i = 0; i < HP; ++i)
                    row[i] = i < H ? lbuf[at_row + i] : 0.0f;
            } else {
                load_row<HP>(a.ring + (size_t)(ran - 1) * a.ring_stride + at_row, row);
            }
            store_row_nt<HP>(a.buf_out + at_row, row);
        }
    }
    if (tid == 0 && wg == 0) {
        a.status->ran = ran;
        a.status->stopped = stopped;
        a.status->last = previous;
        a.status->before = before;
        __hip_atomic_store(&a.status->run, a.meeting.run, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

} // namespace

/* ------------------------------------------------------------------------ */
/* host side                                                                 */

namespace {

/* Slots per thread that the registers (128 per thread) and LDS (two
 * iterations' messages) hold. */
unsigned most_slots(unsigned S) { return S == 2 ? 8 : S == 3 ? 4 : S == 4 ? 3 : 1; }

/* slots per thread go 1, 2, 4, 8; for three and four states 1, 2, 3, 4 */
unsigned next_slots(unsigned ns, unsigned S) { return S > 2 && ns >= 2 ? ns + 1 : 2 * ns; }

/* Most workgroups of a plan with ns slots per thread.  All CUs: fewer slots
 * per thread are worth more than the barrier among more workgroups costs
 * (1.25 us among 64, 1.4 among 256).  Per iteration, us, at most 64 ns
 * workgroups / all: 100k binary nodes 5.47 / 5.00, 20k nodes of 3 states
 * 4.11 / 3.90, 100k nodes of 2-4 states 7.15 / 6.63; gradients, a backward
 * of 31 steps: 20k nodes of 3 states 457 / 330, 120k 782 / 602.  Binary
 * networks with a slot per thread have too little to do: 40k nodes 3.79 /
 * 3.87 and with the stop test 5.05 / 5.26, 60k 4.29 / 4.50 and 5.59 / 6.05,
 * so half the CUs there, except for gradients (40k nodes 311 / 233). */
unsigned most_groups(unsigned ns, unsigned S, bool gradients, unsigned cus)
{
    const unsigned full = std::min(cus, MAX_G);
    return S == 2 && ns == 1 && !gradients ? (full + 1) / 2 : full;
}

/* Largest network of one workgroup, in slots per thread: messages and
 * combine buffers share 160 KB of LDS. */
unsigned single_slots(unsigned S) { return S == 2 ? 4 : S <= 4 ? 2 : 1; }

unsigned most_nodes(unsigned ns, unsigned S) { return S > 4 ? RB / 2 : (ns + 1) / 2 * RB; }

/* Workgroup ranges: consecutive nodes with at most `slots` in-slots and
 * `nodes` nodes, cut at multiples of `align` nodes.  Empty when a node group
 * does not fit. */
bool cut_ranges(const std::vector<unsigned> &in_off, unsigned V, unsigned slots, unsigned nodes, unsigned align,
                std::vector<unsigned> &first)
{
    first.assign(1, 0);
    unsigned v = 0;
    while (v < V) {
        unsigned b = v;
        while (v < V) {
            unsigned e = std::min(V, (v / align + 1) * align);
            if (in_off[e] - in_off[b] > slots || e - b > nodes)
                break;
            v = e;
        }
        if (v == b)
            return false;
        first.push_back(v);
    }
    return first.size() > 1;
}

/* Each workgroup's slots in order of their source, `per` places for each
 * workgroup.  Sorted by digits of 11 bits: comparisons took 45 us for the
 * thousand slots of a workgroup, half a millisecond more to upload a network
 * of 5,000 nodes. */
void deal_slots(const std::vector<unsigned> &in_off, const std::vector<unsigned> &slot_src,
                const std::vector<unsigned> &first, unsigned per, std::vector<unsigned short> &order)
{
    const unsigned G = (unsigned)first.size() - 1;
    order.assign((size_t)G * per, 0);
    auto deal = [&](unsigned w0, unsigned w1) {
        constexpr unsigned BITS = 11, DIGITS = 1u << BITS;
        std::vector<uint64_t> key, next;
        unsigned count[DIGITS];
        for (unsigned w = w0; w < w1; ++w) {
            const unsigned s0 = in_off[first[w]], s1 = in_off[first[w + 1]];
            uint64_t bits = 0;
            key.resize(s1 - s0);
            next.resize(s1 - s0);
            for (unsigned s = s0; s < s1; ++s) {
                key[s - s0] = (uint64_t)slot_src[s] << 16 | (s - s0);
                bits |= slot_src[s];
            }
            for (unsigned shift = 16; bits; shift += BITS, bits >>= BITS) {
                std::fill_n(count, DIGITS, 0u);
                for (uint64_t x : key)
                    ++count[x >> shift & (DIGITS - 1)];
                unsigned at = 0;
                for (unsigned &c : count) {
                    const unsigned n = c;
                    c = at;
                    at += n;
                }
                for (uint64_t x : key)
                    next[count[x >> shift & (DIGITS - 1)]++] = x;
                key.swap(next);
            }
            for (unsigned i = 0; i < key.size(); ++i)
                order[(size_t)w * per + i] = (unsigned short)key[i];
        }
    };
    par_for(G, std::max<size_t>(1, 8192 / (slot_src.size() / G + 1)),
            [&](size_t a, size_t b) { deal((unsigned)a, (unsigned)b); });
}

/* One resident launch at a time per device: the launches of two streams,
 * each partly on the chip, would wait for each other.  A launch on another
 * stream than the last one waits for an event behind that one.
 *
 * If the last stream is a handle's, which lives until bp_resident_free, the
 * event is recorded by the launch that needs it: recorded behind every launch
 * it took 1 to 5 us of each call (10 iterations of 5,000 nodes with deltas
 * and beliefs read back 73 / 78 us, 500k nodes 321 / 326).  The stream's
 * owner may be another thread, so captures on a handle's stream are made
 * under the same lock: an event recorded in one would become part of it, and
 * so would the launch that waits for it.
 *
 * A caller's stream may be in capture or gone by then: its event is recorded
 * with the launch, and every launch waits for it, since equal values do not
 * say that it is the same stream (hipStreamPerThread is one value for all
 * threads, and that of a destroyed stream is given out again). */
constexpr int MAX_DEVICES = 64;
std::mutex turn_mu;
struct {
    bool any, foreign; /* foreign: on a caller's stream */
    hipStream_t last;
    hipEvent_t ev; /* behind the last launch; created with the device's first plan */
} turn[MAX_DEVICES];

template <int S, bool MIXED, int NS, bool SINGLE>
void launch_d(const ResArgs &a, unsigned G, bool delta, hipStream_t st)
{
    if (delta)
        hipLaunchKernelGGL((k_resident<S, MIXED, NS, SINGLE, true>), dim3(G), dim3(RB), 0, st, a);
    else
        hipLaunchKernelGGL((k_resident<S, MIXED, NS, SINGLE, false>), dim3(G), dim3(RB), 0, st, a);
}

template <int S, bool MIXED>
void launch_s(const ResArgs &a, unsigned ns, unsigned G, bool single, bool delta, hipStream_t st)
{
    if (single) {
        if (ns == 1)
            launch_d<S, MIXED, 1, true>(a, 1, delta, st);
        else if (ns == 2)
            launch_d<S, MIXED, 2, true>(a, 1, delta, st);
        else if constexpr (S == 2)
            launch_d<S, MIXED, 4, true>(a, 1, delta, st);
        return;
    }
    if (ns == 1)
        launch_d<S, MIXED, 1, false>(a, G, delta, st);
    else if (ns == 2)
        launch_d<S, MIXED, 2, false>(a, G, delta, st);
    if constexpr (S > 2)
        if (ns == 3)
            launch_d<S, MIXED, 3, false>(a, G, delta, st);
    if constexpr (S < 4)
        if (ns == 4)
            launch_d<S, MIXED, 4, false>(a, G, delta, st);
    if constexpr (S == 2)
        if (ns == 8)
            launch_d<S, MIXED, 8, false>(a, G, delta, st);
}

void launch(unsigned S, bool mixed, const ResArgs &a, unsigned ns, unsigned G, bool single, bool delta,
            hipStream_t st)
{
    if (S > 4) /* 5 to 8 states: rows are 8 floats apart in every case */
        single ? launch_d<8, true, 1, true>(a, 1, delta, st) : launch_d<8, true, 1, false>(a, G, delta, st);
    else if (S == 2)
        launch_s<2, false>(a, ns, G, single, delta, st);
    else if (S == 3)
        mixed ? launch_s<3, true>(a, ns, G, single, delta, st) : launch_s<3, false>(a, ns, G, single, delta, st);
    else
        mixed ? launch_s<4, true>(a, ns, G, single, delta, st) : launch_s<4, false>(a, ns, G, single, delta, st);
}

} // namespace

std::mutex &bp_resident_mutex() { return turn_mu; }

int bp_resident_turn(int device, hipStream_t stream)
{
    const auto &t = turn[device];
    if (t.any && (t.foreign || t.last != stream)) {
        if (!t.foreign)
            HIP_TRY(hipEventRecord(t.ev, t.last));
        HIP_TRY(hipStreamWaitEvent(stream, t.ev, 0));
    }
    return 0;
}

int bp_resident_turn_taken(int device, hipStream_t stream, bool foreign)
{
    auto &t = turn[device];
    t.any = true;
    t.foreign = foreign;
    t.last = stream;
    if (foreign)
        HIP_TRY(hipEventRecord(t.ev, stream));
    return 0;
}

Meeting bp_resident_meeting(bp_dev *d, unsigned barriers, unsigned after)
{
    bp_resident &r = d->res;
    Meeting m;
    m.counters = r.counters;
    m.met = r.met;
    m.decision = r.counters + COUNTERS * COUNTER_STRIDE;
    m.after = after;
    r.run = (r.run + 1) & 0x7fffffffu;
    m.run = r.run;
    m.timeout = r.timeout;
    r.met += barriers;
    return m;
}

/* Decides whether the graph runs resident and lays out its ranges:
 * uniform state counts of 2 to 8, or mixed ones up to 3 to 8. */
int bp_resident_plan(bp_dev *d, const std::vector<unsigned> &slot_src, bool gradients, int cus)
{
    bp_resident &r = d->res;
    if (d->E == 0 || d->S < 2 || d->S > 8 || (d->mixed && d->S == 2) || d->device >= MAX_DEVICES)
        return 0;
    std::vector<unsigned> first;
    const unsigned align = 32 / d->SP; /* nodes per 128-byte line */
    for (unsigned ns = 1; ns <= single_slots(d->S) && !r.ns; ns *= 2)
        if (d->E <= ns * RB && d->V <= most_nodes(ns, d->S)) {
            r.ns = ns;
            r.single = true;
            first = {0, d->V};
        }
    for (unsigned ns = 1; ns <= most_slots(d->S) && !r.ns; ns = next_slots(ns, d->S)) {
        /* even ranges: the slots spread over as many workgroups as the cap
         * asks for, a few per cent more where node groups do not fit */
        const unsigned cap = ns * RB, full = cap * 31 / 32, groups = most_groups(ns, d->S, gradients, (unsigned)cus);
        const unsigned want = (d->E + full - 1) / full;
        const unsigned even = std::min(cap, (d->E + want - 1) / want + cap / 32);
        if (want <= groups && cut_ranges(d->in_off_h, d->V, even, most_nodes(ns, d->S), align, first) &&
            first.size() - 1 <= groups)
            r.ns = ns;
    }
    if (!r.ns)
        return 0;
    r.G = (unsigned)first.size() - 1;
    r.limit = d->part_cap;
    /* one device allocation, the parts that are copied there first:
     * counters and decision (zero), ranges, dealt slots; then the delta
     * partials of the stop test and the ring */
    std::vector<unsigned short> order;
    deal_slots(d->in_off_h, slot_src, first, r.ns * RB, order);
    const size_t words = COUNTERS * COUNTER_STRIDE + COUNTER_STRIDE;
    std::vector<unsigned> head(words + first.size() + (order.size() + 1) / 2, 0u);
    std::copy(first.begin(), first.end(), head.begin() + words);
    std::memcpy(head.data() + words + first.size(), order.data(), order.size() * sizeof(unsigned short));
    const size_t parts_at = (head.size() * 4 + 127) / 128 * 128, ring_at = parts_at + 2 * MAX_G * sizeof(double);
    size_t bytes = ring_at;
    if (!r.single) {
        /* a place per iteration of a launch: 8 MB of them, 32 at least */
        r.ring_stride = ((size_t)d->V * d->SP + 31) / 32 * 32;
        r.limit = std::min<size_t>(r.limit, std::min<size_t>(256, std::max<size_t>(32, (8u << 20) / (4 * r.ring_stride))));
        bytes += r.ring_stride * r.limit * sizeof(float);
    }
    {
        std::lock_guard<std::mutex> lock(turn_mu);
        if (!turn[d->device].ev)
            HIP_TRY(hipEventCreateWithFlags(&turn[d->device].ev, hipEventDisableTiming));
    }
    int khz = 0;
    HIP_TRY(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, d->device));
    r.timeout = (unsigned long long)khz * 1000; /* a second */
    HIP_TRY(hipMalloc((void **)&r.memory, bytes));
    if (copy_on(d->stream, r.memory, head.data(), head.size() * sizeof(unsigned), hipMemcpyHostToDevice))
        return -1;
    r.counters = (unsigned *)r.memory;
    r.wg_node = r.counters + words;
    r.wg_slots = (unsigned short *)(r.wg_node + first.size());
    r.parts = (double *)(r.memory + parts_at);
    r.ring = (float *)(r.memory + ring_at);
    r.on = true;
    return 0;
}

void bp_resident_free(bp_dev *d)
{
    bp_resident &r = d->res;
    {
        std::lock_guard<std::mutex> lock(turn_mu);
        if (d->stream && d->device < MAX_DEVICES && !turn[d->device].foreign && turn[d->device].last == d->stream)
            turn[d->device].any = false; /* the stream has been waited for */
    }
    if (r.memory)
        (void)hipFree(r.memory);
    r = bp_resident();
}

/* Enqueues up to n (<= res.limit) iterations: with want_delta their deltas
 * go to the status's deltas, and with `until` the stop test ends the run.  ev
 * (nullable): events before and after the kernel. */
int bp_resident_launch(bp_dev *d, unsigned n, bool want_delta, bool until, float conv, double previous,
                       double *partials, const hipEvent_t *ev)
{
    bp_resident &r = d->res;
    ResArgs a;
    a.in_off = d->in_off;
    a.slot_src = d->slot_src;
    a.slot_xy = d->slot_xy;
    a.nvars = d->nvars;
    a.J = d->J;
    a.slot_tab = d->mixed ? d->slot_toff : nullptr;
    a.S = d->S;
    a.keep = nullptr;
    a.wg_node = r.wg_node;
    a.wg_slots = r.wg_slots;
    a.states = d->states;
    a.buf_in = d->buf[d->bcur];
    a.buf_out = d->buf[d->bcur ^ 1];
    a.msg0 = d->msg[d->latest];
    a.msg1 = d->msg[d->latest ^ 1];
    a.ring = r.ring;
    a.ring_stride = r.ring_stride;
    a.n = n;
    a.until = until;
    a.conv = conv;
    a.previous = previous;
    /* one workgroup: its partial is the delta */
    a.partials = r.single ? d->status()->deltas : partials;
    a.parts = r.parts;
    /* with the stop test bp_resident_ran says how many barriers there were */
    a.meeting = bp_resident_meeting(d, until || r.single ? 0 : n + 1, r.npending ? r.pending[r.npending - 1].run : 0u);
    a.status = d->status();
    if (r.single) {
        if (ev)
            HIP_TRY(hipEventRecord(ev[0], d->stream));
        launch(d->S, d->mixed, a, r.ns, 1, true, want_delta || until, d->stream);
        if (ev)
            HIP_TRY(hipEventRecord(ev[1], d->stream));
    } else {
        std::lock_guard<std::mutex> lock(turn_mu);
        if (bp_resident_turn(d->device, d->stream))
            return -1;
        if (ev)
            HIP_TRY(hipEventRecord(ev[0], d->stream));
        launch(d->S, d->mixed, a, r.ns, r.G, false, want_delta || until, d->stream);
        if (ev)
            HIP_TRY(hipEventRecord(ev[1], d->stream));
        if (bp_resident_turn_taken(d->device, d->stream, false))
            return -1;
    }
    if (want_delta && !until && !r.single)
        bp_launch_finish(partials, r.G, n, d->status()->deltas, d->stream);
    HIP_TRY(hipGetLastError());
    return 0;
}

/* The unrolled forward of the adjoint: K iterations from the beliefs st[0]
 * and combine buffers buf[0] to st[1..K] and buf[1..K], rows of a `stride`
 * each, on a caller's stream.  A run that is given up leaves them to
 * k_forward_rescue (bp_resident_diff.hip). */
int bp_resident_forward(bp_dev *d, unsigned K, float *st, float *buf, size_t stride, hipStream_t stream,
                        Meeting *meeting)
{
    bp_resident &r = d->res;
    ResArgs a = {};
    a.in_off = d->in_off;
    a.slot_src = d->slot_src;
    a.slot_xy = d->slot_xy;
    a.nvars = d->nvars;
    a.J = d->J;
    a.wg_node = r.wg_node;
    a.wg_slots = r.wg_slots;
    a.S = d->S;
    a.states = st;
    a.buf_in = buf;
    a.ring = buf + stride;
    a.keep = st + stride;
    a.ring_stride = stride;
    a.n = K;
    a.parts = r.parts;
    a.meeting = bp_resident_meeting(d, r.single ? 0 : K + 1, r.single ? 0 : r.settled);
    if (!r.single)
        r.settled = r.run;
    a.status = d->status();
    *meeting = a.meeting;
    launch(d->S, d->mixed, a, r.ns, r.G, r.single, false, stream);
    HIP_TRY(hipGetLastError());
    return 0;
}

/* After the stream has been waited for: whether the last launch went
 * through. */
bool bp_resident_ran(bp_dev *d, bool until)
{
    bp_resident &r = d->res;
    const bool ran = r.single || d->status()->run == r.run;
    if (ran && until && !r.single)
        r.met += d->status()->ran + 1;
    return ran;
}

/* Ticks of the wall clock that the workgroups of a resident run wait for
 * each other; returns the previous setting.  With 0 a run is given up at its
 * first wait and its iterations run with a launch each. */
extern "C" unsigned long long bp_resident_set_timeout(bp_dev *d, unsigned long long ticks)
{
    unsigned long long before = d->res.timeout;
    d->res.timeout = ticks;
    return before;
}

/* Slots per thread of the handle's resident runs (0: it runs a launch per
 * iteration) and their workgroups. */
extern "C" unsigned bp_resident_shape(const bp_dev *d, unsigned *workgroups)
{
    *workgroups = d->res.on ? d->res.G : 0;
    return d->res.on ? d->res.ns : 0;
}
