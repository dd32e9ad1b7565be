/*
 * bp_diff.hip -- differentiable loopy BP: the parameter -> table map, the
 * unrolled forward with checkpoints, and the hand-written adjoint.
 *
 * Parameters are the TABLEs of a network's CPT definitions.  k_set_params
 * rebuilds every slot's pairwise table from them with the XMLBIF reader's
 * loop (src/bnf-xml-parser/xml-expression.c:384-400, restated in
 * bp_model.c): for parent state j and child state k, the sequential f32 sum
 * of the TABLE entries in the blocks of that parent's state, so the tables
 * are bit-identical to the reader's.  It also puts root priors into the
 * initial beliefs, as graph_set_node_state does (xml-expression.c:290-317).
 *
 * The forward is the loopy kernel in its FWD/FINIT modes: the node-centric
 * iteration of src/graph/graph.c:1121-1183 from init_previous_edge
 * (graph.c:725-751), writing every iterate to the buffer it is given.
 *
 * Adjoint of one iteration t (k_adjoint, one launch over chunks of its own:
 * consecutive nodes with at most 64 x R in-slots).  In exact arithmetic, with N(x) = x / sum(x):
 *   m_t[s]  = N(z_s), z_s = J_s . buf_{t-1}[u],  u = src(s)
 *   T_t[v]  = prod_{s in in(v)} m_t[s]
 *   st_t[v] = N(a_v), a_v = st_{t-1}[v] (.) T_t[v]   (a_v = st_{t-1}[v] without in-edges)
 *   buf_t[v]= st_t[v] (.) T_t[v]
 * Given dst_t (from the loss or iteration t+1) and dbuf_t[v] =
 * sum_{s: src(s)=v} w_{t+1}[s]:
 *   dst_t   += dbuf_t (.) T_t          dT = dbuf_t (.) st_t
 *   da       = (dst_t - <dst_t, st_t>) / sum(a)   (identity when sum(a) <= 0,
 *              where the forward divides by 1)
 *   dst_{t-1} = da (.) T_t,  dT += da (.) st_{t-1}
 *   dm_s     = dT (.) prod_{s' in in(v), s' != s} m_t[s']
 *   dz_s     = (dm_s - <dm_s, m_s>) / sum(z_s)
 *   dJ_s    += dz_s (x) buf_{t-1}[u],  w_t[s] = J_s^T dz_s
 * Step 0 (init) has m_0 from st_0 and buf_0 = st_0 (.) T_0; its w_0 and
 * dbuf_0 (.) T_0 add to dst_0.  Sums over a node's out-edges are gathers in
 * slot order through a source-grouped slot list, so results do not depend
 * on scheduling (no atomics).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <vector>

#include "bp_adjoint.h"
#include "bp_resident.h"
#include "../../include/bp_diff.h"

using namespace bpk;

namespace {

constexpr unsigned NONE = 0xffffffffu;

struct ParentRec {
    unsigned offset, n_par, slot_f, slot_r;
};

__global__ void k_copy(const float *__restrict__ src, float *__restrict__ dst, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        dst[i] = src[i];
}

/* The parameter kernels' share of work: whole definitions, whose tables fit
 * in LDS together, or (BIG) some rows of one that is larger. */
struct Piece {
    unsigned def0, ndefs, row0, row1;
};
constexpr unsigned BIG = 0x80000000u;       /* in ndefs */
constexpr unsigned PIECE_FLOATS = 4608;     /* table entries of a piece, or its parents' gradient entries */
constexpr unsigned PIECE_DEFS = 128;
constexpr int PIECE_THREADS = 256;

struct DefInfo {
    unsigned tb, slice, pbegin, pend, prior, rbegin; /* rbegin: the definition's first softmax row */
    unsigned at;                                     /* its table's place in LDS; rows of slice | 1 floats */
    unsigned pad;
};

/* A pairwise table entry: the sequential f32 sum of the TABLE entries of one
 * child state whose configurations have the parent in one state, in
 * ascending order -- the blocks of the reader's loop, in its order.  p is the
 * first of them; `count` (a power of S, as every node has S states) lie in
 * runs of `o`, one run in every o * S.  They are taken S at a time, which
 * are S apart for o = 1 and adjacent otherwise, so that the place is carried
 * along once per S entries; U times S loads are issued ahead of their adds. */
template <int S, int U> __device__ __forceinline__ float table_sum(const float *p, unsigned count, unsigned o)
{
    float acc = 0.0f;
    if (count < (unsigned)S || S == 1) {
        acc += *p;
        return acc;
    }
    const unsigned apart = o == 1 ? S : 1, run = o == 1 ? 1 : o / S, step = o == 1 ? 0 : S;
    const unsigned jump = o == 1 ? S * S : o * (S - 1), groups = count / S;
    unsigned left = run;
    for (unsigned g = 0; g < groups; g += U) {
        float v[U][S];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < S; ++i)
                v[u][i] = p[i * apart];
            if (g + u + 1 < groups) {
                p += step;
                if (--left == 0) {
                    left = run;
                    p += jump;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (g + u < groups)
#pragma unroll
                for (int i = 0; i < S; ++i)
                    acc += v[u][i];
    }
    return acc;
}

template <int S>
__device__ __forceinline__ void put_table_entry(float *J, const ParentRec &rec, unsigned k, unsigned j, float x)
{
    J[(size_t)rec.slot_f * (S * S) + j * S + k] = x;
    if (rec.slot_r != NONE)
        J[(size_t)rec.slot_r * (S * S) + k * S + j] = x;
}

/* Parameters to tables and initial beliefs.  P is theta, or (LOG) its
 * softmax over each row (a definition's child states under one parent
 * configuration); J_fwd[j][k] of each parent record is table_sum's, written
 * to the forward slot and, transposed, to the reverse slot; a root's prior
 * becomes its initial belief.
 *
 * Bound by reading theta and writing P once each.  P stays in LDS between
 * the two halves: sums that read it from memory eight entries at a time were
 * chains of a dozen and more round trips for a node with six parents (210k
 * definitions of 3 states, 21.6M parameters: softmax 71 us, sums 129, priors
 * 4; now 72 in all, 2.6 TB/s of theta, P and tables).  A row per thread, four at a time: consecutive threads read
 * consecutive floats, in runs of a definition's slice; its rows are an odd
 * number of floats apart in LDS, or all child states of a table would share
 * a bank for two and four states. */
template <int S, bool LOG>
__global__ __launch_bounds__(PIECE_THREADS) void k_set_params(const float *__restrict__ theta,
                                                              const Piece *__restrict__ pieces,
                                                              const DefInfo *__restrict__ defs,
                                                              const unsigned short *__restrict__ row_def,
                                                              const ParentRec *__restrict__ parents,
                                                              const unsigned *__restrict__ par_def,
                                                              float *__restrict__ P, float *__restrict__ J,
                                                              float *__restrict__ st0, unsigned SP)
{
    constexpr int U = S <= 4 ? 4 : 1;
    constexpr unsigned SS = (unsigned)S * S;
    __shared__ float table[PIECE_FLOATS];
    __shared__ DefInfo def[PIECE_DEFS];
    const Piece c = pieces[blockIdx.x];
    const unsigned nd = c.ndefs & ~BIG, tid = threadIdx.x;
    const bool big = c.ndefs & BIG;
    for (unsigned d = tid; d < nd; d += PIECE_THREADS)
        def[d] = defs[c.def0 + d];
    __syncthreads();
    for (unsigned r0 = c.row0 + tid; r0 < c.row1; r0 += U * PIECE_THREADS) {
        float v[U][S];
        unsigned first[U], slice[U], at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            unsigned r = r0 + u * PIECE_THREADS;
            r = r < c.row1 ? r : r0;
            const DefInfo &di = def[row_def[r]];
            slice[u] = di.slice;
            first[u] = di.tb + (r - di.rbegin);
            at[u] = di.at + (r - di.rbegin);
#pragma unroll
            for (int k = 0; k < S; ++k)
                v[u][k] = theta[first[u] + k * slice[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (r0 + u * PIECE_THREADS >= c.row1)
                break;
            if (LOG) {
                float mx = -INFINITY, sum = 0.0f;
#pragma unroll
                for (int k = 0; k < S; ++k)
                    mx = fmaxf(mx, v[u][k]);
#pragma unroll
                for (int k = 0; k < S; ++k) {
                    v[u][k] = expf(v[u][k] - mx);
                    sum += v[u][k];
                }
#pragma unroll
                for (int k = 0; k < S; ++k)
                    v[u][k] = v[u][k] / sum;
            }
#pragma unroll
            for (int k = 0; k < S; ++k) {
                P[first[u] + k * slice[u]] = v[u][k];
                if (!big)
                    table[at[u] + k * (slice[u] | 1)] = v[u][k];
            }
        }
    }
    if (big)
        return;
    __syncthreads();
    const unsigned pb = def[0].pbegin, n = (def[nd - 1].pend - pb) * SS;
    for (unsigned t = tid; t < n; t += PIECE_THREADS) {
        const unsigned pr = pb + t / SS, kj = t % SS, k = kj / S, j = kj % S;
        const ParentRec rec = parents[pr];
        const DefInfo &di = def[par_def[pr] - c.def0];
        const float *p = table + di.at + k * (di.slice | 1) + j * rec.offset;
        put_table_entry<S>(J, rec, k, j, table_sum<S, S == 2 ? 4 : S == 3 ? 3 : S <= 5 ? 2 : 1>(p, di.slice / S, rec.offset));
    }
    for (unsigned d = tid; d < nd; d += PIECE_THREADS)
        if (def[d].prior != NONE)
#pragma unroll
            for (int k = 0; k < S; ++k)
                st0[(size_t)def[d].prior * SP + k] = table[def[d].at + k];
}

/* The table entries of definitions too large for a piece, from P in memory:
 * the time is that of the longest sum's round trips, so 24 and more loads
 * go out together. */
template <int S>
__global__ void k_big_tables(const unsigned *__restrict__ recs, unsigned nrecs, const DefInfo *__restrict__ defs,
                             const ParentRec *__restrict__ parents, const unsigned *__restrict__ par_def,
                             const float *__restrict__ P, float *__restrict__ J)
{
    constexpr unsigned SS = (unsigned)S * S;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)nrecs * SS)
        return;
    const unsigned pr = recs[t / SS], kj = (unsigned)(t % SS), k = kj / S, j = kj % S;
    const ParentRec rec = parents[pr];
    const DefInfo di = defs[par_def[pr]];
    const float *p = P + di.tb + (size_t)k * di.slice + (size_t)j * rec.offset;
    put_table_entry<S>(J, rec, k, j, table_sum<S, (23 + S) / S>(p, di.slice / S, rec.offset));
}

template <int S, int STEP0, int R>
__global__ __launch_bounds__(BLOCK) void k_adjoint(AdjArgs a)
{
    constexpr int W = WAVE * R;
    __shared__ float lm[WAVES_PER_BLOCK][S * W];
    __shared__ float ldt[WAVES_PER_BLOCK][S * W];
    __shared__ unsigned short lnode[WAVES_PER_BLOCK][W];
    __shared__ unsigned short lq[WAVES_PER_BLOCK][2 * W];
    unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    unsigned Wt = gridDim.x * WAVES_PER_BLOCK;
    unsigned w = xcd_block(blockIdx.x, gridDim.x) * WAVES_PER_BLOCK + wave;
    unsigned c0 = (unsigned)(((unsigned long long)w * a.nchunks) / Wt);
    unsigned c1 = (unsigned)(((unsigned long long)(w + 1) * a.nchunks) / Wt);
    for (unsigned c = c0; c < c1; ++c)
        adjoint_chunk<S, STEP0, R>(a, c, lm[wave], ldt[wave], lnode[wave], lq[wave], lane);
}

/* dL/dst_0 = the step-0 partial + sum of w_0 over the node's out-slots */
template <int S>
__global__ void k_initial_grad(const float *__restrict__ part, const float *__restrict__ w0,
                               const unsigned *__restrict__ out_off, const unsigned *__restrict__ out_slot,
                               float *__restrict__ out, unsigned V)
{
    constexpr int SP = Stride<S>::value;
    unsigned v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V)
        return;
    float acc[S];
    load_rowp<S, SP>(part + (size_t)v * SP, acc);
    sum_out_w<S, SP>(w0, out_slot, out_off[v], out_off[v + 1], acc);
#pragma unroll
    for (int k = 0; k < SP; ++k)
        out[(size_t)v * SP + k] = (k < S) ? acc[k] : 0.0f;
}

/* dL/dparams, or (LOG) dL/dtheta: the transpose of k_set_params.  Parent
 * record pr of a definition gives each entry with its parent in state j and
 * the child in k
 *   G[pr][k][j] = dJ of the forward slot at [j][k] + of the reverse slot at [k][j],
 * formed in LDS first.  An entry's gradient is the sum over the records, in
 * order; they run from the definition's last GIVEN (offset 1) to its first,
 * so j is a base-S digit of the configuration, from the lowest up.  A thread
 * has a row, whose entries share the configuration, and for LOG sends it
 * through the softmax's transpose dtheta = P (.) (dP - <P, dP>).
 *
 * Bound by reading P and writing the gradient once.  (As two launches with G
 * in memory: 21 + 61 us for 21.6M parameters; now 55, 3.5 TB/s.) */
template <int S, bool LOG>
__global__ __launch_bounds__(PIECE_THREADS) void k_param_grad(const float *__restrict__ jbar,
                                                              const Piece *__restrict__ pieces,
                                                              const DefInfo *__restrict__ defs,
                                                              const unsigned short *__restrict__ row_def,
                                                              const ParentRec *__restrict__ parents,
                                                              const float *__restrict__ dst0,
                                                              const float *__restrict__ P, float *__restrict__ out,
                                                              unsigned SP)
{
    constexpr int U = S <= 4 ? 2 : 1;
    constexpr unsigned SS = (unsigned)S * S;
    __shared__ float G[PIECE_FLOATS];
    __shared__ DefInfo def[PIECE_DEFS];
    const Piece c = pieces[blockIdx.x];
    const unsigned nd = c.ndefs & ~BIG, tid = threadIdx.x;
    for (unsigned d = tid; d < nd; d += PIECE_THREADS)
        def[d] = defs[c.def0 + d];
    const unsigned pb = defs[c.def0].pbegin, n = (defs[c.def0 + nd - 1].pend - pb) * SS;
    for (unsigned t = tid; t < n; t += PIECE_THREADS) {
        const unsigned kj = t % SS, k = kj / S, j = kj % S;
        const ParentRec rec = parents[pb + t / SS];
        float g = jbar[(size_t)rec.slot_f * SS + j * S + k];
        if (rec.slot_r != NONE)
            g = g + jbar[(size_t)rec.slot_r * SS + k * S + j];
        G[t] = g;
    }
    __syncthreads();
    for (unsigned r0 = c.row0 + tid; r0 < c.row1; r0 += U * PIECE_THREADS) {
        float pv[U][S], g[U][S];
        unsigned first[U], slice[U];
        const DefInfo *di[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            unsigned r = r0 + u * PIECE_THREADS;
            r = r < c.row1 ? r : r0;
            di[u] = def + row_def[r];
            slice[u] = di[u]->slice;
            first[u] = di[u]->tb + (r - di[u]->rbegin);
            if (LOG)
#pragma unroll
                for (int k = 0; k < S; ++k)
                    pv[u][k] = P[first[u] + k * slice[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            unsigned x = first[u] - di[u]->tb;
            const float *Gd = G + (di[u]->pbegin - pb) * SS;
#pragma unroll
            for (int k = 0; k < S; ++k)
                g[u][k] = 0.0f;
            for (unsigned m = di[u]->pend - di[u]->pbegin; m; --m, Gd += SS) {
                const unsigned q = x / (unsigned)S, j = x - q * (unsigned)S;
                x = q;
#pragma unroll
                for (int k = 0; k < S; ++k)
                    g[u][k] = g[u][k] + Gd[k * S + j];
            }
            if (di[u]->prior != NONE)
#pragma unroll
                for (int k = 0; k < S; ++k)
                    g[u][k] = g[u][k] + dst0[(size_t)di[u]->prior * SP + k];
            if (LOG) {
                float dot = 0.0f;
#pragma unroll
                for (int k = 0; k < S; ++k)
                    dot += pv[u][k] * g[u][k];
#pragma unroll
                for (int k = 0; k < S; ++k)
                    g[u][k] = pv[u][k] * (g[u][k] - dot);
            }
            if (r0 + u * PIECE_THREADS < c.row1)
#pragma unroll
                for (int k = 0; k < S; ++k)
                    out[first[u] + k * slice[u]] = g[u][k];
        }
    }
}

/* dst[i] = src[idx[i]] for rows of SP floats (between the caller's node
 * numbering and the device's) */
__global__ void k_gather_rows(const float *__restrict__ src, const unsigned *__restrict__ idx,
                              float *__restrict__ dst, unsigned V, unsigned SP)
{
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)V * SP)
        return;
    unsigned i = (unsigned)(t / SP), k = (unsigned)(t % SP);
    dst[t] = src[(size_t)idx[i] * SP + k];
}

/* slot order -> reference edge order */
__global__ void k_slot_to_edge(const float *__restrict__ src, const unsigned *__restrict__ slot_edge,
                               float *__restrict__ dst, unsigned E, unsigned width)
{
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)E * width)
        return;
    unsigned s = (unsigned)(t / width), i = (unsigned)(t % width);
    dst[(size_t)slot_edge[s] * width + i] = src[t];
}

/* fn<states>(...) */
#define FOR_STATES(states, fn, ...)                                                                              \
    switch (states) {                                                                                            \
    case 1: fn<1>(__VA_ARGS__); break;                                                                           \
    case 2: fn<2>(__VA_ARGS__); break;                                                                           \
    case 3: fn<3>(__VA_ARGS__); break;                                                                           \
    case 4: fn<4>(__VA_ARGS__); break;                                                                           \
    case 5: fn<5>(__VA_ARGS__); break;                                                                           \
    case 6: fn<6>(__VA_ARGS__); break;                                                                           \
    case 7: fn<7>(__VA_ARGS__); break;                                                                           \
    case 8: fn<8>(__VA_ARGS__); break;                                                                           \
    case 9: fn<9>(__VA_ARGS__); break;                                                                           \
    case 10: fn<10>(__VA_ARGS__); break;                                                                         \
    }

inline unsigned blocks_for(size_t n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }

} // namespace

struct bp_diff {
    bp_dev *d = nullptr;
    unsigned V = 0, E = 0, S = 0, SP = 0;
    unsigned num_params = 0, num_rows = 0;
    std::vector<uint64_t> row_first;
    std::vector<uint32_t> row_stride, row_len;

    unsigned *par_def = nullptr; /* definition of each parent record */
    unsigned *out_off = nullptr, *out_slot = nullptr, *slot_pos = nullptr, *slot_edge = nullptr;
    DefInfo *defs = nullptr;
    ParentRec *parents = nullptr;
    Piece *pieces = nullptr;
    unsigned npieces = 0;
    unsigned short *row_def = nullptr; /* each softmax row's definition, from its piece's first */
    unsigned *big_recs = nullptr;      /* records of definitions larger than a piece */
    unsigned nbig = 0;

    float *P = nullptr;     /* parameters */
    unsigned *perm_d = nullptr, *inv_d = nullptr; /* node -> device node, device node -> node */
    float *st0 = nullptr;   /* initial beliefs */
    float *gin = nullptr;   /* dL/dbeliefs (copy) */
    float *gst[2] = {nullptr, nullptr};
    float *w[2] = {nullptr, nullptr};
    float *jbar = nullptr;
    float *dst0p = nullptr, *dst0 = nullptr;
    /* the adjoint's chunks: at most 64 x adj_R slots and nodes each */
    uint2 *adj_chunk = nullptr;
    unsigned adj_R = 1, adj_nchunks = 0, adj_G = 8;

    /* iterates: checkpoints t = 0, c, 2c, ...; a segment's recomputed ones;
     * the forward's scratch; the last beliefs */
    unsigned K = 0, c = 0, nck = 0;
    /* Iterates (beliefs and combine buffers) up to this many bytes are all
     * kept: recomputing the ones between checkpoints of every fifth took 24
     * launches of a 30-iteration backward, 290 of its 1460 us on 200k nodes,
     * to save 150 of the card's 288,000 MB. */
    size_t keep_bytes = 512u << 20;
    size_t stride = 0;          /* floats between two iterates: whole 128-byte lines */
    unsigned max_in = 0;        /* largest in-degree */
    bool have_forward = false, have_params = false;
    bool kept = false;          /* the last forward's iterates are all in ck_st, ck_buf */
    float *ck_st = nullptr, *ck_buf = nullptr;
    float *seg_st = nullptr, *seg_buf = nullptr;
    float *fw_st[2] = {nullptr, nullptr}, *fw_buf[2] = {nullptr, nullptr};
    float *final_st = nullptr;
    /* resident backward: the rows of w of every step, and where each is */
    float *rows = nullptr;
    unsigned *out_at = nullptr;
    std::map<std::pair<unsigned, unsigned>, hipGraphExec_t> fwd_graphs, bwd_graphs;
};

static void diff_release_storage(bp_diff *x)
{
    float *ps[] = {x->ck_st, x->ck_buf, x->seg_st, x->seg_buf, x->fw_st[0], x->fw_st[1], x->fw_buf[0], x->fw_buf[1],
                   x->final_st, x->rows};
    for (float *p : ps)
        if (p)
            (void)hipFree(p);
    x->ck_st = x->ck_buf = x->seg_st = x->seg_buf = x->final_st = x->rows = nullptr;
    x->fw_st[0] = x->fw_st[1] = x->fw_buf[0] = x->fw_buf[1] = nullptr;
    for (auto &kv : x->fwd_graphs)
        (void)hipGraphExecDestroy(kv.second);
    for (auto &kv : x->bwd_graphs)
        (void)hipGraphExecDestroy(kv.second);
    x->fwd_graphs.clear();
    x->bwd_graphs.clear();
    x->K = x->c = x->nck = 0;
}

extern "C" void bp_diff_free(bp_diff *x)
{
    if (!x)
        return;
    if (x->d)
        (void)hipSetDevice(x->d->device);
    diff_release_storage(x); /* hipFree waits for the device, callers' streams included */
    void *ps[] = {x->out_at, x->adj_chunk, x->defs, x->perm_d, x->inv_d, x->row_def, x->par_def, x->pieces, x->big_recs, x->out_off,
                  x->out_slot, x->slot_pos, x->slot_edge, x->parents, x->P, x->st0, x->gin, x->gst[0], x->gst[1],
                  x->w[0], x->w[1], x->jbar, x->dst0p, x->dst0};
    for (void *p : ps)
        if (p)
            (void)hipFree(p);
    bp_free(x->d);
    delete x;
}

template <typename T> static int upload_vec(bp_diff *x, T **dst, const std::vector<T> &v)
{
    return dmalloc(dst, v.size()) ||
           copy_on(x->d->stream, *dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) ? -1 : 0;
}

/* checks that need no device: one state count, in-degrees within a wave's
 * chunk, observations after the parameters, complete tables */
static int diff_validate(const bp_bn *bn, unsigned npd, Graph_t g)
{
    unsigned V = g->current_num_vertices;
    unsigned S = V ? g->node_num_vars[0] : 1;
    const unsigned R = S <= 4 ? (unsigned)BP_ADJ_SLOTS_SMALL : 1u;
    for (unsigned v = 0; v < V; ++v)
        if (g->node_num_vars[v] != S) {
            bp_set_error("bp_diff_create: node %u has %u states, node 0 has %u; the adjoint needs one state count", v,
                         g->node_num_vars[v], S);
            return -1;
        }
    for (unsigned v = 0; v < V; ++v) {
        unsigned deg = bp_csr_end(g, g->dest_nodes_to_edges_node_list, v) - g->dest_nodes_to_edges_node_list[v];
        if (deg > WAVE * R) {
            bp_set_error("bp_diff_create: node %u has %u in-edges (the adjoint handles up to %u)", v, deg, WAVE * R);
            return -1;
        }
    }
    if (bn->def_table_begin[npd] > 0xfffffff0ull) {
        bp_set_error("bp_diff_create: too many parameters");
        return -1;
    }
    for (unsigned dd = 0; dd < bn->num_defs; ++dd) {
        uint64_t g0 = bn->def_given_begin[dd], g1 = bn->def_given_begin[dd + 1];
        uint64_t t0 = bn->def_table_begin[dd], t1 = bn->def_table_begin[dd + 1];
        if (dd >= npd) {
            if (g1 != g0) {
                bp_set_error("bp_diff_create: definition %u after the parameters has GIVENs", dd);
                return -1;
            }
            continue;
        }
        uint64_t expect = bn->num_states[bn->def_for[dd]];
        for (uint64_t i = g0; i < g1; ++i)
            expect *= bn->num_states[bn->def_given[i]];
        if (t1 - t0 != expect) {
            bp_set_error("bp_diff_create: definition %u has %llu TABLE entries, %llu expected", dd,
                         (unsigned long long)(t1 - t0), (unsigned long long)expect);
            return -1;
        }
    }
    return 0;
}

/* cut the definitions into pieces; sets their places in LDS.  Pieces are
 * four times smaller where that gives the card twice as many as it has
 * CUs. */
static int build_pieces(bp_diff *x, std::vector<DefInfo> &defs)
{
    const unsigned S = x->S, SS = S * S, npd = (unsigned)defs.size();
    const unsigned limit = x->num_params < 512 * PIECE_FLOATS ? PIECE_FLOATS / 4 : PIECE_FLOATS;
    const unsigned big_rows = std::max(1u, limit / S);
    std::vector<Piece> pieces;
    std::vector<unsigned short> row_def(x->num_rows);
    std::vector<unsigned> big_recs;
    for (unsigned d = 0; d < npd;) {
        unsigned floats = 0, recs = 0, e = d;
        while (e < npd && e - d < PIECE_DEFS) {
            const DefInfo &di = defs[e];
            const size_t f = (size_t)S * (di.slice | 1), r = (size_t)(di.pend - di.pbegin) * SS;
            if (f > PIECE_FLOATS || (e > d && (floats + f > limit || recs + r > PIECE_FLOATS)))
                break;
            defs[e].at = floats;
            std::fill_n(row_def.begin() + di.rbegin, di.slice, (unsigned short)(e - d));
            floats += (unsigned)f;
            recs += (unsigned)r;
            ++e;
        }
        if (e > d) {
            pieces.push_back({d, e - d, defs[d].rbegin, defs[e - 1].rbegin + defs[e - 1].slice});
            d = e;
            continue;
        }
        const DefInfo &di = defs[d];
        for (unsigned r = 0; r < di.slice; r += big_rows)
            pieces.push_back({d, 1 | BIG, di.rbegin + r, di.rbegin + std::min(r + big_rows, di.slice)});
        for (unsigned q = di.pbegin; q < di.pend; ++q)
            big_recs.push_back(q);
        ++d;
    }
    x->npieces = (unsigned)pieces.size();
    x->nbig = (unsigned)big_recs.size();
    return upload_vec(x, &x->pieces, pieces) || upload_vec(x, &x->row_def, row_def) ||
                   upload_vec(x, &x->big_recs, big_recs)
               ? -1
               : 0;
}

static int diff_build(bp_diff *x, const bp_bn *bn, unsigned npd, Graph_t g)
{
    bp_dev *d = x->d;
    unsigned V = d->V, E = d->E, S = d->S;
    x->num_params = (unsigned)bn->def_table_begin[npd];

    /* replay the reader's edge emission: definitions in order, parents last
     * GIVEN first, forward edge then reverse edge unless the parent is
     * observed (bp_graph_add_cpt_edges) */
    std::vector<unsigned> def_tb(npd), def_slice(npd), def_pbegin(npd + 1, 0), def_prior(npd, NONE);
    std::vector<ParentRec> prs;
    std::vector<unsigned> par_def;
    unsigned e = 0;
    for (unsigned dd = 0; dd < bn->num_defs; ++dd) {
        uint64_t g0 = bn->def_given_begin[dd], g1 = bn->def_given_begin[dd + 1];
        uint64_t t0 = bn->def_table_begin[dd], t1 = bn->def_table_begin[dd + 1];
        unsigned child = bn->def_for[dd];
        unsigned nch = bn->num_states[child];
        if (dd >= npd)
            continue;
        def_tb[dd] = (unsigned)t0;
        unsigned slice = (unsigned)((t1 - t0) / nch);
        def_slice[dd] = slice;
        unsigned offset = 1;
        for (uint64_t pi = g1; pi-- > g0;) {
            unsigned parent = bn->def_given[pi];
            unsigned npar = bn->num_states[parent];
            ParentRec pr{offset, npar, NONE, NONE};
            if (e >= E || g->edges_src_index[e] != parent || g->edges_dest_index[e] != child) {
                bp_set_error("bp_diff_create: edge %u does not follow the reader's order", e);
                return -1;
            }
            pr.slot_f = d->edge_slot[e];
            ++e;
            if (g->observed_nodes[parent] != 1) {
                if (e >= E || g->edges_src_index[e] != child || g->edges_dest_index[e] != parent) {
                    bp_set_error("bp_diff_create: edge %u does not follow the reader's order", e);
                    return -1;
                }
                pr.slot_r = d->edge_slot[e];
                ++e;
            }
            prs.push_back(pr);
            par_def.push_back(dd);
            offset *= npar;
        }
        def_pbegin[dd + 1] = (unsigned)prs.size();
    }
    if (e != E) {
        bp_set_error("bp_diff_create: %u of %u edges come from the definitions", e, E);
        return -1;
    }
    /* initial beliefs: the last GIVEN-less definition of a node sets them */
    std::vector<unsigned> state_def(V, NONE);
    for (unsigned dd = 0; dd < bn->num_defs; ++dd)
        if (bn->def_given_begin[dd + 1] == bn->def_given_begin[dd])
            state_def[bn->def_for[dd]] = dd;
    /* per device node (the handle numbers nodes in its own order) */
    for (unsigned v = 0; v < V; ++v)
        if (state_def[v] != NONE && state_def[v] < npd)
            def_prior[state_def[v]] = d->perm[v];
    std::vector<DefInfo> definfo(npd);
    for (unsigned dd = 0; dd < npd; ++dd)
        definfo[dd] = DefInfo{def_tb[dd], def_slice[dd], def_pbegin[dd], def_pbegin[dd + 1], def_prior[dd], 0, 0, 0};
    for (unsigned dd = 0, rows = 0; dd < npd; ++dd) {
        definfo[dd].rbegin = rows;
        rows += def_slice[dd];
    }
    /* softmax rows */
    x->row_first.clear();
    x->row_stride.clear();
    x->row_len.clear();
    for (unsigned dd = 0; dd < npd; ++dd) {
        unsigned nch = bn->num_states[bn->def_for[dd]];
        for (unsigned cc = 0; cc < def_slice[dd]; ++cc) {
            x->row_first.push_back((uint64_t)def_tb[dd] + cc);
            x->row_stride.push_back(def_slice[dd]);
            x->row_len.push_back(nch);
        }
    }
    x->num_rows = (unsigned)x->row_first.size();
    if (build_pieces(x, definfo))
        return -1;
    /* source-grouped slots */
    std::vector<unsigned> out_off(V + 1, 0), out_slot(E), slot_src(E);
    for (unsigned s = 0; s < E; ++s) {
        slot_src[s] = d->perm[g->edges_src_index[d->slot_edge[s]]];
        out_off[slot_src[s] + 1]++;
    }
    for (unsigned v = 0; v < V; ++v)
        out_off[v + 1] += out_off[v];
    {
        std::vector<unsigned> fill(out_off.begin(), out_off.end() - 1);
        for (unsigned s = 0; s < E; ++s)
            out_slot[fill[slot_src[s]]++] = s;
    }
    std::vector<unsigned> slot_pos(E);
    for (unsigned o = 0; o < E; ++o)
        slot_pos[out_slot[o]] = o;
    {
        std::vector<unsigned> in_off(V + 1, 0);
        for (unsigned s = 0; s < E; ++s)
            in_off[d->perm[g->edges_dest_index[d->slot_edge[s]]] + 1]++;
        for (unsigned v = 0; v < V; ++v)
            in_off[v + 1] += in_off[v];
        x->adj_R = (S <= 4) ? (unsigned)BP_ADJ_SLOTS_SMALL : 1u;
        std::vector<uint2> ch;
        bp_build_chunks(in_off, V, WAVE * x->adj_R, ch);
        x->adj_nchunks = (unsigned)ch.size() - 1;
        unsigned want = (x->adj_nchunks + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
        x->adj_G = std::max(8u, (want + 7u) & ~7u);
        if (upload_vec(x, &x->adj_chunk, ch))
            return -1;
    }
    size_t VS = (size_t)V * d->SP, ES = (size_t)E * d->SP;
    if (upload_vec(x, &x->perm_d, d->perm) || upload_vec(x, &x->inv_d, d->inv) || upload_vec(x, &x->out_off, out_off) ||
        upload_vec(x, &x->out_slot, out_slot) || upload_vec(x, &x->slot_pos, slot_pos) ||
        upload_vec(x, &x->slot_edge, d->slot_edge) || upload_vec(x, &x->defs, definfo) ||
        upload_vec(x, &x->parents, prs) || upload_vec(x, &x->par_def, par_def) || dmalloc(&x->P, x->num_params) ||
        dmalloc(&x->st0, VS) || dmalloc(&x->gin, VS) || dmalloc(&x->gst[0], VS) || dmalloc(&x->gst[1], VS) ||
        dmalloc(&x->w[0], ES) || dmalloc(&x->w[1], ES) || dmalloc(&x->jbar, (size_t)E * S * S) ||
        dmalloc(&x->dst0p, VS) || dmalloc(&x->dst0, VS))
        return -1;
    return 0;
}

extern "C" int bp_diff_create(const bp_bn *bn, unsigned int num_param_defs, int device, bp_diff **out)
{
    bp_clear_error();
    if (!bn || !out) {
        bp_set_error("bp_diff_create: NULL argument");
        return -1;
    }
    *out = nullptr;
    if (num_param_defs > bn->num_defs) {
        bp_set_error("bp_diff_create: %u parameter definitions of %u", num_param_defs, bn->num_defs);
        return -1;
    }
    int abort_prev = bp_set_abort_on_error(0);
    Graph_t g = bp_bn_to_graph(bn);
    if (g) {
        set_up_src_nodes_to_edges(g);
        set_up_dest_nodes_to_edges(g);
    }
    bp_set_abort_on_error(abort_prev);
    if (!g || bp_has_error()) {
        if (g)
            graph_destroy(g);
        return -1;
    }
    if (diff_validate(bn, num_param_defs, g)) {
        graph_destroy(g);
        return -1;
    }
    bp_diff *x = new bp_diff();
    int rc = bp_upload_graph(g, device, &x->d);
    if (rc == 0) {
        x->V = x->d->V;
        x->E = x->d->E;
        x->S = x->d->S;
        x->SP = x->d->SP;
        x->stride = ((size_t)x->V * x->SP + 31) / 32 * 32;
        for (unsigned v = 0; v < x->V; ++v)
            x->max_in = std::max(x->max_in, x->d->in_off_h[v + 1] - x->d->in_off_h[v]);
        rc = diff_build(x, bn, num_param_defs, g);
        /* nodes without a parameter prior keep their initial beliefs */
        if (rc == 0 && x->V &&
            taken(hipMemcpyAsync(x->st0, x->d->states0, (size_t)x->V * x->SP * sizeof(float), hipMemcpyDeviceToDevice,
                                 x->d->stream)) != hipSuccess) {
            bp_set_error("bp_diff_create: copying the initial beliefs failed");
            rc = -1;
        }
        if (rc == 0 && taken(hipStreamSynchronize(x->d->stream)) != hipSuccess)
            rc = -1;
        if (rc == 0 && bp_resident_diff_fits(x->d, x->max_in) &&
            (dmalloc(&x->out_at, x->E) || bp_resident_diff_places(x->d, x->slot_pos, x->out_at)))
            rc = -1;
    }
    graph_destroy(g);
    if (rc) {
        bp_diff_free(x);
        return -1;
    }
    *out = x;
    return 0;
}

extern "C" int bp_diff_info(const bp_diff *x, uint64_t *info)
{
    if (!x || !info) {
        bp_set_error("bp_diff_info: NULL argument");
        return -1;
    }
    info[0] = x->V;
    info[1] = x->E;
    info[2] = x->S;
    info[3] = x->SP;
    info[4] = x->num_params;
    info[5] = x->num_rows;
    return 0;
}

extern "C" int bp_diff_rows(const bp_diff *x, uint64_t *row_first, uint32_t *row_stride, uint32_t *row_len)
{
    if (!x || !row_first || !row_stride || !row_len) {
        bp_set_error("bp_diff_rows: NULL argument");
        return -1;
    }
    std::copy(x->row_first.begin(), x->row_first.end(), row_first);
    std::copy(x->row_stride.begin(), x->row_stride.end(), row_stride);
    std::copy(x->row_len.begin(), x->row_len.end(), row_len);
    return 0;
}

template <int S> static void launch_set_params(bp_diff *x, bool log, const float *theta, hipStream_t st)
{
    if (x->npieces)
        hipLaunchKernelGGL((log ? k_set_params<S, true> : k_set_params<S, false>), dim3(x->npieces),
                           dim3(PIECE_THREADS), 0, st, theta, x->pieces, x->defs, x->row_def, x->parents, x->par_def,
                           x->P, x->d->J, x->st0, x->SP);
    if (x->nbig)
        hipLaunchKernelGGL(k_big_tables<S>, dim3(blocks_for((size_t)x->nbig * S * S, 64)), dim3(64), 0, st,
                           x->big_recs, x->nbig, x->defs, x->parents, x->par_def, x->P, x->d->J);
}

static int set_params(bp_diff *x, bool log, const float *theta, const char *who, void *stream)
{
    bp_clear_error();
    if (!x || !theta) {
        bp_set_error("%s: NULL argument", who);
        return -1;
    }
    HIP_TRY(hipSetDevice(x->d->device));
    FOR_STATES(x->S, launch_set_params, x, log, theta, (hipStream_t)stream);
    HIP_TRY(hipGetLastError());
    x->have_params = true;
    x->have_forward = false;
    return 0;
}

extern "C" int bp_diff_set_params(bp_diff *x, const float *params, void *stream)
{
    return set_params(x, false, params, "bp_diff_set_params", stream);
}

extern "C" int bp_diff_set_log_params(bp_diff *x, const float *theta, void *stream)
{
    return set_params(x, true, theta, "bp_diff_set_log_params", stream);
}

static int diff_storage(bp_diff *x, unsigned K, unsigned c)
{
    diff_release_storage(x);
    size_t VS = x->stride;
    unsigned nck = K / c + 1;
    if (dmalloc(&x->ck_st, nck * VS) || dmalloc(&x->ck_buf, nck * VS) || dmalloc(&x->seg_st, (size_t)c * VS) ||
        dmalloc(&x->seg_buf, (size_t)c * VS) || dmalloc(&x->fw_st[0], VS) || dmalloc(&x->fw_st[1], VS) ||
        dmalloc(&x->fw_buf[0], VS) || dmalloc(&x->fw_buf[1], VS) || dmalloc(&x->final_st, VS)) {
        diff_release_storage(x);
        return -1;
    }
    /* (without the memory for it the backward runs its launches) */
    if (c == 1 && x->out_at) {
        const size_t rows = ((size_t)K + 1) * bp_resident_diff_rows(x->d);
        if (rows * sizeof(float) <= x->keep_bytes &&
            taken(hipMalloc((void **)&x->rows, rows * sizeof(float))) != hipSuccess)
            x->rows = nullptr;
    }
    x->K = K;
    x->c = c;
    x->nck = nck;
    return 0;
}

/* one FWD (or FINIT) launch: (st_in, buf_in) -> (st_out, buf_out) */
static void fwd_step(bp_diff *x, int mode, const float *st_in, const float *buf_in, float *st_out, float *buf_out,
                     hipStream_t st)
{
    LoopyArgs a = bp_make_args(x->d);
    a.states = const_cast<float *>(st_in);
    a.states_out = st_out;
    a.buf_in = buf_in;
    a.buf_out = buf_out;
    a.msg_in = nullptr;
    a.msg_out = nullptr;
    a.partials = nullptr;
    a.stop = nullptr;
    bp_launch_loopy(x->d, mode, a, st);
}

static int capture_begin(bp_diff *x)
{
    HIP_TRY(hipStreamBeginCapture(x->d->stream, hipStreamCaptureModeThreadLocal));
    return 0;
}

static int capture_end(bp_diff *x, hipGraphExec_t *exec)
{
    hipGraph_t graph = nullptr;
    HIP_TRY(hipStreamEndCapture(x->d->stream, &graph));
    hipError_t err = taken(hipGraphInstantiate(exec, graph, nullptr, nullptr, 0));
    (void)hipGraphDestroy(graph);
    if (err != hipSuccess) {
        bp_set_error("hipGraphInstantiate failed: %s", hipGetErrorString(err));
        return -1;
    }
    return 0;
}

static void enqueue_forward(bp_diff *x, hipStream_t st)
{
    const size_t VS = x->stride;
    unsigned K = x->K, c = x->c;
    fwd_step(x, FINIT, x->st0, nullptr, nullptr, x->ck_buf, st);
    const float *sp = x->st0, *bp = x->ck_buf;
    for (unsigned t = 1; t <= K; ++t) {
        float *so, *bo;
        if (t % c == 0) {
            so = x->ck_st + (size_t)(t / c) * VS;
            bo = x->ck_buf + (size_t)(t / c) * VS;
        } else {
            so = x->fw_st[t & 1];
            bo = x->fw_buf[t & 1];
        }
        fwd_step(x, FWD, sp, bp, so, bo, st);
        sp = so;
        bp = bo;
    }
    const size_t n = (size_t)x->V * x->SP;
    hipLaunchKernelGGL(k_copy, dim3(blocks_for(n)), dim3(256), 0, st, sp, x->final_st, n);
}

static bool is_capturing(hipStream_t st)
{
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (st)
        (void)taken(hipStreamIsCapturing(st, &capturing));
    return capturing != hipStreamCaptureStatusNone;
}

/* Whether the iterates, all kept, are run resident (not into a graph that is
 * being captured: a run counts its barriers once). */
static bool use_resident(bp_diff *x, hipStream_t st)
{
    return x->c == 1 && !is_capturing(st) && bp_resident_diff_fits(x->d, x->max_in);
}

/* enqueue's launches on the caller's stream, by way of a graph that is kept
 * for this K and c; one by one into a graph of the caller's, which a graph
 * launched here would not become part of. */
static int run_launches(bp_diff *x, std::map<std::pair<unsigned, unsigned>, hipGraphExec_t> &graphs,
                        void (*enqueue)(bp_diff *, hipStream_t), hipStream_t st)
{
    if (is_capturing(st)) {
        enqueue(x, st);
        return 0;
    }
    const auto key = std::make_pair(x->K, x->c);
    auto it = graphs.find(key);
    if (it == graphs.end()) {
        hipGraphExec_t exec = nullptr;
        {
            std::lock_guard<std::mutex> lock(bp_resident_mutex());
            if (capture_begin(x))
                return -1;
            enqueue(x, x->d->stream);
            if (capture_end(x, &exec))
                return -1;
        }
        it = graphs.emplace(key, exec).first;
    }
    HIP_TRY(hipGraphLaunch(it->second, st));
    return 0;
}

extern "C" int bp_diff_forward(bp_diff *x, unsigned int K, unsigned int c, float *beliefs, void *stream)
{
    bp_clear_error();
    if (!x || !beliefs || c == 0) {
        bp_set_error("bp_diff_forward: NULL argument or zero checkpoint interval");
        return -1;
    }
    if (!x->have_params) {
        bp_set_error("bp_diff_forward: bp_diff_set_params has not been called");
        return -1;
    }
    HIP_TRY(hipSetDevice(x->d->device));
    size_t VS = (size_t)x->V * x->SP;
    const unsigned every = 2 * ((size_t)K + 1) * x->stride * sizeof(float) <= x->keep_bytes ? 1 : c;
    hipStream_t st = (hipStream_t)stream;
    /* (where the memory for all of them is not to be had, the storage for the
     * interval stays: trying again each time freed and allocated everything) */
    const bool stored = x->final_st && x->K == K && (x->c == every || x->c == c);
    if (!stored && is_capturing(st)) {
        bp_set_error("bp_diff_forward: the first call with %u iterations and interval %u allocates and cannot be captured",
                     K, c);
        return -1;
    }
    if (!stored && diff_storage(x, K, every)) {
        if (every == c)
            return -1;
        bp_clear_error(); /* not the memory for all of them */
        if (diff_storage(x, K, c))
            return -1;
    }
    c = x->c;
    /* the ck_st[0] slot is the initial beliefs themselves */
    hipLaunchKernelGGL(k_copy, dim3(blocks_for(VS)), dim3(256), 0, st, x->st0, x->ck_st, VS);
    if (K && use_resident(x, st)) {
        fwd_step(x, FINIT, x->st0, nullptr, nullptr, x->ck_buf, st);
        if (bp_resident_diff_forward(x->d, K, x->ck_st, x->ck_buf, x->stride, st))
            return -1;
        hipLaunchKernelGGL(k_gather_rows, dim3(blocks_for(VS)), dim3(256), 0, st, x->ck_st + K * x->stride, x->perm_d,
                           beliefs, x->V, x->SP);
        HIP_TRY(hipGetLastError());
        x->have_forward = x->kept = true;
        return 0;
    }
    if (run_launches(x, x->fwd_graphs, enqueue_forward, st))
        return -1;
    hipLaunchKernelGGL(k_gather_rows, dim3(blocks_for(VS)), dim3(256), 0, st, x->final_st, x->perm_d, beliefs, x->V,
                       x->SP);
    HIP_TRY(hipGetLastError());
    x->have_forward = true;
    x->kept = false;
    return 0;
}

static void adj_step(bp_diff *x, int step0, const float *st_prev, const float *st_cur, const float *bsrc,
                     const float *gst_in, float *gst_out, const float *w_in, float *w_out, int first, hipStream_t st)
{
    bp_dev *d = x->d;
    AdjArgs a;
    a.in_off = d->in_off;
    a.slot_src = d->slot_src;
    a.out_off = x->out_off;
    a.out_slot = x->out_slot;
    a.slot_pos = x->slot_pos;
    a.J = d->J;
    a.chunk = x->adj_chunk;
    a.nchunks = x->adj_nchunks;
    a.st_prev = st_prev;
    a.st_cur = st_cur;
    a.bsrc = bsrc;
    a.gst_in = gst_in;
    a.gst_out = gst_out;
    a.w_in = w_in;
    a.w_out = w_out;
    a.jbar = x->jbar;
    a.jbar_first = first;
    dim3 grid(x->adj_G), block(BLOCK);
    constexpr int RS = BP_ADJ_SLOTS_SMALL;
#define BP_ADJ_CASE(SS)                                                                   \
    case SS:                                                                              \
        if (step0)                                                                        \
            hipLaunchKernelGGL((k_adjoint<SS, 1, (SS <= 4 ? RS : 1)>), grid, block, 0, st, a); \
        else                                                                              \
            hipLaunchKernelGGL((k_adjoint<SS, 0, (SS <= 4 ? RS : 1)>), grid, block, 0, st, a); \
        break;
    switch (d->S) {
        BP_ADJ_CASE(1)
        BP_ADJ_CASE(2)
        BP_ADJ_CASE(3)
        BP_ADJ_CASE(4)
        BP_ADJ_CASE(5)
        BP_ADJ_CASE(6)
        BP_ADJ_CASE(7)
        BP_ADJ_CASE(8)
        BP_ADJ_CASE(9)
        BP_ADJ_CASE(10)
    }
#undef BP_ADJ_CASE
}

static void enqueue_backward_tail(bp_diff *x, const float *w0, hipStream_t st);

static void enqueue_backward(bp_diff *x, hipStream_t st)
{
    const size_t VS = x->stride;
    unsigned K = x->K, c = x->c;
    unsigned nseg = (K + c - 1) / c;
    const float *gin = x->gin; /* dL/dst_K */
    const float *w_in = nullptr;
    int first = 1;
    std::vector<const float *> stp(c + 1), bufp(c + 1);
    for (unsigned k = nseg; k-- > 0;) {
        unsigned t0 = k * c, t1 = std::min(t0 + c, K);
        stp[0] = x->ck_st + (size_t)k * VS;
        bufp[0] = x->ck_buf + (size_t)k * VS;
        for (unsigned t = t0 + 1; t < t1; ++t) {
            float *so = x->seg_st + (size_t)(t - t0) * VS, *bo = x->seg_buf + (size_t)(t - t0) * VS;
            fwd_step(x, FWD, stp[t - 1 - t0], bufp[t - 1 - t0], so, bo, st);
            stp[t - t0] = so;
            bufp[t - t0] = bo;
        }
        stp[t1 - t0] = (t1 == K) ? x->final_st : x->ck_st + (size_t)(k + 1) * VS;
        for (unsigned t = t1; t > t0; --t) {
            float *gout = x->gst[(t - 1) & 1];
            float *wout = x->w[t & 1];
            adj_step(x, 0, stp[t - 1 - t0], stp[t - t0], bufp[t - 1 - t0], gin, gout, w_in, wout, first, st);
            gin = gout;
            w_in = wout;
            first = 0;
        }
    }
    /* step 0: init */
    adj_step(x, 1, nullptr, x->st0, x->st0, gin, x->dst0p, w_in, x->w[0] == w_in ? x->w[1] : x->w[0], first, st);
    enqueue_backward_tail(x, (x->w[0] == w_in) ? x->w[1] : x->w[0], st);
}

/* dL/d(initial beliefs) and the per-parent sums */
template <int S> static void launch_initial_grad(bp_diff *x, const float *w0, hipStream_t st)
{
    hipLaunchKernelGGL(k_initial_grad<S>, dim3(blocks_for(x->V)), dim3(256), 0, st, x->dst0p, w0, x->out_off,
                       x->out_slot, x->dst0, x->V);
}

static void enqueue_backward_tail(bp_diff *x, const float *w0, hipStream_t st)
{
    FOR_STATES(x->S, launch_initial_grad, x, w0, st);
}

/* The gradient of the parameters or (log) of the log-parameters from the
 * tables' and initial beliefs' of the last backward. */
template <int S> static void launch_param_grad(bp_diff *x, bool log, float *out, hipStream_t st)
{
    if (x->npieces)
        hipLaunchKernelGGL((log ? k_param_grad<S, true> : k_param_grad<S, false>), dim3(x->npieces),
                           dim3(PIECE_THREADS), 0, st, x->jbar, x->pieces, x->defs, x->row_def, x->parents, x->dst0,
                           x->P, out, x->SP);
}

extern "C" int bp_diff_backward_ex(bp_diff *x, const float *grad_beliefs, float *grad_params, float *grad_tables,
                                   float *grad_initial, void *stream)
{
    bp_clear_error();
    if (!x || !grad_beliefs) {
        bp_set_error("bp_diff_backward: NULL argument");
        return -1;
    }
    if (!x->have_forward) {
        bp_set_error("bp_diff_backward: no forward since the parameters were set");
        return -1;
    }
    HIP_TRY(hipSetDevice(x->d->device));
    hipStream_t st = (hipStream_t)stream;
    size_t VS = (size_t)x->V * x->SP;
    hipLaunchKernelGGL(k_gather_rows, dim3(blocks_for(VS)), dim3(256), 0, st, grad_beliefs, x->inv_d, x->gin, x->V,
                       x->SP);
    if (x->kept && x->rows && use_resident(x, st)) {
        bp_adjoint_arrays arrays = {x->out_off, x->out_slot, x->slot_pos, x->adj_chunk, x->adj_nchunks, x->st0, x->gin,
                                    {x->gst[0], x->gst[1]}, {x->w[0], x->w[1]}, x->jbar, x->dst0p, x->dst0,
                                    x->out_at, x->rows};
        if (bp_resident_diff_backward(x->d, x->K, x->ck_st, x->ck_buf, x->stride, arrays, st))
            return -1;
    } else {
        if (x->kept) /* the launches look for the last beliefs here */
            hipLaunchKernelGGL(k_copy, dim3(blocks_for(VS)), dim3(256), 0, st, x->ck_st + x->K * x->stride,
                               x->final_st, VS);
        if (run_launches(x, x->bwd_graphs, enqueue_backward, st))
            return -1;
    }
    if (grad_params)
        FOR_STATES(x->S, launch_param_grad, x, false, grad_params, st);
    size_t SS = (size_t)x->S * x->S;
    if (grad_tables && x->E)
        hipLaunchKernelGGL(k_slot_to_edge, dim3(blocks_for((size_t)x->E * SS)), dim3(256), 0, st, x->jbar,
                           x->slot_edge, grad_tables, x->E, (unsigned)SS);
    if (grad_initial)
        hipLaunchKernelGGL(k_gather_rows, dim3(blocks_for(VS)), dim3(256), 0, st, x->dst0, x->perm_d, grad_initial,
                           x->V, x->SP);
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int bp_diff_backward(bp_diff *x, const float *grad_beliefs, float *grad_params, void *stream)
{
    return bp_diff_backward_ex(x, grad_beliefs, grad_params, nullptr, nullptr, stream);
}

extern "C" int bp_diff_backward_log(bp_diff *x, const float *grad_beliefs, float *grad_theta, void *stream)
{
    if (!grad_theta) {
        bp_set_error("bp_diff_backward_log: NULL argument");
        return -1;
    }
    if (bp_diff_backward_ex(x, grad_beliefs, nullptr, nullptr, nullptr, stream))
        return -1;
    FOR_STATES(x->S, launch_param_grad, x, true, grad_theta, (hipStream_t)stream);
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int bp_diff_tables(bp_diff *x, float *out)
{
    bp_clear_error();
    if (!x || !out) {
        bp_set_error("bp_diff_tables: NULL argument");
        return -1;
    }
    HIP_TRY(hipSetDevice(x->d->device));
    HIP_TRY(hipDeviceSynchronize());
    size_t SS = (size_t)x->S * x->S;
    std::vector<float> tmp((size_t)x->E * SS);
    if (!tmp.empty())
        HIP_TRY(hipMemcpy(tmp.data(), x->d->J, tmp.size() * sizeof(float), hipMemcpyDeviceToHost));
    for (unsigned s = 0; s < x->E; ++s)
        std::memcpy(out + (size_t)x->d->slot_edge[s] * SS, tmp.data() + (size_t)s * SS, SS * sizeof(float));
    return 0;
}

/* For checks: the handle a network's runs use, whether a run of it was given
 * up (ask after the stream has been waited for), and the bytes of iterates
 * that are kept whatever the checkpoint interval. */
extern "C" bp_dev *bp_diff_device(bp_diff *x) { return x->d; }
extern "C" unsigned bp_diff_gave_up(const bp_diff *x) { return x->d->status()->gave_up; }
extern "C" void bp_diff_set_keep(bp_diff *x, unsigned long long bytes) { x->keep_bytes = bytes; }
