/*
 * bp_adjoint.h -- one iteration of the adjoint over one chunk (bp_diff.hip's
 * launches, and the single workgroup that makes up for a resident run that
 * was given up, bp_resident_diff.hip).
 */
#pragma once

#include "bp_dev.h"

/* Slots per lane of the adjoint for four or fewer states (one above). */
#ifndef BP_ADJ_SLOTS_SMALL
#define BP_ADJ_SLOTS_SMALL 2
#endif
/* 1: each slot's w is written at the slot's position in the source-grouped
 * list, so a node reads its out-edges' w contiguously; 0: w in slot order,
 * gathered through the list */
#ifndef BP_ADJ_W_SRC
#define BP_ADJ_W_SRC 1
#endif

namespace bpk {

struct AdjArgs {
    const unsigned *in_off, *slot_src, *out_off, *out_slot;
    const unsigned *slot_pos; /* position of each slot in the source-grouped list (out_slot's inverse) */
    const float *J;
    const uint2 *chunk;
    unsigned nchunks;
    const float *st_prev; /* st_{t-1} */
    const float *st_cur;  /* st_t (step 0: st_0) */
    const float *bsrc;    /* buf_{t-1} (step 0: st_0) */
    const float *gst_in;  /* dL/dst_t along paths through later iterates and the loss */
    float *gst_out;       /* dL/dst_{t-1} through st_t (step 0: dL/dst_0 without w_0) */
    const float *w_in;    /* w_{t+1} or NULL */
    float *w_out;         /* w_t */
    float *jbar;          /* [E][S*S] */
    int jbar_first;       /* write instead of accumulate */
};

/* acc += rows[o] for o in [o0, o1), in order; four rows loaded before any
 * is added */
template <int S, int SP>
__device__ __forceinline__ void sum_rows_contig(const float *__restrict__ rows, unsigned o0, unsigned o1, float *acc)
{
    for (unsigned o = o0; o < o1; o += 4) {
        float x[4][S];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            load_rowp<S, SP>(rows + (size_t)((o + u < o1) ? o + u : o) * SP, x[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (o + u < o1)
#pragma unroll
                for (int k = 0; k < S; ++k)
                    acc[k] = acc[k] + x[u][k];
    }
}

/* the node's sum of its out-edges' w (BP_ADJ_W_SRC: stored in list order) */
template <int S, int SP>
__device__ __forceinline__ void sum_out_w(const float *__restrict__ w, const unsigned *__restrict__ out_slot,
                                          unsigned o0, unsigned o1, float *acc);

/* acc += rows[out_slot[o]] for o in [o0, o1), in order; four index loads,
 * then four row loads, are issued before any is added */
template <int S, int SP>
__device__ __forceinline__ void sum_out_rows(const float *__restrict__ rows, const unsigned *__restrict__ out_slot,
                                             unsigned o0, unsigned o1, float *acc)
{
    for (unsigned o = o0; o < o1; o += 4) {
        unsigned idx[4];
        float x[4][S];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            idx[u] = out_slot[(o + u < o1) ? o + u : o];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            load_rowp<S, SP>(rows + (size_t)idx[u] * SP, x[u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (o + u < o1)
#pragma unroll
                for (int k = 0; k < S; ++k)
                    acc[k] = acc[k] + x[u][k];
    }
}

template <int S, int SP>
__device__ __forceinline__ void sum_out_w(const float *__restrict__ w, const unsigned *__restrict__ out_slot,
                                          unsigned o0, unsigned o1, float *acc)
{
    if constexpr (BP_ADJ_W_SRC)
        sum_rows_contig<S, SP>(w, o0, o1, acc);
    else
        sum_out_rows<S, SP>(w, out_slot, o0, o1, acc);
}

/* LM, LDT: S * 64 R floats of the wave's in LDS; LN: 64 R, LQ: 128 R. */
template <int S, int STEP0, int R>
__device__ __forceinline__ void adjoint_chunk(const AdjArgs &a, unsigned c, float *LM, float *LDT, unsigned short *LN,
                                              unsigned short *LQ, unsigned lane)
{
    constexpr int SP = Stride<S>::value;
    constexpr int W = WAVE * R;
            uint2 lo = bpk::uniform_load(a.chunk + c), hi = bpk::uniform_load(a.chunk + c + 1);
            unsigned nb = lo.x, sb = lo.y, ne = hi.x, se = hi.y;
            /* slot phase 1: the message of every slot, kept with its operands */
            float Jr[R][S * S], b[R][S], m[R][S], sig[R];
            bool pos[R];
            unsigned u[R];
            /* lanes past the chunk's end load a valid neighbour (results
             * dropped): branch-free loads, all in flight before the gathers */
            const bool any_slots = se > sb; /* uniform: no stand-in slot otherwise */
            const unsigned s_last = se - 1;
            if (any_slots) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    unsigned s = sb + r * WAVE + lane;
                    if (s >= se)
                        s = s_last;
                    u[r] = a.slot_src[s];
                    load_row<S * S>(a.J + (size_t)s * S * S, Jr[r]);
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
                    load_rowp<S, SP>(a.bsrc + (size_t)u[r] * SP, b[r]);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                unsigned s = sb + r * WAVE + lane;
                if (s < se) {
                    float sum = 0.0f;
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        float acc = 0.0f;
#pragma unroll
                        for (int j = 0; j < S; ++j)
                            acc = acc + Jr[r][i * S + j] * b[r][j];
                        m[r][i] = acc;
                        sum = sum + acc;
                    }
                    pos[r] = sum > 0.0f;
                    if (!pos[r])
                        sum = 1.0f;
                    sig[r] = sum;
#pragma unroll
                    for (int i = 0; i < S; ++i) {
                        m[r][i] = m[r][i] / sum;
                        LM[i * W + r * WAVE + lane] = m[r][i];
                    }
                }
            }
            wave_sync();
            /* node phase: dT, dst_{t-1} */
#pragma unroll
            for (int r = 0; r < R; ++r) {
                unsigned v = nb + r * WAVE + lane;
                if (v < ne) {
                    unsigned q0 = a.in_off[v] - sb, q1 = a.in_off[v + 1] - sb;
                    unsigned o0 = a.out_off[v], o1 = a.out_off[v + 1];
                    float st[S], g[S], T[S], gb[S], dT[S];
                    load_rowp<S, SP>(a.st_cur + (size_t)v * SP, st);
                    load_rowp<S, SP>(a.gst_in + (size_t)v * SP, g);
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        T[k] = 1.0f;
                        gb[k] = 0.0f;
                    }
                    for (unsigned q = q0; q < q1; ++q) {
#pragma unroll
                        for (int k = 0; k < S; ++k) {
                            float mk = LM[k * W + q];
                            if (mk == mk)
                                T[k] = T[k] * mk;
                        }
                    }
                    if (a.w_in)
                        sum_out_w<S, SP>(a.w_in, a.out_slot, o0, o1, gb);
                    float out[S];
                    if (STEP0) {
#pragma unroll
                        for (int k = 0; k < S; ++k) {
                            dT[k] = gb[k] * st[k];
                            out[k] = g[k] + gb[k] * T[k];
                        }
                    } else {
                        float sp[S], ds[S], av[S];
                        load_rowp<S, SP>(a.st_prev + (size_t)v * SP, sp);
                        bool indeg = q1 > q0;
                        float sa = 0.0f, dot = 0.0f;
#pragma unroll
                        for (int k = 0; k < S; ++k) {
                            ds[k] = g[k] + gb[k] * T[k];
                            dT[k] = gb[k] * st[k];
                            av[k] = indeg ? sp[k] * T[k] : sp[k];
                            sa = sa + av[k];
                            dot = dot + ds[k] * st[k];
                        }
#pragma unroll
                        for (int k = 0; k < S; ++k) {
                            float da = (sa > 0.0f) ? (ds[k] - dot) / sa : ds[k];
                            out[k] = indeg ? da * T[k] : da;
                            if (indeg)
                                dT[k] = dT[k] + da * sp[k];
                        }
                    }
#pragma unroll
                    for (int k = 0; k < SP; ++k)
                        a.gst_out[(size_t)v * SP + k] = (k < S) ? out[k] : 0.0f;
                    unsigned l = r * WAVE + lane;
#pragma unroll
                    for (int k = 0; k < S; ++k)
                        LDT[k * W + l] = dT[k];
                    LQ[2 * l] = (unsigned short)q0;
                    LQ[2 * l + 1] = (unsigned short)q1;
                    for (unsigned q = q0; q < q1; ++q)
                        LN[q] = (unsigned short)l;
                }
            }
            wave_sync();
            /* slot phase 2: dm, dz, dJ, w */
#pragma unroll
            for (int r = 0; r < R; ++r) {
                unsigned s = sb + r * WAVE + lane;
                if (s < se) {
                    unsigned q = r * WAVE + lane;
                    unsigned l = LN[q], q0 = LQ[2 * l], q1 = LQ[2 * l + 1];
                    float P[S];
#pragma unroll
                    for (int k = 0; k < S; ++k)
                        P[k] = 1.0f;
                    for (unsigned p = q0; p < q1; ++p) {
                        if (p == q)
                            continue;
#pragma unroll
                        for (int k = 0; k < S; ++k) {
                            float mk = LM[k * W + p];
                            if (mk == mk)
                                P[k] = P[k] * mk;
                        }
                    }
                    float dm[S], dz[S], dot = 0.0f;
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        dm[k] = (m[r][k] == m[r][k]) ? LDT[k * W + l] * P[k] : 0.0f;
                        dot = dot + dm[k] * m[r][k];
                    }
#pragma unroll
                    for (int k = 0; k < S; ++k)
                        dz[k] = pos[r] ? (dm[k] - dot) / sig[r] : dm[k];
                    float *jb = a.jbar + (size_t)s * S * S;
                    float gJ[S * S];
                    if (!a.jbar_first)
                        load_row<S * S>(jb, gJ);
#pragma unroll
                    for (int i = 0; i < S; ++i)
#pragma unroll
                        for (int j = 0; j < S; ++j)
                            gJ[i * S + j] = a.jbar_first ? dz[i] * b[r][j] : gJ[i * S + j] + dz[i] * b[r][j];
#pragma unroll
                    for (int i = 0; i < S * S; ++i)
                        jb[i] = gJ[i];
                    float wv[SP];
#pragma unroll
                    for (int j = 0; j < SP; ++j) {
                        float acc = 0.0f;
                        if (j < S) {
#pragma unroll
                            for (int i = 0; i < S; ++i)
                                acc = acc + Jr[r][i * S + j] * dz[i];
                        }
                        wv[j] = acc;
                    }
                    size_t wrow = BP_ADJ_W_SRC ? (size_t)a.slot_pos[s] : (size_t)s;
#pragma unroll
                    for (int j = 0; j < SP; ++j)
                        a.w_out[wrow * SP + j] = wv[j];
                }
            }
            wave_sync();
}

} // namespace bpk
