/*
 * bp_resident.h -- what the resident kernels (bp_resident.hip: loopy
 * iterations; bp_resident_diff.hip: the adjoint) share: the grid barrier, rows
 * exchanged through memory and in LDS, the in-messages of a node.
 */
#pragma once

#include "bp_dev.h"

namespace bpk {

constexpr int RB = 1024;            /* threads per workgroup */
constexpr int RW = RB / WAVE;
constexpr unsigned MAX_G = 256;
constexpr unsigned COUNTERS = 16, COUNTER_STRIDE = 64; /* unsigneds between two counters */
constexpr int PAD = 8; /* rows past the messages that a node's first read may touch */

/* Where the workgroups of a run meet. */
struct Meeting {
    unsigned *counters;
    unsigned met;     /* barriers that the counters have counted */
    unsigned *decision;
    unsigned run;
    unsigned after;   /* the run that this one goes on from, 0: none outstanding */
    unsigned long long timeout;
};

enum { GO_ON = 0, COMMIT = 1 };

/* Settles the run for all workgroups: the first word wins. */
__device__ __forceinline__ bool settle(unsigned *decision, unsigned run, unsigned commit)
{
    const unsigned mine = run << 1 | commit;
    unsigned cur = __hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (cur >> 1 != run)
        if (__hip_atomic_compare_exchange_strong(decision, &cur, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return commit;
    return cur & 1u;
}

/* The run before this one was given up: so is this one. */
__device__ __forceinline__ bool called_off(const Meeting &a)
{
    return a.after &&
           __hip_atomic_load(a.decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (a.after << 1 | COMMIT);
}

/* The grid barrier in two halves, with work between them that needs nothing
 * of other workgroups.  All threads of the workgroup call both; arriving is
 * also a workgroup barrier. */
__device__ __forceinline__ void grid_arrive(const Meeting &a, unsigned wg)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); /* this wave's rows are in memory */
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_fetch_add(a.counters + (wg % COUNTERS) * COUNTER_STRIDE, 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

/* Waits until every workgroup has been at barrier number `number` (from 1).
 * False: this run has been given up.  `ok` is shared. */
__device__ __forceinline__ bool grid_wait(const Meeting &a, unsigned G, unsigned number, unsigned *ok)
{
    if (threadIdx.x < WAVE) {
        const unsigned lane = threadIdx.x;
        const unsigned members = lane < COUNTERS ? (G - lane + COUNTERS - 1) / COUNTERS : 0u;
        const unsigned want = (a.met + number) * members;
        const unsigned long long t0 = wall_clock64();
        bool there = false;
        while (!there) {
            bool all = true;
            if (members)
                all = (int)(__hip_atomic_load(a.counters + lane * COUNTER_STRIDE, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT) - want) >= 0;
            there = __ballot(!all) == 0;
            if (!there && wall_clock64() - t0 > a.timeout) {
                /* given up, unless another workgroup is already past the
                 * last barrier: then all have been here */
                unsigned c = lane == 0 ? (unsigned)settle(a.decision, a.run, GO_ON) : 0u;
                there = __builtin_amdgcn_readfirstlane(c) != 0;
                break;
            }
        }
        if (lane == 0)
            *ok = there;
    }
    __syncthreads();
    asm volatile("" ::: "memory"); /* no gather moves above the barrier */
    return *ok != 0;
}

__device__ __forceinline__ bool grid_step(const Meeting &a, unsigned wg, unsigned G, unsigned number, unsigned *ok)
{
    grid_arrive(a, wg);
    return grid_wait(a, G, number, ok);
}

template <int N> __device__ __forceinline__ void store_row_agent(float *p, const float *v)
{
    static_assert(N % 2 == 0, "rows are float pairs");
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const unsigned long long lo = __float_as_uint(v[2 * i]), hi = __float_as_uint(v[2 * i + 1]);
        __hip_atomic_store(reinterpret_cast<unsigned long long *>(p) + i, lo | hi << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

/* Keeps packed values packed: the compiler takes them for new in every
 * iteration, instead of unpacking them once into registers that the tables
 * need (77 spilled in the adjoint otherwise). */
template <int N> __device__ __forceinline__ void hold(unsigned (&v)[N])
{
#pragma unroll
    for (int i = 0; i < N; ++i)
        asm volatile("" : "+v"(v[i]));
}

/* rows of S floats in LDS */
template <int S> __device__ __forceinline__ void put_row(float *p, const float *v)
{
    if constexpr (S == 2)
        *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
    else if constexpr (S % 4 == 0)
#pragma unroll
        for (int i = 0; i < S; i += 4)
            *reinterpret_cast<float4 *>(p + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
    else
#pragma unroll
        for (int i = 0; i < S; ++i)
            p[i] = v[i];
}

template <int S> __device__ __forceinline__ void get_row(const float *p, float *v) { load_row<S>(p, v); }

/* N in-messages from p on, S floats apart, as factors, H entries of each:
 * those past the node's last one are 1, and so are NaN entries (CLEAN: there
 * may be some), which the products skip.  All reads are issued before the
 * first product: a read at a time made the node phase a chain of LDS
 * latencies as long as the largest in-degree of the wave's nodes (1.5 of
 * 2.3 us on a 700-node network). */
template <int S, int H, int N, bool CLEAN>
__device__ __forceinline__ void factors(const float *p, unsigned cnt, float (&f)[N][H])
{
#pragma unroll
    for (int j = 0; j < N; ++j)
        get_row<H>(p + j * S, f[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) {
#pragma unroll
        for (int i = 0; i < H; ++i)
            f[j][i] = (unsigned)j < cnt ? f[j][i] : 1.0f;
        if (CLEAN)
            nan_to_one<H>(f[j]);
    }
}

} // namespace bpk

/* The host's side of a meeting (bp_resident.hip): the next run of the
 * handle, with `barriers` of them, and its turn on the device; foreign: on a
 * stream that is not the handle's own. */
bpk::Meeting bp_resident_meeting(bp_dev *d, unsigned barriers, unsigned after);
int bp_resident_turn(int device, hipStream_t stream);
int bp_resident_turn_taken(int device, hipStream_t stream, bool foreign);

/* The unrolled forward and its adjoint (bp_diff.hip) as resident runs on a
 * caller's stream.  st, buf: the iterates' beliefs and combine buffers, K + 1
 * arrays `stride` floats apart, all kept.  A run that is given up is made up
 * for on the device by one workgroup, which needs no other. */
bool bp_resident_diff_fits(const bp_dev *d, unsigned max_in_degree);
int bp_resident_diff_forward(bp_dev *d, unsigned K, float *st, float *buf, size_t stride, hipStream_t stream);
struct bp_adjoint_arrays {
    const unsigned *out_off, *out_slot, *slot_pos;
    const uint2 *chunk;    /* at most 64 R slots and nodes each */
    unsigned nchunks;
    const float *st0, *gin; /* initial beliefs; dL/dst_K */
    float *gst[2], *w[2];
    float *jbar, *dst0p, *dst0;
    const unsigned *out_at; /* bp_resident_diff_places */
    float *rows;            /* K + 1 times bp_resident_diff_rows floats */
};
size_t bp_resident_diff_rows(const bp_dev *d);
int bp_resident_diff_places(bp_dev *d, const unsigned *slot_pos, unsigned *out_at);
int bp_resident_diff_backward(bp_dev *d, unsigned K, const float *st, const float *buf, size_t stride,
                              const bp_adjoint_arrays &x, hipStream_t stream);
int bp_resident_forward(bp_dev *d, unsigned K, float *st, float *buf, size_t stride, hipStream_t stream,
                        bpk::Meeting *meeting);
