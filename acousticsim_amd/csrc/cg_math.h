// Device code that the tolerance-mode solvers share (cg.hip: one launch per
// phase; resident.hip: one launch per solve).
#pragma once
#include "device.h"

namespace bw
{

// field-wise state copies: whole-struct copies make the compiler keep a
// per-thread copy of the state in LDS or scratch
template <typename SP> __device__ inline CgState load_state(SP p)
{
    CgState s;
    s.rho = p->rho;
    s.rr_ref = p->rr_ref;
    s.bb = p->bb;
    s.rr_true = p->rr_true;
    s.rr = p->rr;
    s.start = p->start;
    s.first = p->first;
    s.iter = p->iter;
    s.total = p->total;
    s.since = p->since;
    s.updates = p->updates;
    s.done = p->done;
    s.breakdown = p->breakdown;
    s.pending = p->pending;
    s.force_check = p->force_check;
    s.final_check = p->final_check;
    s.w64 = p->w64;
    s.stalls = p->stalls;
    return s;
}

template <typename SP> __device__ inline void store_state(SP p, const CgState &s)
{
    p->rho = s.rho;
    p->rr_ref = s.rr_ref;
    p->bb = s.bb;
    p->rr_true = s.rr_true;
    p->rr = s.rr;
    p->start = s.start;
    p->first = s.first;
    p->iter = s.iter;
    p->total = s.total;
    p->since = s.since;
    p->updates = s.updates;
    p->done = s.done;
    p->breakdown = s.breakdown;
    p->pending = s.pending;
    p->force_check = s.force_check;
    p->final_check = s.final_check;
    p->w64 = s.w64;
    p->stalls = s.stalls;
}

// The solver's arithmetic is written out operation by operation, fused
// multiply-adds included, and the files that include this one are compiled
// without floating-point contraction: every kernel and variant that computes
// the same quantity rounds it the same way, whatever the surrounding code (a
// cloth's result cannot depend on which launch shape or kernel variant
// computed it).
__device__ inline float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

// d = z + beta d_prev, z = P r
template <typename T> __device__ inline T dir_value(T z, T dold, T beta, bool first)
{
    return first ? z : fma_t(beta, dold, z);
}

// one row of a 3x3 block times a 3-vector: (m0 v0 + m1 v1) + m2 v2 with the
// two additions fused
template <typename T> __device__ inline T block_row(T m0, T m1, T m2, T v0, T v1, T v2)
{
    return fma_t(m2, v2, fma_t(m1, v1, m0 * v0));
}

// the solver vectors of precision T
template <typename T> struct Vecs;
template <> struct Vecs<float>
{
    __device__ static const float *W(const DeviceBatch &d) { return d.W32; }
    __device__ static const float *P(const DeviceBatch &d) { return d.P32; }
    __device__ static float *r(const DeviceBatch &d) { return d.r32; }
    __device__ static float *z(const DeviceBatch &d) { return d.z32; }
    __device__ static float *q(const DeviceBatch &d) { return d.q32; }
    __device__ static float *d0(const DeviceBatch &d) { return d.d32[0]; }
    __device__ static float *d1(const DeviceBatch &d) { return d.d32[1]; }
};
template <> struct Vecs<double>
{
    __device__ static const double *W(const DeviceBatch &d) { return d.W64; }
    __device__ static const double *P(const DeviceBatch &d) { return d.P64; }
    __device__ static double *r(const DeviceBatch &d) { return d.r64; }
    __device__ static double *z(const DeviceBatch &d) { return d.z64; }
    __device__ static double *q(const DeviceBatch &d) { return d.q64; }
    __device__ static double *d0(const DeviceBatch &d) { return d.d64[0]; }
    __device__ static double *d1(const DeviceBatch &d) { return d.d64[1]; }
};

} // namespace bw
