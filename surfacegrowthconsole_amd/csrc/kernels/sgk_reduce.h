// sgk_reduce.h - per-block partial reductions (the force and props kernels) and the per-step
// bookkeeping that k_finalize / kb_finalize run over them.
#pragma once

#include "sgk.h"
#include "sgk_device.h"

namespace sgk {

template <class T>
__device__ __forceinline__ void partial_identity(Partial<T> &q) {
    q.u = q.fr = q.vv = q.vmax = q.vir = T(0);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        q.com[d] = q.cmv[d] = q.vs[d] = T(0);
        q.bmin[d] = T(3.0e38f);
        q.bmax[d] = T(-3.0e38f);
    }
}

template <class T>
__device__ __forceinline__ void partial_combine(Partial<T> &r, const Partial<T> &s) {
    r.u += s.u;
    r.vir += s.vir;
    r.fr += s.fr;
    r.vv += s.vv;
    r.vmax = s.vmax > r.vmax ? s.vmax : r.vmax;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        r.com[d] += s.com[d];
        r.cmv[d] += s.cmv[d];
        r.vs[d] += s.vs[d];
        r.bmin[d] = s.bmin[d] < r.bmin[d] ? s.bmin[d] : r.bmin[d];
        r.bmax[d] = s.bmax[d] > r.bmax[d] ? s.bmax[d] : r.bmax[d];
    }
}

// Wave reduction of a Partial (result in lane 63).
template <class T>
__device__ __forceinline__ void partial_wave(Partial<T> &q) {
    q.u = wave_reduce63<OpSum>(q.u);
    q.vir = wave_reduce63<OpSum>(q.vir);
    q.vv = wave_reduce63<OpSum>(q.vv);
    q.vmax = wave_reduce63<OpMax>(q.vmax);
    q.fr = wave_reduce63<OpSum>(q.fr);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        q.vs[d] = wave_reduce63<OpSum>(q.vs[d]);
        q.com[d] = wave_reduce63<OpSum>(q.com[d]);
        q.cmv[d] = wave_reduce63<OpSum>(q.cmv[d]);
        q.bmin[d] = wave_reduce63<OpMin>(q.bmin[d]);
        q.bmax[d] = wave_reduce63<OpMax>(q.bmax[d]);
    }
}

// Reduce one Partial per thread of the block; thread 0 returns the total (fixed order).  Every
// thread of the block must call it.
template <class T>
__device__ Partial<T> block_reduce_partial(Partial<T> q) {
    __shared__ Partial<T> sh[16];
    partial_wave(q);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if (lane == 63) sh[w] = q;
    __syncthreads();
    Partial<T> r = sh[0];
    if (threadIdx.x == 0)
        for (int k = 1; k < nw; ++k) partial_combine(r, sh[k]);
    return r;
}

// The block's Partial into *out and its v^2 maximum into *vmax (if given), for the force pass: one atom
// per G lanes, its contribution in the group's last lane (METAL), or one carbon per lane (G = 1).
// The sums are those of block_reduce_partial, bit for bit, by fewer instructions (20 FP64 fields by 6
// exchange steps each were 8 % of the force pass's VALU work and 2-3 us of a small launch's latency):
//   metal   the exchange steps within a group are left out, its other lanes hold nothing;
//   carbon  the six sums are exchanged in halves: after the steps over 2, 4 and 8 lanes a lane holds
//           one sum over its 8 lanes instead of all six, and the rows of 16 meet in LDS;
//   both    20 threads combine the waves, one field each, instead of one thread all of them.
// Force launch at 1.1 M atoms 99.8 -> 96.4 us; whole step 26.0 -> 25.6 us at 1,161 atoms, 35.2 -> 34.2
// at 44,353, 112.3 -> 110.0 for 64 replicas.
constexpr int kPartVv = 11, kPartVmax = 12, kPartBmin = 13, kPartBmax = 16, kPartVir = 19, kPartFields = 20;

// Half of a pair of sums: a lane with `hi` keeps b and gives a away, the others the reverse.
template <int CTRL, class T>
__device__ __forceinline__ T half_sum(bool hi, T a, T b) {
    const T keep = hi ? b : a, give = hi ? a : b;
    return keep + dpp_all<CTRL>(give);
}

template <bool METAL, int G, class T>
__device__ __forceinline__ void block_store_partial(Partial<T> q, Partial<T> *out, T *vmax) {
    static_assert(sizeof(Partial<T>) == kPartFields * sizeof(T), "fields of Partial in their order");
    __shared__ Partial<T> sh[4];
    __shared__ T row[4][4][8];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, f = threadIdx.x;
    if (METAL) {
        q.u = wave_reduce63_of<OpSum, G>(q.u);
        q.vir = wave_reduce63_of<OpSum, G>(q.vir);
        q.vv = wave_reduce63_of<OpSum, G>(q.vv);
        q.vmax = wave_reduce63_of<OpMax, G>(q.vmax);
        q.fr = wave_reduce63_of<OpSum, G>(q.fr);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            q.vs[d] = wave_reduce63_of<OpSum, G>(q.vs[d]);
            q.com[d] = wave_reduce63_of<OpSum, G>(q.com[d]);
            q.cmv[d] = wave_reduce63_of<OpSum, G>(q.cmv[d]);
            q.bmin[d] = wave_reduce63_of<OpMin, G>(q.bmin[d]);
            q.bmax[d] = wave_reduce63_of<OpMax, G>(q.bmax[d]);
        }
        if (lane == 63) sh[w] = q;
    } else {
        // a lane's place among its 8 lanes, counted backwards in the upper four: lanes that the
        // mirror of 8 pairs then hold the same sums
        const int m = lane & 4 ? ~lane : lane;
        const bool h1 = m & 1, h2 = m & 2, h4 = lane & 4;
        const T a0 = half_sum<kQuadSwap1>(h1, q.u, q.vs[0]), a1 = half_sum<kQuadSwap1>(h1, q.vir, q.vs[1]),
                a2 = half_sum<kQuadSwap1>(h1, q.vv, q.vs[2]);
        const T b0 = half_sum<kQuadSwap2>(h2, a0, a2);
        T b1 = a1 + dpp_all<kQuadSwap2>(a1);
        T c = half_sum<kRowHalfMirror>(h4, b0, b1);
        c = c + dpp_all<kRowRor8>(c);
        q.vmax = wave_reduce63<OpMax>(q.vmax);
        if ((lane & 15) < 8) row[w][lane >> 4][lane & 7] = c;
        if (lane == 63) sh[w].vmax = q.vmax;
    }
    __syncthreads();
    if (f >= kPartFields) return;
    T r;
    if (METAL || f == kPartVmax) {
        const T *s = (const T *)sh;
        r = s[f];
        for (int k = 1; k < 4; ++k) {
            const T x = s[k * kPartFields + f];
            if (f >= kPartBmin && f < kPartBmax)
                r = x < r ? x : r;
            else if (f == kPartVmax || (f >= kPartBmax && f < kPartVir))
                r = x > r ? x : r;
            else
                r += x;
        }
    } else {
        // field -> the lane of the 8 that holds its sum (-1: a field carbons leave at its identity)
        const int at = f == 0 ? 0 : f == 8 ? 1 : f == kPartVv ? 2 : f == 10 ? 3 : f == kPartVir ? 7 : f == 9 ? 6 : -1;
        r = f >= kPartBmin && f < kPartBmax ? T(3.0e38f) : (f >= kPartBmax && f < kPartVir ? T(-3.0e38f) : T(0));
        if (at >= 0) {
            for (int k = 0; k < 4; ++k) {
                const T x = (row[k][3][at] + row[k][2][at]) + (row[k][1][at] + row[k][0][at]);
                r = k ? r + x : x;
            }
        }
    }
    ((T *)out)[f] = r;
    if (vmax && f == kPartVmax) *vmax = r;
}

// First stage of the step reduction: one wave reduces a chunk of up to kPartChunk partials (lane k
// takes partial k; fixed order), the result goes to *out.  The chunk count is wave-uniform.
constexpr int kPartChunk = 64;
template <class T>
__device__ __forceinline__ void reduce_chunk(const Partial<T> *part, int n, Partial<T> *out) {
    const int lane = threadIdx.x & 63;
    Partial<T> q;
    partial_identity(q);
    if (lane < n) q = part[lane];
    partial_wave(q);
    if (lane == 63) *out = q;
}

// The next state's step, rebuild flag and displacement bound after a step with v^2 maximum vmax
// (SurfaceGrowth.cu:2383-2395); the state itself is only read.  Every kernel that closes a step
// calls it, so all round alike.
template <class A>
struct StepNext {
    int step, nebrNow, cellbuf, rebuilds, displaced;
    double dispHi;
};
__device__ __forceinline__ float fmaA(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaA(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <class A>
__device__ __forceinline__ StepNext<A> step_next(const DevParams &p, const DevState *st, A vmax) {
    StepNext<A> n;
    n.step = st->step + 1;
    A dispHi = (A)st->dispHi;
    n.cellbuf = st->cellbuf;
    n.rebuilds = st->rebuilds;
    if (st->nebrNow) {  // this step rebuilt: the new cell buffer becomes current (SurfaceGrowth.cu:2193-2195)
        n.cellbuf ^= 1;
        n.rebuilds += 1;
        dispHi = A(0);
    }
    const A root = (A)sqrt(vmax), dt = (A)p.deltaT;
    dispHi = fmaA(root, dt, dispHi);  // SurfaceGrowth.cu:2390-2391
    // the reference's skin rule; a fixed cadence adds rebuilds but never removes one
    n.nebrNow = dispHi > A(0.5f) * (A)p.rNebrShell;
    if (p.rebuildEvery > 0 && n.step % p.rebuildEvery == 0) n.nebrNow = 1;
    n.displaced = (double)fmaA(root, dt, dispHi) > (double)p.dispBound && !n.nebrNow;
    n.dispHi = (double)dispHi;
    return n;
}

// Total of nParts partials, in thread 0: each thread a strided subset, then the block tree (the order
// is fixed, so the result is bitwise reproducible).
template <class A>
__device__ __forceinline__ Partial<A> reduce_parts(const Partial<A> *part, int nParts) {
    Partial<A> q;
    partial_identity(q);
    for (int k = threadIdx.x; k < nParts; k += blockDim.x) partial_combine(q, part[k]);
    return block_reduce_partial(q);
}

// The sums of a record, with the reference's host arithmetic (SurfaceGrowth.cu:2307-2395); returns the
// metal's x velocity and the kinetic sum that the thermostat takes.
template <class A>
__device__ __forceinline__ void record_sums(const DevParams &p, const Partial<A> &P, sgk_record &rec, A &cmVelX,
                                            A &vvSum) {
    const int nMe = p.nMolMe, nMol = p.nMol;
    rec.shear = 0;
    rec.shearCount = 0;
    // cmVel.val = cmVel.x / nMolMe (SurfaceGrowth.cu:2308)
    cmVelX = nMe ? P.cmv[0] / (A)nMe : A(0);
    // ComputeVvSumK subtracts cmVel.val from metal vx in regime 2 (SurfaceGrowth.cu:1230-1234):
    // sum m((vx-c)^2+vy^2+vz^2) = sum m|v|^2 - m c sum vx, since sum vx = nMe c.
    vvSum = P.vv;
    if (p.iRegime == 2 && nMe) vvSum = vvSum - (A)p.massMe * cmVelX * P.cmv[0];
    // the metal bounding box includes the reference reduction's zero padding (SurfaceGrowth.cu:1671-1682)
    const bool pad = nMe != 1024 * 1024;
    for (int d = 0; d < 3; ++d) {
        rec.vSum[d] = (double)P.vs[d];
        rec.comSum[d] = nMe ? (double)P.com[d] : 0.0;
        rec.cmVelSum[d] = nMe ? (double)P.cmv[d] : 0.0;
        A mn = P.bmin[d], mx = P.bmax[d];
        if (pad) {
            mn = mn < A(0) ? mn : A(0);
            mx = mx > A(0) ? mx : A(0);
        }
        rec.bboxMin[d] = nMe ? (double)mn : 0.0;
        rec.bboxMax[d] = nMe ? (double)mx : 0.0;
    }
    const A ke = A(0.5f) * vvSum / (A)nMol, pe = P.u / (A)nMol;
    rec.kinEnergy = (double)ke;
    rec.potEnergy = (double)pe;
    rec.totEnergy = (double)(ke + pe);
    rec.vvSum = (double)vvSum;
    rec.vvMax = (double)P.vmax;
    rec.uSum = (double)P.u;
    rec.virial = (double)P.vir;
    rec.frict = (p.iRegime != 0 && nMe) ? (double)P.fr : 0.0;
    rec.pad = 0;
}

// Reduce nParts partials with the whole block, then evaluate the reference's host arithmetic of
// SurfaceGrowth.cu:2307-2395 in thread 0.
// mode 0: one step - advance the step counter, commit a rebuild, update dispHi / nebrNow / shear,
//         append a record.  mode 1: evaluation only - write records[0], leave the state alone.
template <class A>
__device__ void finalize_body(const DevParams &p, const Partial<A> *part, int nParts, DevState *st,
                              sgk_record *records, int recCap, int mode) {
    const Partial<A> P = reduce_parts(part, nParts);
    if (threadIdx.x != 0) return;
    const int nMe = p.nMolMe;
    sgk_record rec;
    A cmVelX, vvSum;
    record_sums(p, P, rec, cmVelX, vvSum);
    if (mode == 1) {
        rec.step = st->step;
        rec.rebuilt = 0;
        rec.nebrNow = st->nebrNow;
        rec.errors = st->errors | st->errPrev;
        rec.dispHi = st->dispHi;
        rec.nMolDeposited = st->nMolDeposited;
        records[0] = rec;
        return;
    }
    const StepNext<A> n = step_next(p, st, P.vmax);
    const int step = n.step;
    rec.step = step;
    rec.rebuilt = st->nebrNow;
    st->step = step;
    st->cellbuf = n.cellbuf;
    st->rebuilds = n.rebuilds;
    if (n.displaced) st->errors |= SGK_FLAG_DISPLACEMENT;
    st->nebrNow = n.nebrNow;
    st->dispHi = n.dispHi;
    st->vvSum = (double)vvSum;
    st->cmVelX = (double)cmVelX;
    st->comX = nMe ? (double)(P.com[0] / (A)nMe) : 0.0;
    // shear increment (SurfaceGrowth.cu:2398-2404)
    if (p.iRegime == 2 && nMe && step > p.stepEquil + p.stepCool) {
        if ((float)cmVelX < 0.005f) st->shear = (double)((A)st->shear + (A)p.deltaF);
    }
    // deposition schedule (SurfaceGrowth.cu:2148-2168): the step's group counts from now on
    if (p.iRegime == 1 && step > p.stepEquil && st->nMolDeposited < nMe && p.stepDeposit > 0 &&
        (step - p.stepEquil) % p.stepDeposit == 0)
        st->nMolDeposited += p.nMolToDeposit;
    rec.nMolDeposited = st->nMolDeposited;
    rec.shear = st->shear;
    rec.nebrNow = n.nebrNow;
    rec.dispHi = n.dispHi;
    rec.errors = st->errors | st->errPrev;
    if (st->rec < recCap) records[st->rec] = rec;
    st->rec += 1;
}

// ---- step closing folded into the next step --------------------------------------------------------
// After a step that no thermostat, shear, deposition or sample follows, nothing needs the step's sums
// before the next force pass, only its v^2 maximum (the skin rule).  Such a step has no closing
// launches of its own: the next step's k_bin_next takes the maximum and advances the state into the
// other DevState, and one workgroup of the next force launch reduces the sums and writes the record
// while the others work (the force launch, not the density one: its registers cover the reduction, and it
// is longer than the reduction's ~11 us at 1,000 partials).  The two closing launches cost a small
// step ~6 us of latency.  Whole step, closed by launches / folded (us): 1,161 atoms 34.6 / 29.0,
// 44,353 41.4 / 35.2, 137,940 (FP32) 50.3 / 45.3, 1.1 M 224.2 / 223.5.
constexpr int kCloseLdsChunks = 16;                           // chunk totals kept in LDS
// Partials closed without k_reduce1: beyond, every workgroup of k_bin_next would read more than 8 KB
// of maxima and the closing workgroup's chunks would outlast the force launch.
constexpr int kCloseDirectParts = kCloseLdsChunks * kPartChunk;

template <class A>
struct StepClose {
    const Partial<A> *part;  // force-pass partials, or chunk totals (direct = 0)
    int n, direct;           // their number; 1: reduce the chunks here
    DevState *old, *st;      // the closed step's state, and the advanced one
    sgk_record *records;
    int recCap, on;
};

// The record of the closed step and the sums of the advanced state; called by one whole workgroup.
// The sums are those of k_reduce1 and k_finalize, bit for bit.
template <class A>
__device__ __forceinline__ void close_body(const DevParams &p, const StepClose<A> &c) {
    __shared__ Partial<A> tot[kCloseLdsChunks];
    const Partial<A> *src = c.part;
    int n = c.n;
    if (c.direct) {  // as k_reduce1, one wave per chunk
        n = (c.n + kPartChunk - 1) / kPartChunk;
        for (int j = threadIdx.x >> 6; j < n; j += (int)blockDim.x >> 6)
            reduce_chunk(c.part + j * kPartChunk, min(kPartChunk, c.n - j * kPartChunk), tot + j);
        __syncthreads();
        src = tot;
    }
    const Partial<A> P = reduce_parts(src, n);
    if (threadIdx.x != 0) return;
    sgk_record rec;
    A cmVelX, vvSum;
    record_sums(p, P, rec, cmVelX, vvSum);
    rec.step = c.st->step;
    rec.rebuilt = c.old->nebrNow;
    rec.nebrNow = c.st->nebrNow;
    rec.errors = c.st->errPrev;
    rec.dispHi = c.st->dispHi;
    rec.shear = c.old->shear;
    rec.nMolDeposited = c.old->nMolDeposited;
    const int slot = c.old->rec;
    if (slot < c.recCap) c.records[slot] = rec;
    c.st->vvSum = (double)vvSum;
    c.st->cmVelX = (double)cmVelX;
    c.st->comX = p.nMolMe ? (double)(P.com[0] / (A)p.nMolMe) : 0.0;
    c.old->errors = 0;  // taken over into errPrev; this state is the next advance's target
}

}  // namespace sgk
