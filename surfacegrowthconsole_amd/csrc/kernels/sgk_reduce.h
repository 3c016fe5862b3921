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
    r.vmax = OpMax::f(r.vmax, s.vmax);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        r.com[d] += s.com[d];
        r.cmv[d] += s.cmv[d];
        r.vs[d] += s.vs[d];
        r.bmin[d] = OpMin::f(r.bmin[d], s.bmin[d]);
        r.bmax[d] = OpMax::f(r.bmax[d], s.bmax[d]);
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

// Field f of a workgroup's partial as it is stored: the identity for a maximum or minimum over nothing but NaNs.
// No NaN is then among the values that later joins compare, and every way of closing a step takes the same maximum.
template <class T>
__device__ __forceinline__ T held(int f, T r) {
    if (f < kPartVmax || f >= kPartVir || r == r) return r;
    return f < kPartBmin ? T(0) : (f < kPartBmax ? T(3.0e38f) : T(-3.0e38f));
}

// Half of a pair of sums: a lane with `hi` keeps b and gives a away, the others the reverse.
template <int CTRL, class T>
__device__ __forceinline__ T half_sum(bool hi, T a, T b) {
    const T keep = hi ? b : a, give = hi ? a : b;
    return keep + dpp_all<CTRL>(give);
}

// A workgroup's v^2 maximum: into its place, or joined with a replica's others (as the bits of a double,
// which order non-negative values; 0 is what a step starts from).
template <class T>
__device__ __forceinline__ void store_vmax(T r, T *vmax, unsigned long long *vmaxAll) {
    if (vmax) *vmax = r;
    if (vmaxAll && r > T(0)) atomicMax(vmaxAll, (unsigned long long)__double_as_longlong((double)r));
}

template <bool METAL, int G, class T>
__device__ __forceinline__ void block_store_partial(Partial<T> q, Partial<T> *out, T *vmax,
                                                    unsigned long long *vmaxAll) {
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
                r = OpMin::f(r, x);
            else if (f == kPartVmax || (f >= kPartBmax && f < kPartVir))
                r = OpMax::f(r, x);
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
    r = held(f, r);
    ((T *)out)[f] = r;
    if (f == kPartVmax) store_vmax(r, vmax, vmaxAll);
}

// The same sums for a workgroup with four lanes per carbon (64 carbons), each of which holds its carbon's
// contribution: lane l of a quad takes two fields, the quads of a row of 16 lanes are summed in it and the
// rows in LDS.  The tree is that of one wave of block_store_partial with a carbon per lane.
template <class T>
__device__ __forceinline__ void block_store_quad(Partial<T> q, Partial<T> *out, T *vmax, unsigned long long *vmaxAll) {
    __shared__ T rows[16][8];
    const int l = threadIdx.x & 3, f = threadIdx.x;
    T a = q.vmax, b = q.vs[2];
    if (l == 2) a = q.vv;
    if (l == 1) {
        a = q.vir;
        b = q.vs[1];
    }
    if (l == 0) {
        a = q.u;
        b = q.vs[0];
    }
    const T a4 = dpp<kRowShr4, 0xF>(T(0), a);
    a = l == 3 ? OpMax::f(a, a4) : a + a4;
    b += dpp<kRowShr4, 0xF>(T(0), b);
    const T a8 = dpp<kRowShr8, 0xF>(T(0), a);
    a = l == 3 ? OpMax::f(a, a8) : a + a8;
    b += dpp<kRowShr8, 0xF>(T(0), b);
    if ((threadIdx.x & 15) >= 12) {
        rows[threadIdx.x >> 4][2 * l] = a;
        rows[threadIdx.x >> 4][2 * l + 1] = b;
    }
    __syncthreads();
    if (f >= kPartFields) return;
    const int at = f == 0 ? 0 : f == 8 ? 1 : f == kPartVir ? 2 : f == 9 ? 3 : f == kPartVv ? 4 : f == 10 ? 5 : f == kPartVmax ? 6 : -1;
    T r = f >= kPartBmin && f < kPartBmax ? T(3.0e38f) : (f >= kPartBmax && f < kPartVir ? T(-3.0e38f) : T(0));
    if (at >= 0) {
        T x[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = rows[k][at];
#pragma unroll
        for (int d = 1; d < 16; d *= 2)
#pragma unroll
            for (int k = 0; k < 16; k += 2 * d) x[k] = f == kPartVmax ? OpMax::f(x[k], x[k + d]) : x[k] + x[k + d];
        r = x[0];
    }
    r = held(f, r);
    ((T *)out)[f] = r;
    if (f == kPartVmax) store_vmax(r, vmax, vmaxAll);
}

// First stage of the step reduction: one wave reduces a chunk of up to kPartChunk partials (lane k
// takes partial k; fixed order), the result goes to *out.  The chunk count is wave-uniform.
// Chunk j of the map's partials.
constexpr int kPartChunk = 64;
template <class T>
__device__ __forceinline__ void reduce_chunk(const Partial<T> *part, const PartMap &map, int j, Partial<T> *out) {
    const int lane = threadIdx.x & 63, k = j * kPartChunk + lane;
    Partial<T> q;
    partial_identity(q);
    if (k < map.count()) {
        const Partial<T> *at = part + map.first(k);
        q = at[0];
        for (int s = 1; s < map.parts(k); ++s) partial_combine(q, at[s]);
    }
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

// Total of the map's n partials by one workgroup of 256 threads, returned to every thread.  A thread takes
// one field of four partials: their loads are all in flight at once and a field's tree is a few
// operations in registers, where a lane per partial moved 20 fields through 6 exchange steps each,
// twice, and a launch of one workgroup has nothing to hide them behind.  The trees are reduce_chunk's
// (fours, rows of 16, then the rows of a chunk) and so are the sums, bit for bit.
// totals: the n are chunk totals (any number): thread t of 256 first adds totals t, t + 256, ... in order.
// Otherwise at most kSumParts partials: chunks of 64, then the chunk totals as the first 16 lanes of a wave.
// One launch in place of k_reduce1 and k_finalize, for a few partials or beside other work: a sheared step of 997
// atoms (FP32) 29.1 -> 26.8 us, a deposition step of 4,393 27.2 -> 25.3, kb_finalize of 64 replicas 8.0 -> 6.5.
constexpr int kSumFours = 64, kSumParts = kFoldParts, kSumGroups = 256 / kPartFields;

// One field of a tree: sums add, the others keep the larger value, minima with their sign turned.
template <class A>
struct Field {
    bool sum, turn;
    A id;
    __device__ explicit Field(int f)
        : sum(f < kPartVmax || f >= kPartVir), turn(f >= kPartBmin && f < kPartBmax),
          id(f >= kPartBmin && f < kPartVir ? A(-3.0e38f) : A(0)) {}
    __device__ __forceinline__ A in(A x) const { return turn ? -x : x; }  // its own inverse
    __device__ __forceinline__ A join(A x, A y) const {
        const A s = x + y, m = y > x ? y : x;
        return sum ? s : m;
    }
    __device__ __forceinline__ A four(A a, A b, A c, A d) const { return join(join(a, b), join(c, d)); }
};

// Partials 4q .. 4q + 3 of the map's first `lanes`, one field, joined as the tree takes them.
template <class A>
__device__ __forceinline__ A field_four(const Field<A> &fl, const A *src, const PartMap &map, int q, int lanes) {
    const int k0 = 4 * q;
    if (map.quad && k0 >= map.nbM && k0 + 4 <= lanes) {  // sixteen in a row
        const A *s = src + (size_t)map.first(k0) * kPartFields;
        A v[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) v[t] = fl.in(s[t * kPartFields]);
#pragma unroll
        for (int t = 0; t < 16; t += 4) v[t] = fl.join(fl.join(fl.join(v[t], v[t + 1]), v[t + 2]), v[t + 3]);
        return fl.four(v[0], v[4], v[8], v[12]);
    }
    A x[4];
    if (!map.quad || k0 + 4 <= map.nbM) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = src[(size_t)min(k0 + j, map.stored - 1) * kPartFields];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = k0 + j < lanes ? fl.in(x[j]) : fl.id;
    } else {  // metal and carbon, or the last: all loads in flight, those past an end discarded
        A v[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int s = 0; s < 4; ++s) v[j][s] = src[(size_t)min(map.first(k0 + j) + s, map.stored - 1) * kPartFields];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int have = k0 + j < lanes ? map.parts(k0 + j) : 0;
            x[j] = have > 0 ? fl.in(v[j][0]) : fl.id;
#pragma unroll
            for (int s = 1; s < 4; ++s) x[j] = have > s ? fl.join(x[j], fl.in(v[j][s])) : x[j];
        }
    }
    return fl.four(x[0], x[1], x[2], x[3]);
}

template <class A>
__device__ __forceinline__ Partial<A> sum_parts(const Partial<A> *part, const PartMap &map, bool totals) {
    static_assert(sizeof(Partial<A>) == kPartFields * sizeof(A), "fields of Partial in their order");
    __shared__ A fours[kSumFours][kPartFields], chunks[16][kPartFields];
    __shared__ Partial<A> total;
    const int f = threadIdx.x % kPartFields, g = threadIdx.x / kPartFields;
    const bool mine = g < kSumGroups;
    const Field<A> fl(f);
    const int n = map.count(), lanes = totals ? min(n, 256) : n, nFours = (lanes + 3) / 4, nChunks = (lanes + 63) / 64;
    const A *src = (const A *)part + f;
    // four fours in a row per thread where one would leave it with 4 loads in flight and many rounds
    const bool rows = !map.quad && nFours > 2 * kSumGroups;
    for (int pass = 0; pass * kSumFours < nFours; ++pass) {
        const int q0 = pass * kSumFours, here = min(kSumFours, nFours - q0);
        if (pass) __syncthreads();
        if (mine && totals && n > 256) {
            for (int q = g; q < here; q += kSumGroups) {
                A x[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    x[j] = fl.in(src[(size_t)(4 * q + j) * kPartFields]);
                    for (int k = 4 * q + j + 256; k < n; k += 256) x[j] = fl.join(x[j], fl.in(src[(size_t)k * kPartFields]));
                }
                fours[q][f] = fl.four(x[0], x[1], x[2], x[3]);
            }
        } else if (mine && rows) {
            for (int q = 4 * g; q < here; q += 4 * kSumGroups) {
                const int k0 = 4 * (q0 + q);
                A v[16];
#pragma unroll
                for (int t = 0; t < 16; ++t) v[t] = src[(size_t)min(k0 + t, n - 1) * kPartFields];
#pragma unroll
                for (int t = 0; t < 16; ++t) v[t] = k0 + t < lanes ? fl.in(v[t]) : fl.id;
#pragma unroll
                for (int t = 0; t < 16; t += 4) fours[q + t / 4][f] = fl.four(v[t], v[t + 1], v[t + 2], v[t + 3]);
            }
        } else if (mine) {
            for (int q = g; q < here; q += kSumGroups) fours[q][f] = field_four(fl, src, map, q0 + q, lanes);
        }
        __syncthreads();
        if (g < 4 && 16 * g < here) {
            A r[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                auto four = [&](int j) { return 16 * g + 4 * k + j < here ? fours[16 * g + 4 * k + j][f] : fl.id; };
                r[k] = fl.four(four(0), four(1), four(2), four(3));
            }
            chunks[4 * pass + g][f] = fl.four(r[3], r[2], r[1], r[0]);
        }
    }
    __syncthreads();
    if (g == 0) {
        A r = n > 0 ? chunks[0][f] : fl.id;
        if (totals) {
            for (int c = 1; c < nChunks; ++c) r = fl.join(r, chunks[c][f]);
        } else if (nChunks > 1) {
            A x[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) x[c] = c < nChunks ? chunks[c][f] : fl.id;
#pragma unroll
            for (int d = 1; d < 16; d *= 2)
#pragma unroll
                for (int j = 0; j < 16; j += 2 * d) x[j] = fl.join(x[j], x[j + d]);
            r = x[0];
        }
        ((A *)&total)[f] = fl.in(r);
    }
    __syncthreads();
    return total;
}

// Total of n > 256 chunk totals by one workgroup of 256, returned to thread 0: a thread joins whole partials
// t, t + 256, ... and the workgroup's tree the threads'.  The sums are sum_parts's, bit for bit.  Its loads
// are all in flight, where sum_parts walks a field's totals one by one; up to 256 each thread has one, and there
// sum_parts is the quicker.  sgk_eval_props by sum_parts / so (us, mixed): 44,353 atoms (174 totals) 30.6 / 31.2,
// 82,000 (321) 40.0 / 32.7, 163,280 (638) 49.6 / 34.6, 1.1 M (4,311) 162 / 60.
template <class A>
__device__ Partial<A> sum_strided(const Partial<A> *part, int n) {
    Partial<A> q;
    partial_identity(q);
    for (int k = threadIdx.x; k < n; k += blockDim.x) partial_combine(q, part[k]);
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

// The shear increment after step `step` (SurfaceGrowth.cu:2398-2404) and the atoms deposited by then (the
// step's group counts from now on, SurfaceGrowth.cu:2148-2168).
template <class A>
__device__ __forceinline__ double shear_next(const DevParams &p, int step, double shear, A cmVelX) {
    if (p.iRegime == 2 && p.nMolMe && step > p.stepEquil + p.stepCool && (float)cmVelX < 0.005f)
        shear = (double)((A)shear + (A)p.deltaF);
    return shear;
}
__device__ __forceinline__ int deposited_next(const DevParams &p, int step, int deposited) {
    if (p.iRegime == 1 && step > p.stepEquil && deposited < p.nMolMe && p.stepDeposit > 0 &&
        (step - p.stepEquil) % p.stepDeposit == 0)
        deposited += p.nMolToDeposit;
    return deposited;
}

// Reduce the map's partials (totals: chunk totals) with the whole workgroup of 256, then evaluate the
// reference's host arithmetic of SurfaceGrowth.cu:2307-2395 in thread 0.
// mode 0: one step - advance the step counter, commit a rebuild, update dispHi / nebrNow / shear,
//         append a record.  mode 1: evaluation only - write records[0], leave the state alone.
template <class A, bool STRIDED = false>
__device__ void finalize_body(const DevParams &p, const Partial<A> *part, const PartMap &map, bool totals, DevState *st,
                              sgk_record *records, int recCap, int mode) {
    const DevState s0 = *st;  // before the sums: its latency passes meanwhile
    const Partial<A> P = STRIDED ? sum_strided(part, map.stored) : sum_parts(part, map, totals);
    if (threadIdx.x != 0) return;
    const int nMe = p.nMolMe;
    sgk_record rec;
    A cmVelX, vvSum;
    record_sums(p, P, rec, cmVelX, vvSum);
    if (mode == 1) {
        rec.step = s0.step;
        rec.rebuilt = 0;
        rec.nebrNow = s0.nebrNow;
        rec.errors = s0.errors | s0.errPrev;
        rec.dispHi = s0.dispHi;
        rec.nMolDeposited = s0.nMolDeposited;
        records[0] = rec;
        return;
    }
    const StepNext<A> n = step_next(p, &s0, P.vmax);
    const int step = n.step, errors = s0.errors | (n.displaced ? SGK_FLAG_DISPLACEMENT : 0);
    const double shear = shear_next(p, step, s0.shear, cmVelX);
    const int deposited = deposited_next(p, step, s0.nMolDeposited);
    st->step = step;
    st->cellbuf = n.cellbuf;
    st->rebuilds = n.rebuilds;
    st->errors = errors;
    st->nebrNow = n.nebrNow;
    st->dispHi = n.dispHi;
    st->vvSum = (double)vvSum;
    st->cmVelX = (double)cmVelX;
    st->comX = nMe ? (double)(P.com[0] / (A)nMe) : 0.0;
    st->shear = shear;
    st->nMolDeposited = deposited;
    st->rec = s0.rec + 1;
    rec.step = step;
    rec.rebuilt = s0.nebrNow;
    rec.nMolDeposited = deposited;
    rec.shear = shear;
    rec.nebrNow = n.nebrNow;
    rec.dispHi = n.dispHi;
    rec.errors = errors | s0.errPrev;
    if (s0.rec < recCap) records[s0.rec] = rec;
}

// ---- step closing folded into the next step --------------------------------------------------------
// After a step that no thermostat, shear, deposition or sample follows, nothing needs the step's sums
// before the next force pass, only its v^2 maximum (the skin rule).  Such a step has no closing
// launches of its own: the next step's k_bin_next takes the maximum and advances the state into the
// other DevState, and one workgroup of the next force launch reduces the sums and writes the record
// while the others work (the force launch, not the density one: its registers cover the reduction, and it
// is longer than the reduction's 9 us (FP32) or 12 (mixed) at 1,000 partials).  The two closing launches cost a small
// step ~6 us of latency.  Whole step, closed by launches / folded (us): 1,161 atoms 34.6 / 29.0,
// 44,353 41.4 / 35.2, 137,940 (FP32) 50.3 / 45.3, 1.1 M 224.2 / 223.5.
//
// Partials closed without k_reduce1: beyond, every workgroup of k_bin_next would read more than 8 KB
// of maxima and the closing workgroup's rows would outlast the force launch.
constexpr int kCloseDirectParts = kSumParts;

// A step that only a shear or a deposition follows closes the same way: k_lf1_next (sgk_step.hip) takes the
// place of k_bin_next, up to kCloseLf1Parts partials.

// The advanced state, all but errors, which the launch's binning may raise.
template <class A>
__device__ __forceinline__ void advance_state(DevState *st, const DevState *old, const StepNext<A> &s, double shear,
                                              int deposited) {
    st->step = s.step;
    st->nebrNow = s.nebrNow;
    st->cellbuf = s.cellbuf;
    st->rec = old->rec + 1;
    st->rebuilds = s.rebuilds;
    st->dispHi = s.dispHi;
    st->shear = shear;
    st->nMolDeposited = deposited;
    st->errPrev = old->errPrev | old->errors | (s.displaced ? SGK_FLAG_DISPLACEMENT : 0);
}

// Maximum of n values v[0], v[stride], ... by one workgroup of 256 threads, returned to every thread.
template <class A>
__device__ __forceinline__ A block_max(const A *__restrict__ v, int n, int stride) {
    __shared__ A sh[4];
    A m = A(0);
    for (int k = threadIdx.x; k < n; k += 256) m = OpMax::f(m, v[(size_t)k * stride]);
    m = wave_reduce63<OpMax>(m);
    if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    return OpMax::f(OpMax::f(sh[0], sh[1]), OpMax::f(sh[2], sh[3]));
}

template <class A>
struct StepClose {
    const Partial<A> *part;  // force-pass partials, or chunk totals (direct = 0)
    PartMap map;
    int direct;              // 1: reduce the chunks here
    DevState *old, *st;      // the closed step's state, and the advanced one
    sgk_record *records;
    int recCap, on;
};

// The record of the closed step and the sums of the advanced state; called by one whole workgroup.
// The sums are those of k_reduce1 and k_finalize, bit for bit.
template <class A>
__device__ __forceinline__ void close_body(const DevParams &p, const StepClose<A> &c) {
    const Partial<A> P = sum_parts(c.part, c.map, !c.direct);
    if (threadIdx.x != 0) return;
    sgk_record rec;
    A cmVelX, vvSum;
    record_sums(p, P, rec, cmVelX, vvSum);
    rec.step = c.st->step;
    rec.rebuilt = c.old->nebrNow;
    rec.nebrNow = step_next(p, c.old, P.vmax).nebrNow;  // its own rule's: a batch may rebuild for another replica
    rec.errors = c.st->errPrev;
    rec.dispHi = c.st->dispHi;
    // Without an increment the rule only rounds the shear to A; it needs the sums, so k_bin_next leaves it
    // to this place.  With one, a launch that takes the sums (k_lf1_next) has applied it.
    if (p.deltaF == 0.f) c.st->shear = shear_next(p, rec.step, c.st->shear, cmVelX);
    rec.shear = c.st->shear;
    rec.shearCount = (double)c.old->shearCount;
    rec.nMolDeposited = c.st->nMolDeposited;
    const int slot = c.old->rec;
    if (slot < c.recCap) c.records[slot] = rec;
    c.st->vvSum = (double)vvSum;
    c.st->cmVelX = (double)cmVelX;
    c.st->comX = p.nMolMe ? (double)(P.com[0] / (A)p.nMolMe) : 0.0;
    c.old->errors = 0;  // taken over into errPrev; this state is the next advance's target
    c.old->shearCount = 0u;
}

}  // namespace sgk
