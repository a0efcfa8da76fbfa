// Stage kernels of the hx3d engine on Gauss-Lobatto nodes of one order (one explicit RK3 stage =
// k_grad, k_volume).
// Included by hx3d_engine.hip.  See that file for the device data layout.
#pragma once
#include <hip/hip_runtime.h>

#include "physics.hpp"

namespace hxk {

using hx::NV;
using hx::Phys;

struct Ops {  // NodalStorage for GL nodes (NodalStorageClass.f90:170-337), row-major (i,l)
    double D[64], hatD[64], sharpD[64], w[8];
};

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a contiguous range of
// elements so that face neighbours (gathered through L2) mostly share an XCD.  The grid is a
// multiple of 8, which makes this a bijection of [0, grid); logical blocks past the last
// element exit.
__host__ __device__ inline int xcd_block(int b, int grid)
{
    const int per = grid >> 3;
    return (b & 7) * per + (b >> 3);
}

// Keeps a value opaque to the compiler until this point: the consumers of a value loaded early
// (to overlap its latency with other work) cannot be hoisted above it, so the wait for the
// load stays here.  No instruction is emitted.
__device__ __forceinline__ void hold(double &x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#else
    (void)x;
#endif
}

// A kernel argument wanted in scalar registers at this point
template <class T>
__device__ __forceinline__ void wanted(T x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : : "s"(x));
#else
    (void)x;
#endif
}

// Element i of an array through its (wave-uniform) base and a 32-bit offset: the access takes
// the base from scalar registers and one 32-bit vector offset, with no 64-bit address
// arithmetic per access.  Every array plane the kernels index holds fewer than 2^29 elements
// (checked at engine creation), so the byte offset fits 32 bits.
// The base is made opaque in scalar registers (global address space kept), so that the
// compiler does not fold the plane offset into a per-lane 64-bit address.
#if defined(__HIP_DEVICE_COMPILE__)
#define HX_GLOBAL __attribute__((address_space(1)))
#else
#define HX_GLOBAL
#endif
template <class T>
__device__ __forceinline__ HX_GLOBAL T *sbase(T *x)
{
    auto g = (HX_GLOBAL T *)x;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(g));
#endif
    return g;
}
template <class T>
__device__ __forceinline__ T ldg(const T *x, unsigned i)
{
    return *(const HX_GLOBAL T *)((const HX_GLOBAL char *)sbase(x) + i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ void stg(T *x, unsigned i, T v)
{
    *(HX_GLOBAL T *)((HX_GLOBAL char *)sbase(x) + i * (unsigned)sizeof(T)) = v;
}

// Instructions are not moved across this point (no instruction is emitted).
__device__ __forceinline__ void sched_fence()
{
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// Entry t of an (N+1) x (N+1) operator (row stride 8 in Ops); threads t >= (N+1)^2 get 0.
// Loaded before the node data and stored to LDS after it has been issued, so the wait for it
// does not hold back the other loads.
template <int n1>
__device__ __forceinline__ double operator_entry(const double *src, int t)
{
    const int x = t < n1 * n1 ? t : 0;   // an unconditional load (see k_volume)
    return src[(x / n1) * 8 + (x % n1)];
}

__device__ __forceinline__ void block_min_pair(double a, double b, double *part, int t, int slot);
__device__ __forceinline__ void block_min_slot(double a, double b, unsigned long long *slots, int t, int cs, int lb);

// Several independent cases of one order in one engine (batching): each case has its own
// physics constants, dt, time, divergence flag and active mask; element blocks never straddle
// cases, so a block's case and constants are uniform.  All pointers null: one case.
struct CaseConst {
    double gammaM2, mu, mu_to_kappa, les_c;   // the constants that differ between cases
};
struct Multi {
    const int4 *blocks;     // per logical block: first element, element count, case, first block of its case
    const CaseConst *cc;    // [cases]
    const int *active;      // [cases]: 0 = finished, its blocks do no work (both copies of its state agree)
    int cases;
};

__device__ __forceinline__ void case_physics(Phys &ph, const CaseConst &c)
{
    ph.gammaM2 = c.gammaM2;
    ph.mu = c.mu;
    ph.mu_to_kappa = c.mu_to_kappa;
    ph.les_c = c.les_c;
}

// The elements of logical block lb: first element e0, count cnt (0: nothing to do), case cs,
// and whether the block is its case's first.  One case: EPB elements per block.
template <int EPB>
__device__ __forceinline__ void block_elements(const Multi &mc, int lb, int K, int &e0, int &cnt, int &cs, bool &first,
                                               Phys &ph)
{
    if (mc.blocks) {
        const int4 b = mc.blocks[lb];
        const bool on = mc.active[b.z] != 0;
        e0 = b.x;
        cs = b.z;
        cnt = on ? b.y : 0;
        first = b.w != 0;
        case_physics(ph, mc.cc[cs]);
    } else {
        e0 = lb * EPB;
        cnt = e0 < K ? (K - e0 < EPB ? K - e0 : EPB) : 0;
        cs = 0;
        first = lb == 0;
    }
}

// MaxTimeStep of the state a stage starts from, accumulated by the stage's gradient kernel.
// Mixed orders (part; null: not this stage): block minima of the convective and viscous limits to
// part[2*block + 0/1], reduced by the face kernel that follows (DtReduce).  One order (slots; null: not
// this stage): each block's minima by atomics into one of the case's DT_FAN slots, from which every block
// of the volume kernel that follows takes the minimum.  The minimum of doubles does not depend on the order; limits of either sign (those
// of a negative CFL number are negative) take their places like the numbers (slot_min), and NaN is
// passed over as fmin passes it over.  DT_FAN slots on lines of their own: one slot alone
// serialises (16k atomics on one address cost 150 us), 32 leave at most a few hundred per line at 24^3
// elements.
struct DtLimits {
    double *part;
    double cfl, dcfl, dcsi;
    unsigned long long *slots;
};
constexpr int DT_FAN = 32, DT_LINE = 16;   // slots per case; slot stride in 8-byte words (128 B)

// *slot, the bits of a double, to the smaller of it and x: positive numbers order as their bits do as signed
// whole numbers, below which every negative one lies; of two negative numbers the one with the larger bits,
// read as unsigned, is the smaller.  (Slots of keys that order like the numbers need no case here, but are
// turned back in every volume kernel: 16^3 Gauss elements of order 4 55.0 -> 55.9 us.)
__device__ __forceinline__ void slot_min(unsigned long long *slot, double x)
{
    const long long b = __double_as_longlong(fmin(x, INFINITY));   // NaN: +inf
    if (b < 0) atomicMax(slot, (unsigned long long)b);
    else atomicMin(reinterpret_cast<long long *>(slot), b);
}

// Averaging selectors of the templated split-form kernel (RiemannSolvers_NS.f90:229-285)
enum { AVG_STANDARD = 0, AVG_DUCROS = 1, AVG_KG = 2, AVG_PIROZZOLI = 3, AVG_MORINISHI = 4, FORM_STANDARD = -1 };

// Element face node x = (6e + slot) N1^2 + a + N1 b (a, b the slot's face coordinates); the
// face quantities the element kernels read are stored in this order, so an element reads its
// own contiguous range without an index lookup.
template <int N>
__device__ __forceinline__ unsigned efx(int e, int slot, int a, int b)
{
    return ((unsigned)e * 6 + slot) * ((N + 1) * (N + 1)) + a + (N + 1) * b;
}

// ------------------------------------------------------------------------------------
// k_grad: per element, local gradient (HexElement_ComputeLocalGradient,
// HexElementClass.f90:427-531) + BR1 lifting (EllipticBR1.f90:168-397), then the viscous flux
// tensor at every node (nine values, against twelve of the gradients it is formed from; the volume
// kernel's faces and nodes read it, and neither forms a viscosity), or with LES what it is formed
// from (viscous_values).
//   nbr[x]         2 * (neighbour's node) + (1 if this element is the face's right side)
//   mt             metric terms; face frames: normal (c = 0..2) and surface Jacobian |Ja| (c = 3)
//   visc[c*S+g]    out: the viscous flux tensor or the LES values
// ------------------------------------------------------------------------------------
// Registers: at most 128, which the attribute holds it to (114 to 124 are taken: the state is read again
// after the gradient, LES is a template flag, and order 7 takes its directions one at a time), since a
// block of six or eight waves finds room beside another only at four waves per SIMD: 9^3 elements of order 6 24.0 -> 19.9 us, of order 7 31.6 -> 25.7 (with
// LES).  Below that it makes no difference: at 16^3 elements of order 4 the kernel moves 135 MB in 25.7 us, 24^3
// of order 5 with LES 795 MB in 194 us, 0.76 and 0.82 of the copy rate (6.9 TB/s from the caches, 5 from memory).

// Metric terms of a case of one order: Ja^d_c in planes Ja[c*S + i], J[i], and the face frames
// face[c*FS + i].  Where they are the same bits at every node of each element (each face), as on boxes of
// straight elements, they are stored and read once per element (per face): i is the element (the
// element face) then, else the node.  The wave's loads fall on one line each and the planes
// stay in the caches: 80 bytes less of 208 per node for the gradient kernel, 80 of 312 and 32..80 of
// 280 per face node for the volume kernel.  9^3 elements of order 6: k_grad 26.0 -> 24.2 us, k_volume
// 35.5 -> 32.5; 64 cases of 4^3, order 3: 16.2 -> 14.7 and 25.4 -> 23.0; 20^3, orders 2..7: km_grad 133 ->
// 121, km_volume 123 -> 109.  By node where they vary (curved elements) there is no other way.
struct Metric {
    const double *Ja, *J, *face;
    long S, FS;
    int per_elem, per_face;
    __device__ __forceinline__ unsigned node(int e, unsigned g) const { return per_elem ? (unsigned)e : g; }
    template <int NF2>
    __device__ __forceinline__ unsigned face_node(unsigned x) const { return per_face ? x / NF2 : x; }
};

// The gradient at node (i, j, k) of the element whose state is sQ[v*ne + m] (LDS), in the
// reference's order: with u_d = sum_l D(own, l) q(l) along reference direction d,
// gr[c][v] = (sum_d u_d Ja^d_c) / J + gr[c][v] / J, the lifting sums given in gr.  One variable at a
// time, its results pinned (hold), so that the sums of a variable, not of all five, hold registers
// (k_volume at N = 4: 255 registers with all in flight).
template <int n1>
__device__ __forceinline__ void element_gradient(const double *sQ, const double *sD, int i, int j, int k,
                                                 const double *ja, double iJ, double (*gr)[NV])
{
    constexpr int nf = n1 * n1, ne = nf * n1;
    const double *lx = sQ + n1 * (j + n1 * k), *ly = sQ + i + nf * k, *lz = sQ + i + n1 * j;
    if constexpr (n1 < 8) {
        double dx[n1], dy[n1], dz[n1];
#pragma unroll
        for (int l = 0; l < n1; ++l) { dx[l] = sD[i * n1 + l]; dy[l] = sD[j * n1 + l]; dz[l] = sD[k * n1 + l]; }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double u0 = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
            for (int l = 0; l < n1; ++l) {
                u0 = u0 + lx[v * ne + l] * dx[l];
                u1 = u1 + ly[v * ne + n1 * l] * dy[l];
                u2 = u2 + lz[v * ne + nf * l] * dz[l];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                gr[c][v] = (u0 * ja[c] + u1 * ja[3 + c] + u2 * ja[6 + c]) * iJ + gr[c][v] * iJ;
                hold(gr[c][v]);
            }
            sched_fence();
        }
    } else {
        // order 7: a direction at a time, so that one row of the operator holds registers, not three
        double u[3][NV];
        auto along = [&](double *ud, const double *line, const double *row, int step) {
            double w[n1];
#pragma unroll
            for (int l = 0; l < n1; ++l) w[l] = row[l];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                ud[v] = 0.0;
#pragma unroll
                for (int l = 0; l < n1; ++l) ud[v] = ud[v] + line[v * ne + step * l] * w[l];
                hold(ud[v]);
            }
            sched_fence();
        };
        along(u[0], lx, sD + i * n1, 1);
        along(u[1], ly, sD + j * n1, n1);
        along(u[2], lz, sD + k * n1, nf);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int v = 0; v < NV; ++v)
                gr[c][v] = (u[0][v] * ja[c] + u[1][v] * ja[3 + c] + u[2][v] * ja[6 + c]) * iJ + gr[c][v] * iJ;
    }
}

// BR1 lifting of one face (BR1_ComputeElementInterfaceAverage, EllipticBR1.f90:571-627, and
// BR1_GradientFaceLoop, :531-569): unStar = 1/2 (U_R - U_L) |Ja| n with the face frame of the left
// element, the same value for both sides; the GL surface integral weights it by b = 1/w_0.  qn: the
// neighbour's state; jac: |Ja|, negated on the face's right side (so that 1/2 (qn - q) jac is the
// jump's product on both sides, bit for bit).
__device__ __forceinline__ void lift_face(const double *q, const double *qn, const double *n, double jac, double b0,
                                          double (*gr)[NV])
{
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double uS = 0.5 * (qn[v] - q[v]) * jac;
#pragma unroll
        for (int c = 0; c < 3; ++c) gr[c][v] = gr[c][v] + (uS * n[c]) * b0;
    }
}

// What the gradient kernel leaves per node: the viscous flux tensor (NVF values); with LES, whose
// eddy viscosity takes the element's filter width at the nodes and the face's on the faces, what
// the tensor is formed from: the stress without its viscosity (6), grad T (3), mu, and the
// filter-width-free factor X of the eddy viscosity.
constexpr int NVF = 9, NVL = 11;
constexpr int viscous_values(bool les) { return les ? NVL : NVF; }

// The tensor of a node's LES values with filter width d (mu, kappa of SD.f90:403-436 and :1345-1398)
__device__ __forceinline__ void les_tensor(const Phys &ph, const double *q, double ir, const double *x, double d,
                                           double *f)
{
    const double mt = hx::les_mu(ph, d, q[0], x[10]);
    const double mu = x[9] + mt, kappa = x[9] * ph.mu_to_kappa + mt * ph.mu_to_kappa;
    hx::viscous_tensor(mu, kappa, q[1] * ir, q[2] * ir, q[3] * ir, x, x + 6, f);
}

template <int N, int EPB, bool LES>
__global__ void __launch_bounds__(((EPB * (N + 1) * (N + 1) * (N + 1) + 63) / 64) * 64)
__attribute__((amdgpu_waves_per_eu(4)))
k_grad(const double *__restrict__ Q, Metric mt, const int *__restrict__ nbr,
       double *__restrict__ visc, double *__restrict__ curl_out, int K, long S, Ops ops, Phys ph, DtLimits dtl, Multi mc)
{
    constexpr int n1 = N + 1, nf = n1 * n1, ne = nf * n1;
    __shared__ double sQ[EPB][NV][ne];
    __shared__ double sD[n1 * n1];
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int t = threadIdx.x;
    int e0, cnt, cs;
    bool first;
    block_elements<EPB>(mc, lb, K, e0, cnt, cs, first, ph);
    if (cnt == 0) return;   // uniform: a padding block or a finished case
    const int el = t / ne, n = t - el * ne;
    const int e = e0 + el;
    const bool active = el < cnt;
    const int i = n % n1, j = (n / n1) % n1, k = n / nf;
    // Every load is unconditional (padding threads read a clamped element and discard it; see
    // k_volume).  The node's (at most three) faces: x-face slot 5 / 3, y-face 0 / 1, z-face
    // 2 / 4; faces the node is not on get zero traces and zero geometry, so their lifting term
    // is an exact zero and the accumulation below is branch-free.
    const int ec = active ? e : e0 + cnt - 1;
    const unsigned gc = (unsigned)ec * ne + n, g = (unsigned)e * ne + n;
    const bool onx = i == 0 || i == N, ony = j == 0 || j == N, onz = k == 0 || k == N;
    const int sx = i == 0 ? 5 : 3, sy = j == 0 ? 0 : 1, sz = k == 0 ? 2 : 4;
    const unsigned fx = efx<N>(ec, sx, j, k), fy = efx<N>(ec, sy, i, k), fz = efx<N>(ec, sz, i, j);
    const double dop = operator_entry<n1>(ops.D, t);
    const int cx = ldg(nbr, fx), cy = ldg(nbr, fy), cz = ldg(nbr, fz);
    double q[NV], ja[9], gx[4], gy[4], gz[4];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = ldg(Q + v * S, gc);
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = ldg(mt.Ja + c * mt.S, mt.node(ec, gc));
    const double jg = ldg(mt.J, mt.node(ec, gc));
    const double iJ = 1.0 / jg;   // the same bits as a stored 1/J
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const double a = ldg(mt.face + c * mt.FS, mt.face_node<nf>(fx)), b = ldg(mt.face + c * mt.FS, mt.face_node<nf>(fy)),
                     d = ldg(mt.face + c * mt.FS, mt.face_node<nf>(fz));
        gx[c] = onx ? a : 0.0;
        gy[c] = ony ? b : 0.0;
        gz[c] = onz ? d : 0.0;
    }
    // neighbour traces, issued before the barrier so that they arrive during the derivative
    double qx[NV], qy[NV], qz[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const double a = ldg(Q + v * S, (unsigned)cx >> 1), b = ldg(Q + v * S, (unsigned)cy >> 1),
                     d = ldg(Q + v * S, (unsigned)cz >> 1);
        qx[v] = onx ? a : 0.0;
        qy[v] = ony ? b : 0.0;
        qz[v] = onz ? d : 0.0;
    }
    if (t < n1 * n1) sD[t] = dop;
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sQ[el][v][n] = q[v];
    }
    __syncthreads();
    double tc = INFINITY, tv = INFINITY;   // MaxTimeStep limits of this node (stage 1)
    if (active) {
        double gr[3][NV];
        // Faces in slot order 5, 3, 0, 1, 2, 4 (ELEFT/ERIGHT, EFRONT/EBACK, EBOTTOM/ETOP)
        const double b0 = 1.0 / ops.w[0];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = 0; v < NV; ++v) gr[d][v] = 0.0;
        lift_face(q, qx, gx, cx & 1 ? -gx[3] : gx[3], b0, gr);
        lift_face(q, qy, gy, cy & 1 ? -gy[3] : gy[3], b0, gr);
        lift_face(q, qz, gz, cz & 1 ? -gz[3] : gz[3], b0, gr);
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = 0; v < NV; ++v) hold(gr[d][v]);
        sched_fence();
        element_gradient<n1>(&sQ[el][0][0], sD, i, j, k, ja, iJ, gr);
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = *(const volatile double *)&sQ[el][v][n];   // again: not held through the gradient
        double vg[12], sh[6], mu, kappa, X = 0.0;
        if (LES) {
            X = hx::les_factor(ph, q, gr[0], gr[1], gr[2]);
            hold(X);
            sched_fence();
        }
        hx::viscous_state(ph, q, gr[0], gr[1], gr[2], vg);
        if (curl_out) {   // |curl u|^2 of the enstrophy monitor
            const double a = vg[5] - vg[7], b = vg[6] - vg[2], c = vg[1] - vg[3];
            stg(curl_out, g, a * a + b * b + c * c);
        }
        hx::laminar_mu_kappa(ph, q, mu, kappa);
        hx::stress_shape(vg, sh);
        if (LES) {
#pragma unroll
            for (int c = 0; c < 6; ++c) stg(visc + c * S, g, sh[c]);
#pragma unroll
            for (int c = 0; c < 3; ++c) stg(visc + (6 + c) * S, g, vg[9 + c]);
            stg(visc + 9 * S, g, mu);
            stg(visc + 10 * S, g, X);
        } else {
            double f[NVF];
            const double ir = 1.0 / q[0];
            hx::viscous_tensor(mu, kappa, q[1] * ir, q[2] * ir, q[3] * ir, sh, vg + 9, f);
#pragma unroll
            for (int c = 0; c < NVF; ++c) stg(visc + c * S, g, f[c]);
        }
        if (dtl.slots) hx::dt_limits(ph, q, ja, jg, dtl.dcsi, dtl.dcsi, dtl.dcsi, dtl.cfl, dtl.dcfl, tc, tv);
    }
    if (dtl.slots) block_min_slot(tc, tv, dtl.slots, t, cs, lb);
}

// dtred: (partials, count, slot) of the step's dt limits, reduced by block 0 of the mixed-order face
// kernels
__device__ __forceinline__ void reduce_dt_partials(const double *part, int n, unsigned long long *bits, int t);
struct DtReduce {
    const double *part;
    int n;
    unsigned long long *bits;
};

// ------------------------------------------------------------------------------------
// k_volume: per element, the face fluxes of its six faces (computeElementInterfaceFlux,
// SD.f90:1710-1799), the volume integral (standard or split form), the surface integral, 1/J and
// the Williamson RK3 register update.
// ------------------------------------------------------------------------------------
struct DtArgs {
    const unsigned long long *in;   // [2]: convective, viscous limit bit patterns of this step's dt
    double *time;                   // t += dt by one thread (or null)
    int *nan;                       // set to 1 when an updated state value is NaN (or null)
    DtLimits lim;                   // consumed by the stage's gradient kernel
    DtReduce red;                   // consumed by the stage's face kernel (mixed orders)
    // One order: the first stage takes dt from the limits' slots (not from
    // `in`) and leaves it in `in`'s place, fin, for the later stages; the second stage empties the
    // slots for the next step (each null in the other stages)
    const unsigned long long *slots;
    unsigned long long *fin, *empty;
};

__device__ __forceinline__ double bits_to_double(unsigned long long b) { return __longlong_as_double((long long)b); }

// Block minimum of (a, b) written to part[2*blockIdx.x + 0/1]; every thread of the block calls
// it (inactive threads with +inf).  The minimum of doubles is exact and independent of order,
// so the two-level reduction (here, then k_dt_reduce) gives the same bits as a serial one,
// without contended atomics.
__device__ __forceinline__ void block_min_pair(double a, double b, double *part, int t, int slot)
{
    __shared__ double sm[2][16];
    for (int o = 32; o > 0; o >>= 1) {
        a = fmin(a, __shfl_xor(a, o, 64));
        b = fmin(b, __shfl_xor(b, o, 64));
    }
    if ((t & 63) == 0) { sm[0][t >> 6] = a; sm[1][t >> 6] = b; }
    __syncthreads();
    if (t == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int w = 1; w < nw; ++w) { a = fmin(a, sm[0][w]); b = fmin(b, sm[1][w]); }
        part[2 * slot] = a;
        part[2 * slot + 1] = b;
    }
}

// Block minimum of (a, b) by atomicMin into slot lb mod DT_FAN of case cs (see DtLimits)
__device__ __forceinline__ void block_min_slot(double a, double b, unsigned long long *slots, int t, int cs, int lb)
{
    __shared__ double sm[2][16];
    for (int o = 32; o > 0; o >>= 1) {
        a = fmin(a, __shfl_xor(a, o, 64));
        b = fmin(b, __shfl_xor(b, o, 64));
    }
    if ((t & 63) == 0) { sm[0][t >> 6] = a; sm[1][t >> 6] = b; }
    __syncthreads();
    if (t == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int w = 1; w < nw; ++w) { a = fmin(a, sm[0][w]); b = fmin(b, sm[1][w]); }
        unsigned long long *s = slots + (long)(cs * DT_FAN + lb % DT_FAN) * DT_LINE;
        slot_min(s, a);
        slot_min(s + 1, b);
    }
}

// The minima of n (convective, viscous) pairs of part as the bit patterns of a dt slot; every
// thread of the calling block takes part.
__device__ __forceinline__ void reduce_dt_partials(const double *part, int n, unsigned long long *bits, int t)
{
    __shared__ double sm[2][16];
    double a = INFINITY, b = INFINITY;
    for (int x = t; x < n; x += blockDim.x) {
        a = fmin(a, part[2 * x]);
        b = fmin(b, part[2 * x + 1]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        a = fmin(a, __shfl_xor(a, o, 64));
        b = fmin(b, __shfl_xor(b, o, 64));
    }
    if ((t & 63) == 0) { sm[0][t >> 6] = a; sm[1][t >> 6] = b; }
    __syncthreads();
    if (t == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int w = 1; w < nw; ++w) { a = fmin(a, sm[0][w]); b = fmin(b, sm[1][w]); }
        bits[0] = (unsigned long long)__double_as_longlong(a);
        bits[1] = (unsigned long long)__double_as_longlong(b);
    }
}

// This step's dt limits in a block of a volume kernel, by its first wave: load_dt asks for the
// case's slots (or the reduced pair), reduce_dt takes their minimum to sDt (visible after the next
// barrier); the case's first block leaves the reduced pair for the later stages, or empties the
// slots (see DtArgs).
__device__ __forceinline__ void load_dt(const DtArgs &dta, int cs, int t, double &a, double &b)
{
    const unsigned long long *s = dta.slots ? dta.slots + (long)(cs * DT_FAN + t % DT_FAN) * DT_LINE : dta.in + 2 * cs;
    a = bits_to_double(s[0]);
    b = bits_to_double(s[1]);
}
__device__ __forceinline__ void reduce_dt(const DtArgs &dta, int cs, bool first, int t, double a, double b, double &sDt)
{
    for (int o = 32; o > 0; o >>= 1) {
        a = fmin(a, __shfl_xor(a, o, 64));
        b = fmin(b, __shfl_xor(b, o, 64));
    }
    if (t == 0) {
        sDt = fmin(a, b);
        if (first && dta.slots) {
            dta.fin[2 * cs] = (unsigned long long)__double_as_longlong(a);
            dta.fin[2 * cs + 1] = (unsigned long long)__double_as_longlong(b);
        }
    }
    if (first && dta.empty && t < DT_FAN) {
        unsigned long long *sl = dta.empty + (long)(cs * DT_FAN + t) * DT_LINE;
        sl[0] = sl[1] = (unsigned long long)__double_as_longlong(INFINITY);
    }
}

// Offset of the node pair (lo, hi), lo < hi, of an (N+1)-node line in the pair table (pairs
// lo-major).
__host__ __device__ constexpr int pair_slot(int n1, int lo, int hi)
{
    return lo * n1 - (lo * (lo + 1)) / 2 + (hi - lo - 1);
}

// One thread per node, EPB elements per block.  First the face fluxes, one thread per element face
// node, through LDS.  Then the contravariant fluxes of all three
// directions (split form: the viscous ones, whose mass entry is zero; standard form: inviscid
// minus viscous) go to LDS once.  Per direction each node accumulates, in l order,
// qd = (qd + sharpD F#) + hatD Fv (DGIntegrals.f90:92-129) or qd = qd + hatD F (:56-87).
// Split form, per direction: the node data and the metric rows (times metric_scale) go to LDS;
// each unordered node pair of a line is evaluated once, lower node index first as the reference
// evaluates both (i, l) and (l, i) (HyperbolicSplitForm.f90:64-116), by node lo of the pair
// (lo, lo + s mod N+1), s = 1..(N+1)/2 (for even N+1, s = (N+1)/2 only for lo < (N+1)/2); the
// pair fluxes then replace the node data in LDS and every node reads its N off-diagonal
// entries from there (at N = 5 each node evaluates its own row of N pair fluxes instead: ROW).
// The diagonal entry is the node's inviscid contravariant flux.
// Minimum waves per SIMD asked of the register allocator: 3 for the standard form, and for
// Kennedy-Gruber and Pirozzoli up to N = 5 (no spills in 168 VGPRs up to N = 4; at N = 5 the
// few spilled registers cost less than a third wave gains), else no constraint.  From N = 6 on a block
// has six or eight waves, and a second one finds room on a CU only at four waves per SIMD: standard form,
// 9^3 elements of order 6 with LES 32.4 us at 130 registers, 25.9 at 128; order 7 43.7 and 34.6;
// Kennedy-Gruber at order 6 54.5 and 53.2 (27 to 43 spills); the other averagings spill more and lost 3 to
// 5%; at order 7 the split form's LDS admits one block.  The compiler holds to four only where it does not
// see the block's LDS, so the pool is dynamic.
#ifndef HX3D_VOL_WAVES
#define HX3D_VOL_WAVES 3
#endif
// Split form at N = 5 without the pair table (each node evaluates its own row); built with
// HX3D_ROW5=0, the pair table as at the other orders (for comparison).
#ifndef HX3D_ROW5
#define HX3D_ROW5 1
#endif
constexpr int volume_waves(int n, int form)
{
    if (n >= 6 && form == -1) return 4;
    if (n == 6 && (form == 2 || form == 3)) return 4;
    return form == -1 ? 3 : (form == 2 || form == 3) && n <= 5 ? HX3D_VOL_WAVES : 1;
}

// Element face node x of an element (x = slot nf + a + (N+1) b) as the element's node index
template <int N>
__device__ __forceinline__ int face_element_node(int x)
{
    constexpr int n1 = N + 1, nf = n1 * n1;
    const int s = x / nf, r = x - s * nf, a = r % n1, b = r / n1;
    if (s == 3 || s == 5) return n1 * a + nf * b + (s == 3 ? N : 0);   // x faces: (a, b) = (j, k)
    if (s < 2) return a + nf * b + (s == 1 ? n1 * N : 0);              // y faces: (i, k)
    return r + (s == 4 ? nf * N : 0);                                  // z faces: (i, j)
}

// Doubles of k_volume's LDS pool per block: first the elements' state [NV][ne] and viscous
// values [9 or 11][ne] and the face fluxes [NV] per element face node; then the contravariant fluxes and
// the direction loop's space.
constexpr int vol_max(int a, int b) { return a > b ? a : b; }
// VIS: the viscous model (INVISCID, LAMINAR, EDDY).  INVISCID: no viscous values, and no viscous fluxes in the
// split form's direction loop (a quarter of its LDS reads at N = 5: each added an exact zero); 11^3
// elements of order 5, Ducros, 44.3 -> 40.5 us; 16^3 of order 4, Pirozzoli, 53.6 -> 51.4 us.
enum { INVISCID = 0, LAMINAR = 1, EDDY = 2 };
template <int N, int EPB, int FORM, int VIS>
struct VolumeLds {
    static constexpr int n1 = N + 1, nf = n1 * n1, ne = nf * n1, NI = 6 * nf;
    static constexpr bool SPLIT = FORM >= 0;
    static constexpr int ND = hx::node_data_size(SPLIT ? FORM : 0);
    static constexpr int NF = SPLIT ? 4 : 5;
    // split form: node data [ND][ne] and metric rows [3][ne], then the pair fluxes
    // [pair][NV][line] of the current direction, in one space per element; at N = 5 each node
    // evaluates its own row of pair fluxes (ROW), without the pair table
    static constexpr bool ROW = SPLIT && N == 5 && HX3D_ROW5;
    static constexpr int RN = (ND + 3) * ne, RP = ROW ? 0 : n1 * (n1 - 1) / 2 * NV * nf;
    static constexpr int RSZ = SPLIT ? vol_max(RN, RP) : 0;
    static constexpr int FSZ = SPLIT && VIS == INVISCID ? 0 : 3 * NF * ne;
    static constexpr int NVT = VIS == INVISCID ? 0 : viscous_values(VIS == EDDY);
    static constexpr int FACES = EPB * NI;
    static constexpr int SIZE = vol_max(EPB * (NV + NVT) * ne + NV * FACES, EPB * (FSZ + RSZ));
};

// What bounds it: bytes first.  Per node 312 B (Q, Ja, J, G, viscous tensor in; G, Q out; 328 B with
// LES), per element face node 172 B with Lax-Friedrichs, 148 B with Roe (the neighbour's state and
// viscous values, 16 B more with LES, the face frame, the neighbour index).  The face fluxes are formed by both elements
// of a face, from the same values in the same order, hence with the same bits: that costs 1.2
// instead of 0.6 Riemann fluxes per node at N = 4, and saves the launch, the 80 B per face node
// of stored fluxes each way and the second read of both traces.  Measured per stage (k_grad and
// k_volume; before, with a face kernel between them and the gradients stored): 16^3 x N=4 Pirozzoli
// 81 us (91), 24^3 x N=5 Kennedy-Gruber + WALE 587 (701), 4^3 x N=3 13 (18), 9^3 x N=6 44 (62).
// At 16^3 x N=4 the kernel moves 241 MB in 55 us.  Without the direction loop it took 40 us where it took 59
// with it, the rate of a large copy; the loop's LDS traffic (97 accesses per node and direction) adds the
// rest.  Forming the gradient again here instead of reading the viscous values measured 76 us.
// New state to Qn, not in place: the neighbours of later blocks still read Q.
// LXF: the engine's Riemann solver is Lax-Friedrichs, the one that reads the tangents (Roe does not).
template <int N, int EPB, int FORM, bool LXF, int VIS>
__global__ void __launch_bounds__(((EPB * (N + 1) * (N + 1) * (N + 1) + 63) / 64) * 64)
__attribute__((amdgpu_waves_per_eu(volume_waves(N, FORM))))
k_volume(const double *__restrict__ Q, double *__restrict__ Qn, const double *__restrict__ visc,
         const double *__restrict__ edelta, const double *__restrict__ efdelta, const int *__restrict__ nbx,
         Metric mt, int t2x, double *__restrict__ G, double *__restrict__ qdot_out, double a_k, double c_k, int update,
         DtArgs dta, int K, long S, Ops ops, Phys ph, Multi mc)
{
    using L = VolumeLds<N, EPB, FORM, VIS>;
    constexpr bool LES = VIS == EDDY, EULER = VIS == INVISCID;
    constexpr int NVT = viscous_values(LES);
    constexpr int n1 = L::n1, nf = L::nf, ne = L::ne, NI = L::NI, ND = L::ND, NF = L::NF, FACES = L::FACES;
    constexpr bool SPLIT = L::SPLIT, ROW = L::ROW;
    constexpr int AVG = SPLIT ? FORM : 0, V0 = SPLIT ? 1 : 0, NP = n1 / 2;
    constexpr bool SYM = hx::two_point_symmetric(AVG);
    constexpr int TPB = ((EPB * ne + 63) / 64) * 64, P = (FACES + TPB - 1) / TPB;
    HIP_DYNAMIC_SHARED(double, pool)   // [L::SIZE]
    __shared__ double sHat[n1 * n1], sSharp[SPLIT ? n1 * n1 : 1], sDt;
    __shared__ int sSlot[SPLIT ? n1 * n1 : 1];   // pair table offset of (own, l); 0 on the diagonal
    double *const sQ = pool;                       // [EPB][NV][ne]
    double *const sT = sQ + EPB * NV * ne;         // [EPB][NVT][ne]
    double *const sFb = sT + EPB * L::NVT * ne;       // [NV][FACES]
    const int lb = xcd_block(blockIdx.x, gridDim.x);
    const int t = threadIdx.x;
    int e0, cnt, cs;
    bool first;
    if (N <= 3) {
        // one wave per block: the first loads' addresses ahead of the early return, with the scalar loads
        // before it (15^3 x N=2: 13.03 -> 12.60 us).  Larger blocks hide that wait behind one another, and
        // the registers spill (9^3 x N=6 with LES: 10% slower).
        wanted(Q);
        wanted(nbx);
        wanted(visc);
        wanted(mt.Ja);
        wanted(mt.face);
        wanted(K);
        wanted(S);
        wanted(mt.S);
        wanted(mt.FS);
    }
    if (SPLIT) ph.averaging = FORM;   // the Lax-Friedrichs flux averages as the volume fluxes do
    block_elements<EPB>(mc, lb, K, e0, cnt, cs, first, ph);
    const int el = t / ne, n = t - el * ne;
    const int e = e0 + el;
    if (cnt == 0) return;   // uniform: a padding block or a finished case
    const bool active = el < cnt;
    const int i = n % n1, j = (n / n1) % n1, k = n / nf;
    const bool onx = i == 0 || i == N, ony = j == 0 || j == N, onz = k == 0 || k == N;
    // ---- Loads are unconditional (padding threads read a clamped element and discard it): a
    // load inside a branch makes the compiler wait for the whole memory queue at the first use
    // of any earlier load.
    const int ec = active ? e : e0 + cnt - 1;
    const unsigned gc = (unsigned)ec * ne + n, gw = (unsigned)e * ne + n;
    int code[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int it = t + p * TPB;
        code[p] = ldg(nbx, (unsigned)e0 * NI + (it < cnt * NI ? it : 0));
    }
    const double hop = operator_entry<n1>(ops.hatD, t),
                 sop = operator_entry<n1>(ops.sharpD, t);
    double q[NV], ja[9], vt[NVT];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = ldg(Q + v * S, gc);
    if (!EULER) {   // uniform
#pragma unroll
        for (int c = 0; c < NVT; ++c) vt[c] = ldg(visc + c * S, gc);
    }
    double dtl0, dtl1;   // this step's dt limits (first wave)
    if (update && t < 64) load_dt(dta, cs, t, dtl0, dtl1);
    if (t < n1 * n1) {
        sHat[t] = hop;
        if (SPLIT) {
            sSharp[t] = sop;
            const int a = t / n1, b = t - a * n1;
            sSlot[t] = a == b ? 0 : pair_slot(n1, a < b ? a : b, a < b ? b : a) * NV * nf;
        }
    }
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = ldg(mt.Ja + c * mt.S, mt.node(ec, gc));
    const double jg = ldg(mt.J, mt.node(ec, gc)), dl = LES ? ldg(edelta, (unsigned)ec) : 0.0;
    const double b0 = 1.0 / ops.w[0];
    // What round p's face flux reads from memory; round 0's is asked for before the barrier, to
    // arrive with the element's own data.
    double qR[NV], nrm[3], jac, t1[3], fn[NVT], fd = 0.0;
    auto load_face = [&](int p) {
        const int it = t + p * TPB;
        const unsigned x = (unsigned)e0 * NI + (it < cnt * NI ? it : 0), xn = (unsigned)code[p] >> 1;
        const unsigned en = xn / NI, gn = en * ne + face_element_node<N>(xn - en * NI);
#pragma unroll
        for (int v = 0; v < NV; ++v) qR[v] = ldg(Q + v * S, gn);
#pragma unroll
        for (int c = 0; c < 3; ++c) nrm[c] = ldg(mt.face + c * mt.FS, mt.face_node<nf>(x));
        jac = ldg(mt.face + 3 * mt.FS, mt.face_node<nf>(x));
        if (!EULER) {
#pragma unroll
            for (int c = 0; c < NVT; ++c) fn[c] = ldg(visc + c * S, gn);
        }
        if (LES) fd = ldg(efdelta, x / nf);
        if (LXF) {
#pragma unroll
            for (int c = 0; c < 3; ++c) t1[c] = ldg(mt.face + (4 + c) * mt.FS, mt.face_node<nf>(x));
        }
    };
    load_face(0);
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sQ[(el * NV + v) * ne + n] = q[v];
        if (!EULER) {
#pragma unroll
            for (int c = 0; c < NVT; ++c) sT[(el * NVT + c) * ne + n] = vt[c];
        }
    }
    __syncthreads();
    const int fx = el * NI + (i == 0 ? 5 : 3) * nf + j + n1 * k, fy = el * NI + (j == 0 ? 0 : 1) * nf + i + n1 * k,
              fz = el * NI + (k == 0 ? 2 : 4) * nf + i + n1 * j;
    // ---- the face fluxes, one thread per element face node, P rounds
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int it = t + p * TPB;
        if (p) load_face(p);
        if (it < cnt * NI) {
            const bool right = code[p] & 1;
            const int eo = it / NI, no = face_element_node<N>(it - eo * NI);
            double qL[NV], vn[NV];
            const double io = 1.0 / sQ[eo * NV * ne + no], in = 1.0 / qR[0];
            vn[0] = 0.0;
            if (!EULER) {
                // BR1_RiemannSolver (EllipticBR1.f90:816-868): the average of both sides' tensors,
                // summed in either order with the same bits, and its product with the normal
                double f[NVF];
                if (LES) {
                    double qo[NV], vo[NVT], fo[NVF];
#pragma unroll
                    for (int v = 0; v < NV; ++v) qo[v] = sQ[(eo * NV + v) * ne + no];
#pragma unroll
                    for (int c = 0; c < NVT; ++c) vo[c] = sT[(eo * NVT + c) * ne + no];
                    les_tensor(ph, qo, io, vo, fd, fo);
                    les_tensor(ph, qR, in, fn, fd, f);
#pragma unroll
                    for (int c = 0; c < NVF; ++c) f[c] = 0.5 * (f[c] + fo[c]);
                } else {
#pragma unroll
                    for (int c = 0; c < NVF; ++c) f[c] = 0.5 * (fn[c] + sT[(eo * NVT + c) * ne + no]);
                }
#pragma unroll
                for (int v = 1; v < NV; ++v) {
                    vn[v] = f[hx::viscous_entry(v, 0)] * nrm[0] + f[hx::viscous_entry(v, 1)] * nrm[1] +
                            f[hx::viscous_entry(v, 2)] * nrm[2];
                    hold(vn[v]);
                }
            } else {
#pragma unroll
                for (int v = 1; v < NV; ++v) vn[v] = 0.0;
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double o = sQ[(eo * NV + v) * ne + no], a = qR[v];
                qL[v] = right ? a : o;
                qR[v] = right ? o : a;
            }
            double inv[NV];
            if (LXF) {
                // t2x: the stored second tangent is n x t1 (vCross, MappedGeometry.f90:745, :807-817)
                // bit for bit at every face node (checked on the host), so it is formed here
                double t2[3];
                if (!t2x) {
                    const unsigned x = mt.face_node<nf>((unsigned)e0 * NI + it);
#pragma unroll
                    for (int c = 0; c < 3; ++c) t2[c] = ldg(mt.face + (7 + c) * mt.FS, x);
                } else {
                    t2[0] = nrm[1] * t1[2] - t1[1] * nrm[2];
                    t2[1] = nrm[2] * t1[0] - t1[2] * nrm[0];
                    t2[2] = nrm[0] * t1[1] - t1[0] * nrm[1];
                }
                hx::lxf_flux(ph, qL, qR, right ? in : io, right ? io : in, nrm, t1, t2, inv);
            } else {
                hx::roe_flux(ph, qL, qR, right ? in : io, right ? io : in, nrm, inv);
            }
            // the right side negated (TimeDerivative_FacesContribution, SD.f90:1686-1701)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double fb = ((inv[v] - vn[v]) * jac) * b0;
                sFb[v * FACES + it] = right ? -fb : fb;
            }
        }
    }
    if (update && t < 64) reduce_dt(dta, cs, first, t, dtl0, dtl1, sDt);
    __syncthreads();
    // The RK register.  The first RK stage (a_k = 0) does not read it: the reference's 0 G + QDot is
    // QDot up to the sign of an exact zero, which no state value sees (Q + c dt (+-0) = Q); every
    // later stage does.  Asked for here in the standard form, whose contractions are short, and at
    // the last direction in the split form, where it would hold registers through two of them.
    double gk[NV];
    auto load_register = [&]() {
        if (a_k != 0.0) {
#pragma unroll
            for (int v = 0; v < NV; ++v) gk[v] = ldg(G + v * S, gc);
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v) gk[v] = 0.0;
        }
    };
    if (!SPLIT) load_register();
    double own[ND] = {};   // this node's two-point data (split form)
    double xs[NV];         // the surface integral at this node
    double Fvc[3][NV];     // contravariant viscous fluxes; standard form: inviscid minus viscous
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = sQ[(el * NV + v) * ne + n];   // held no longer than needed
        // Surface integral (SD.f90:1686-1701) of the node's faces in slot order; faces the node is
        // not on add an exact zero
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double a = sFb[v * FACES + fx], b = sFb[v * FACES + fy], c = sFb[v * FACES + fz];
            xs[v] = ((0.0 + (onx ? a : 0.0)) + (ony ? b : 0.0)) + (onz ? c : 0.0);
            hold(xs[v]);   // summed here, not at its use: one register pair instead of three
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = 0; v < NV; ++v) Fvc[d][v] = 0.0;
        if (!EULER) {
            // BR1_ComputeInnerFluxes (EllipticBR1.f90:740-814)
            double f[NVF];
#pragma unroll
            for (int c = 0; c < NVT; ++c) vt[c] = sT[(el * NVT + c) * ne + n];   // held no longer than needed
            if (LES) {
                les_tensor(ph, q, 1.0 / q[0], vt, dl, f);
            } else {
#pragma unroll
                for (int c = 0; c < NVF; ++c) f[c] = vt[c];
            }
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int v = 1; v < NV; ++v)
                    Fvc[d][v] = f[hx::viscous_entry(v, 0)] * ja[3 * d] + f[hx::viscous_entry(v, 1)] * ja[3 * d + 1] +
                                f[hx::viscous_entry(v, 2)] * ja[3 * d + 2];
        }
        if (SPLIT) {
            hx::node_data<AVG>(ph, q, own);
        } else {
            double Fi[3][NV];
            hx::euler_contravariant(ph, q, ja, Fi);
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int v = 0; v < NV; ++v) Fvc[d][v] = Fi[d][v] - Fvc[d][v];
        }
    }
    __syncthreads();   // the state and the face values are read: the pool takes the fluxes
    double *const sF = pool + el * (L::FSZ + L::RSZ);   // [3][NF][ne]
    double *const sR = sF + L::FSZ;                     // [RSZ]
    constexpr bool VF = !SPLIT || !EULER;   // the direction loop reads sF
    if (VF && active) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = V0; v < NV; ++v) sF[(d * NF + v - V0) * ne + n] = Fvc[d][v];
    }
    double qd[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) qd[v] = 0.0;
    double pu, pv, pw, pp;   // the diagonal's primitives, formed once for the three directions
    hx::euler_primitives(ph, q, pu, pv, pw, pp);
    // xi, then eta, then zeta.  Every thread reaches every barrier; inactive threads (block
    // padding) only skip the work between them.
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int own_i = d == 0 ? i : (d == 1 ? j : k);
        const int stride = d == 0 ? 1 : (d == 1 ? n1 : nf);
        const int base = n - own_i * stride;
        const int line = d == 0 ? j + n1 * k : (d == 1 ? i + n1 * k : i + n1 * j);
        double jh[3];   // this node's metric row times metric_scale
#pragma unroll
        for (int c = 0; c < 3; ++c) jh[c] = hx::metric_scale(AVG) * ja[3 * d + c];
        if (SPLIT) {
            if (d) __syncthreads();     // the previous direction's pair fluxes are read
            if (active) {
#pragma unroll
                for (int c = 0; c < ND; ++c) sR[c * ne + n] = own[c];
#pragma unroll
                for (int c = 0; c < 3; ++c) sR[(ND + c) * ne + n] = jh[c];
            }
        }
        if (SPLIT || d == 0) __syncthreads();
        if (SPLIT && d == 2) load_register();
        if (!SPLIT) {
            if (active) {
#pragma unroll
                for (int l = 0; l < n1; ++l) {
                    const double hh = sHat[own_i * n1 + l];
                    const int m = base + l * stride;
#pragma unroll
                    for (int v = 0; v < NV; ++v) qd[v] = qd[v] + hh * sF[(d * NF + v) * ne + m];
                }
            }
            continue;
        }
        if (ROW) {
            // each node evaluates its whole row of two-point fluxes from the line's node data (a
            // pair twice, once by each of its nodes, with the same arithmetic) and accumulates it
            // in l order; the diagonal is the node's inviscid contravariant flux
            if (active) {
                double fi[NV];
                hx::euler_contravariant_row(q, pu, pv, pw, pp, &ja[3 * d], fi);
#pragma unroll 1
                for (int l = 0; l < n1; ++l) {
                    const double sh = sSharp[own_i * n1 + l], hh = sHat[own_i * n1 + l];
                    const int m = base + l * stride;
                    double b[ND], jb[3], tp[NV];
#pragma unroll
                    for (int c = 0; c < ND; ++c) b[c] = sR[c * ne + m];
#pragma unroll
                    for (int c = 0; c < 3; ++c) jb[c] = sR[(ND + c) * ne + m];
                    if (SYM) {
                        hx::two_point<AVG>(own, jh, b, jb, tp);
                    } else {
                        const bool lo = own_i < l;
                        double x1[ND], x2[ND], j1[3], j2[3];
#pragma unroll
                        for (int c = 0; c < ND; ++c) { x1[c] = lo ? own[c] : b[c]; x2[c] = lo ? b[c] : own[c]; }
#pragma unroll
                        for (int c = 0; c < 3; ++c) { j1[c] = lo ? jh[c] : jb[c]; j2[c] = lo ? jb[c] : jh[c]; }
                        hx::two_point<AVG>(x1, j1, x2, j2, tp);
                    }
                    qd[0] = qd[0] + sh * (l == own_i ? fi[0] : tp[0]);
#pragma unroll
                    for (int v = 1; v < NV; ++v) {
                        qd[v] = qd[v] + sh * (l == own_i ? fi[v] : tp[v]);
                        if (VF) qd[v] = qd[v] + hh * sF[(d * NF + v - V0) * ne + m];
                    }
                }
            }
            continue;
        }
        // this node's pairs (own, own + s mod N+1)
        double pf[NP][NV];
        if (active) {
#pragma unroll
            for (int s = 1; s <= NP; ++s) {
                const int l = own_i + s < n1 ? own_i + s : own_i + s - n1;
                const int m = base + l * stride;
                double b[ND], jb[3];
#pragma unroll
                for (int c = 0; c < ND; ++c) b[c] = sR[c * ne + m];
#pragma unroll
                for (int c = 0; c < 3; ++c) jb[c] = sR[(ND + c) * ne + m];
                if (SYM) {
                    hx::two_point<AVG>(own, jh, b, jb, pf[s - 1]);
                } else {
                    const bool lo = own_i < l;
                    double x1[ND], x2[ND], j1[3], j2[3];
#pragma unroll
                    for (int c = 0; c < ND; ++c) { x1[c] = lo ? own[c] : b[c]; x2[c] = lo ? b[c] : own[c]; }
#pragma unroll
                    for (int c = 0; c < 3; ++c) { j1[c] = lo ? jh[c] : jb[c]; j2[c] = lo ? jb[c] : jh[c]; }
                    hx::two_point<AVG>(x1, j1, x2, j2, pf[s - 1]);
                }
            }
        }
        __syncthreads();   // node data read: the space takes the pair fluxes
        if (active) {
#pragma unroll
            for (int s = 1; s <= NP; ++s) {
                if (2 * s == n1 && own_i >= s) continue;
                const int l = own_i + s < n1 ? own_i + s : own_i + s - n1;
                const int po = sSlot[own_i * n1 + l] + line;
#pragma unroll
                for (int v = 0; v < NV; ++v) sR[po + v * nf] = pf[s - 1][v];
            }
        }
        __syncthreads();
        if (active) {
            double fi[NV];
            hx::euler_contravariant_row(q, pu, pv, pw, pp, &ja[3 * d], fi);
            // unrolled by two at N = 4 (0.8% faster there, same registers); other orders
            // would spill
            constexpr int VU = N == 4 ? 2 : 1;
#pragma unroll VU
            for (int l = 0; l < n1; ++l) {
                const double sh = sSharp[own_i * n1 + l], hh = sHat[own_i * n1 + l];
                const int m = base + l * stride;
                const int po = sSlot[own_i * n1 + l] + line;
                qd[0] = qd[0] + sh * (l == own_i ? fi[0] : sR[po]);
#pragma unroll
                for (int v = 1; v < NV; ++v) {
                    qd[v] = qd[v] + sh * (l == own_i ? fi[v] : sR[po + v * nf]);
                    if (VF) qd[v] = qd[v] + hh * sF[(d * NF + v - V0) * ne + m];
                }
            }
        }
    }
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if (SPLIT) qd[v] = -qd[v];
            qd[v] = qd[v] - xs[v];
        }
        // QDot / J (SD.f90:490) as a product with 1/J: the rounding difference is one ulp of the
        // final derivative, taken after the cancellation of volume and surface terms
        const double ijg = 1.0 / jg;
#pragma unroll
        for (int v = 0; v < NV; ++v) qd[v] = qd[v] * ijg;
        if (qdot_out) {
#pragma unroll
            for (int v = 0; v < NV; ++v) stg(qdot_out + v * S, gw, qd[v]);
        }
        if (update) {
            const double dt = sDt;
            if (dta.time && first && t == 0) dta.time[cs] += dt;
            const double cdt = c_k * dt;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                hold(gk[v]);
                const double gv = a_k * gk[v] + qd[v];
                stg(G + v * S, gw, gv);
                q[v] = q[v] + cdt * gv;
                stg(Qn + v * S, gw, q[v]);
            }
            // checkForNan (ExplicitMethods.f90:1856-1905) of the updated state: a sticky flag,
            // written only where a NaN appears
            if (dta.nan && (isnan(q[0]) || isnan(q[1]) || isnan(q[2]) || isnan(q[3]) || isnan(q[4])))
                atomicOr(dta.nan + cs, 1);
        }
    }
}

}  // namespace hxk
