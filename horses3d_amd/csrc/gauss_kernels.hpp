// Uniform-order kernels of the hx3d engine on Gauss nodes (standard form), one element per block.
// On Gauss nodes no node lies on a face: a face value is the Lagrange basis at the face's end of
// the normal direction applied along it (HexElement_ProlongSolutionToFaces /
// _ProlongGradientsToFaces, HexElementClass.f90:233-372), and the BR1 lift and the surface
// integral reach every node with b = v(+-1)/w (VectorWeakIntegrals_StdFace /
// ScalarWeakIntegrals_StdFace, DGIntegrals.f90:214-443).  Here the traces are formed where the
// element's values are in LDS and stored in element-face order:
//   kg_prolong  Q traces of the resident state (after the state is set from outside);
//   kg_grad     local gradient, BR1 lift from the six faces' unStar, the viscous flux tensors at the
//               nodes and, from the traces of the state and the gradient, at the face nodes;
//   kg_volume   the face fluxes of the element's faces (Riemann + BR1, from both sides' traces),
//               volume integral, surface integral of the six faces with b, 1/J, the RK update,
//               and the updated state's Q traces (a second copy: neighbours still read the first).
// Included by hx3d_engine.hip after stage_kernels.hpp.
#pragma once
#include <hip/hip_runtime.h>

#include "physics.hpp"
#include "stage_kernels.hpp"

namespace hxg {

using hx::NV;
using hx::Phys;
using hxk::ldg;
using hxk::stg;

// v(-1), v(+1) and b = v / w of the Gauss nodes of order N (NodalStorageClass.f90:257-273)
struct GaussOps {
    double vL[8], vR[8], bL[8], bR[8];
};

template <int N>
constexpr int gauss_tpb() { return (((N + 1) * (N + 1) * (N + 1) + 63) / 64) * 64; }

// node index of the element node at position l along slot s's axis and face coordinates (a, b)
// (slots 0..5 = EFRONT, EBACK, EBOTTOM, ERIGHT, ETOP, ELEFT; their axes y, y, z, x, z, x)
template <int N>
__device__ __forceinline__ int line_node(int s, int a, int b, int l)
{
    constexpr int n1 = N + 1;
    int i, j, k;
    if (s == 0 || s == 1) { i = a; j = l; k = b; }
    else if (s == 2 || s == 4) { i = a; j = b; k = l; }
    else { i = l; j = a; k = b; }
    return i + n1 * (j + n1 * k);
}

// The traces of NVAL node arrays sV[c*ne + n] (LDS) of element e on its six faces:
// out[c*ES + (6e + s) nf + a + (N+1) b] = acc, acc = acc + value(l) v(l) for l = 0..N along the
// slot's axis (the reference's order).  One work item is a line of nodes along an axis at face
// coordinates (a, b) and five of the values: it gives both ends of the line, the slot pair
// 5 / 3 (xi), 0 / 1 (eta) or 2 / 4 (zeta) with v(-1) and v(+1), from one read of each node
// value.  Consecutive threads take consecutive lines of one axis (consecutive face nodes).
template <int N, int NVAL>
__device__ __forceinline__ void write_traces(const double *sV, double *out, long ES, int e, const GaussOps &go,
                                             int t, int nthr)
{
    static_assert(NVAL % NV == 0, "values in groups of five");
    constexpr int n1 = N + 1, nf = n1 * n1, ne = nf * n1, NL = 3 * nf, NG = NVAL / NV;
    for (int it = t; it < NL * NG; it += nthr) {
        const int grp = it / NL, L = it - grp * NL;
        const int ax = L / nf, r = L - ax * nf;
        const int sm = ax == 0 ? 5 : (ax == 1 ? 0 : 2), sp = ax == 0 ? 3 : (ax == 1 ? 1 : 4);
        const int n0 = line_node<N>(sm, r % n1, r / n1, 0), st = ax == 0 ? 1 : (ax == 1 ? n1 : nf);
        const long om = (long)(6 * e + sm) * nf + r, op = (long)(6 * e + sp) * nf + r;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = grp * NV + v;
            double am = 0.0, ap = 0.0;
#pragma unroll
            for (int l = 0; l < n1; ++l) {
                const double x = sV[c * ne + n0 + l * st];
                am = am + x * go.vL[l];
                ap = ap + x * go.vR[l];
            }
            out[(long)c * ES + om] = am;   // c varies across the wave: 64-bit addresses
            out[(long)c * ES + op] = ap;
        }
    }
}

// The viscous flux tensors (viscous_tensor's nine values) at element e's face nodes, from the
// gradient sV[c*ne + n] (15 values, LDS) carried to both ends of each line of nodes, the state's
// traces there and the viscosities of compute_viscosity_at_faces (SD.f90:1345-1398).  One thread per
// line, at most 3 (N+1)^2 <= threads, so that each node value is read from LDS once for both ends.
// qm, qp: the state's traces at the line's ends om, op; dm, dp: the filter widths of its two faces.
template <int N>
__device__ __forceinline__ void write_face_tensors(const double *sV, double *out, long ES, int n0, int st, unsigned om,
                                                   unsigned op, const double *qm, const double *qp, double dm, double dp,
                                                   const GaussOps &go, const Phys &ph)
{
    constexpr int n1 = N + 1, ne = n1 * n1 * n1;
    double gm[3 * NV], gp[3 * NV];
#pragma unroll
    for (int c = 0; c < 3 * NV; ++c) {
        double am = 0.0, ap = 0.0;
#pragma unroll
        for (int l = 0; l < n1; ++l) {
            const double x = sV[c * ne + n0 + l * st];
            am = am + x * go.vL[l];
            ap = ap + x * go.vR[l];
        }
        gm[c] = am;
        gp[c] = ap;
        hxk::hold(gm[c]);
        hxk::hold(gp[c]);
    }
    auto tensor = [&](const double *q, const double *g, double d, unsigned x) {
        double vg[12], sh[6], f[9], mu, kappa;
        hx::viscous_state(ph, q, g, g + NV, g + 2 * NV, vg);
        hx::laminar_mu_kappa(ph, q, mu, kappa);
        if (ph.les) {
            const double mt = hx::les_mu(ph, d, q[0], hx::les_factor(ph, q, g, g + NV, g + 2 * NV));
            mu = mu + mt;
            kappa = kappa + mt * ph.mu_to_kappa;
        }
        const double ir = 1.0 / q[0];
        hx::stress_shape(vg, sh);
        hx::viscous_tensor(mu, kappa, q[1] * ir, q[2] * ir, q[3] * ir, sh, vg + 9, f);
#pragma unroll
        for (int c = 0; c < 9; ++c) stg(out + c * ES, x, f[c]);
    };
    tensor(qm, gm, dm, om);
    tensor(qp, gp, dp, op);
}

// ------------------------------------------------------------------------------------
// kg_prolong: Q traces of the resident state (HexMesh_ProlongSolutionToFaces)
// ------------------------------------------------------------------------------------
template <int N>
__global__ void __launch_bounds__(gauss_tpb<N>())
kg_prolong(const double *__restrict__ Q, double *__restrict__ Qtr, int K, long S, long ES, GaussOps go)
{
    constexpr int ne = (N + 1) * (N + 1) * (N + 1);
    __shared__ double sQ[NV * ne];
    const int e = hxk::xcd_block(blockIdx.x, gridDim.x), t = threadIdx.x;
    if (e >= K) return;   // uniform per block
    if (t < ne) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sQ[v * ne + t] = ldg(Q + v * S, (unsigned)e * ne + t);
    }
    __syncthreads();
    write_traces<N, NV>(sQ, Qtr, ES, e, go, t, blockDim.x);
}

// ------------------------------------------------------------------------------------
// kg_grad: local gradient (HexElement_ComputeLocalGradient), BR1 lift (BR1_ComputeElementInterface-
// Average, EllipticBR1.f90:571-627, and BR1_GradientFaceLoop, :531-569): unStar =
// 1/2 (Q_R - Q_L) |Ja| n at every face node of the element, from its own and its neighbour's
// trace, then every node takes the six faces' unStar with its weights b; the viscous flux tensor
// at the node, and those at the face nodes from the gradient's traces
// (HexElement_ProlongGradientsToFaces).
//   nbx[x]  2 * (the neighbour's element face node matching x) + (1 if this element is the face's
//           right side)
//   egeo    normal and |Ja| of the face at x (the left element's face frame on both sides)
// ------------------------------------------------------------------------------------
template <int N>
__global__ void __launch_bounds__(gauss_tpb<N>()) __attribute__((amdgpu_waves_per_eu(3)))
kg_grad(const double *__restrict__ Q, const double *__restrict__ Qtr, const double *__restrict__ Ja,
        const double *__restrict__ Jac, const int *__restrict__ nbx, const double *__restrict__ egeo,
        const double *__restrict__ edelta, const double *__restrict__ efdelta, double *__restrict__ visc,
        double *__restrict__ fvis, double *__restrict__ curl_out, int K, long S, long ES, hxk::Ops ops, GaussOps go,
        Phys ph, hxk::DtLimits dtl)
{
    constexpr int n1 = N + 1, nf = n1 * n1, ne = nf * n1;
    // one LDS space, in turn: the element's state [5][ne]; per face node the jump's 5 values and the
    // normal, whose 15 products every node forms (8 LDS reads a face instead of 15); the gradient
    // [15][ne]
    constexpr int NW = 8 * 6 * nf > 3 * NV * ne ? 8 * 6 * nf : 3 * NV * ne;
    __shared__ double sW[NW];
    __shared__ double sD[n1 * n1];
    double *sQ = sW;
    const int lb = hxk::xcd_block(blockIdx.x, gridDim.x), t = threadIdx.x;
    const int e = lb;
    if (e >= K) return;   // a padding block
    const bool active = t < ne;
    const int n = active ? t : 0;
    const int i = n % n1, j = (n / n1) % n1, k = n / nf;
    const unsigned g = (unsigned)e * ne + n;
    const double dop = hxk::operator_entry<n1>(ops.D, t);
    double q[NV], ja[9];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = ldg(Q + v * S, g);
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = ldg(Ja + c * S, g);
    const double jg = ldg(Jac, g), dl = ldg(edelta, (unsigned)e);
    const double iJ = 1.0 / jg;
    if (t < n1 * n1) sD[t] = dop;
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sQ[v * ne + n] = q[v];
    }
    // unStar at the element's face nodes, the same value on both sides of a face.  The P passes
    // over the face nodes are unrolled so that every pass's index and geometry loads, then its
    // trace loads, are issued before the first is used (here, to arrive during the gradient).
    constexpr int TPB = gauss_tpb<N>(), NFN = 6 * nf, P = (NFN + TPB - 1) / TPB;
    int c2[P];
    double fg[P][4], own[P][NV], nb[P][NV];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int f = t + p * TPB;
        const unsigned x = (unsigned)(6 * e) * nf + (f < NFN ? f : 0);
        c2[p] = ldg(nbx, x);
#pragma unroll
        for (int c = 0; c < 4; ++c) fg[p][c] = ldg(egeo + c * ES, x);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int f = t + p * TPB;
        const unsigned x = (unsigned)(6 * e) * nf + (f < NFN ? f : 0), xn = (unsigned)c2[p] >> 1;
#pragma unroll
        for (int v = 0; v < NV; ++v) { own[p][v] = ldg(Qtr + v * ES, x); nb[p][v] = ldg(Qtr + v * ES, xn); }
    }
    __syncthreads();
    double tc = INFINITY, tv = INFINITY;
    double gr[3][NV];
    if (active) {
        double uxi[NV], ueta[NV], uzeta[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) { uxi[v] = 0.0; ueta[v] = 0.0; uzeta[v] = 0.0; }
#pragma unroll
        for (int l = 0; l < n1; ++l) {
            const double di = sD[i * n1 + l];
#pragma unroll
            for (int v = 0; v < NV; ++v) uxi[v] = uxi[v] + sQ[v * ne + l + n1 * (j + n1 * k)] * di;
        }
#pragma unroll
        for (int l = 0; l < n1; ++l) {
            const double dj = sD[j * n1 + l];
#pragma unroll
            for (int v = 0; v < NV; ++v) ueta[v] = ueta[v] + sQ[v * ne + i + n1 * (l + n1 * k)] * dj;
        }
#pragma unroll
        for (int l = 0; l < n1; ++l) {
            const double dk = sD[k * n1 + l];
#pragma unroll
            for (int v = 0; v < NV; ++v) uzeta[v] = uzeta[v] + sQ[v * ne + i + n1 * (j + n1 * l)] * dk;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            gr[0][v] = (uxi[v] * ja[0] + ueta[v] * ja[3] + uzeta[v] * ja[6]) * iJ;
            gr[1][v] = (uxi[v] * ja[1] + ueta[v] * ja[4] + uzeta[v] * ja[7]) * iJ;
            gr[2][v] = (uxi[v] * ja[2] + ueta[v] * ja[5] + uzeta[v] * ja[8]) * iJ;
        }
    }
    __syncthreads();   // the state has been read: the space takes the faces' unStar
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int f = t + p * TPB;
        if (f < NFN) {
            const bool right = c2[p] & 1;
#pragma unroll
            for (int v = 0; v < NV; ++v)
                sW[v * NFN + f] = 0.5 * (right ? own[p][v] - nb[p][v] : nb[p][v] - own[p][v]) * fg[p][3];
#pragma unroll
            for (int d = 0; d < 3; ++d) sW[(NV + d) * NFN + f] = fg[p][d];
        }
    }
    __syncthreads();
    if (active) {
        // the six faces in the order L, R (xi), FR, BK (eta), BOT, T (zeta): slots 5, 3, 0, 1, 2, 4
        const int fl = 5 * nf + j + n1 * k, fr = 3 * nf + j + n1 * k;
        const int ff = 0 * nf + i + n1 * k, fb = 1 * nf + i + n1 * k;
        const int fo = 2 * nf + i + n1 * j, ft = 4 * nf + i + n1 * j;
        const double bl = go.bL[i], br = go.bR[i], bf = go.bL[j], bb = go.bR[j], bo = go.bL[k], bt = go.bR[k];
        double fi[3][NV];
        auto lift = [&](int f, double w, bool start) {
            double nn[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) nn[d] = sW[(NV + d) * NFN + f];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double uS = sW[v * NFN + f];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double x = (uS * nn[d]) * w;
                    fi[d][v] = start ? x : fi[d][v] + x;
                    hxk::hold(fi[d][v]);
                }
            }
        };
        lift(fl, bl, true);
        lift(fr, br, false);
        lift(ff, bf, false);
        lift(fb, bb, false);
        lift(fo, bo, false);
        lift(ft, bt, false);
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                gr[d][v] = gr[d][v] + fi[d][v] * iJ;
                hxk::hold(gr[d][v]);
            }
        hxk::sched_fence();
        double vg[12], sh[6], f[9], mu, kappa;
        hx::viscous_state(ph, q, gr[0], gr[1], gr[2], vg);
        if (curl_out) {   // |curl u|^2 of the enstrophy monitor
            const double a = vg[5] - vg[7], b = vg[6] - vg[2], c = vg[1] - vg[3];
            stg(curl_out, g, a * a + b * b + c * c);
        }
        // mu, kappa of SD.f90:403-436
        hx::laminar_mu_kappa(ph, q, mu, kappa);
        if (ph.les) {
            const double mt = hx::les_mu(ph, dl, q[0], hx::les_factor(ph, q, gr[0], gr[1], gr[2]));
            mu = mu + mt;
            kappa = kappa + mt * ph.mu_to_kappa;
        }
        const double ir = 1.0 / q[0];
        hx::stress_shape(vg, sh);
        hx::viscous_tensor(mu, kappa, q[1] * ir, q[2] * ir, q[3] * ir, sh, vg + 9, f);
#pragma unroll
        for (int c = 0; c < 9; ++c) stg(visc + c * S, g, f[c]);
        hxk::sched_fence();
        if (dtl.slots) hx::dt_limits(ph, q, ja, jg, dtl.dcsi, dtl.dcsi, dtl.dcsi, dtl.cfl, dtl.dcfl, tc, tv);
    }
    // the line whose ends this thread takes (write_face_tensors), its state traces and filter widths
    const int L = t < 3 * nf ? t : 0, ax = L / nf, r = L - ax * nf;
    const int sm = ax == 0 ? 5 : (ax == 1 ? 0 : 2), sp = ax == 0 ? 3 : (ax == 1 ? 1 : 4);
    const unsigned om = (unsigned)(6 * e + sm) * nf + r, op = (unsigned)(6 * e + sp) * nf + r;
    double qm[NV], qp[NV], dm = 0.0, dp = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v) { qm[v] = ldg(Qtr + v * ES, om); qp[v] = ldg(Qtr + v * ES, op); }
    if (ph.les) { dm = ldg(efdelta, (unsigned)(6 * e + sm)); dp = ldg(efdelta, (unsigned)(6 * e + sp)); }
    __syncthreads();   // the unStar has been read: the space takes the gradient
    if (active) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int v = 0; v < NV; ++v) sW[(d * NV + v) * ne + n] = gr[d][v];
    }
    __syncthreads();
    if (t < 3 * nf)
        write_face_tensors<N>(sW, fvis, ES, line_node<N>(sm, r % n1, r / n1, 0), ax == 0 ? 1 : (ax == 1 ? n1 : nf), om, op,
                              qm, qp, dm, dp, go, ph);
    if (dtl.slots) hxk::block_min_slot(tc, tv, dtl.slots, t, 0, lb);
}

// ------------------------------------------------------------------------------------
// kg_volume: the fluxes of the element's faces (computeElementInterfaceFlux, SD.f90:1710-1799, from
// both sides' traces and viscous flux tensors; formed by both elements of a face from the same
// values in the same order, hence with the same bits), the standard-form volume integral with hatD
// (TimeDerivative_VolumetricContribution), the surface integral of the six faces' fluxes with the
// node's weights b, 1/J, the Williamson RK3 update (TakeRK3Step) and, after an update, the new
// state's Q traces to Qtn.
// ------------------------------------------------------------------------------------
template <int N, bool LXF>
__global__ void __launch_bounds__(gauss_tpb<N>()) __attribute__((amdgpu_waves_per_eu(3)))
kg_volume(double *__restrict__ Q, const double *__restrict__ Qtr, double *__restrict__ Qtn,
          const double *__restrict__ visc, const double *__restrict__ fvis, const int *__restrict__ nbx,
          const double *__restrict__ egeo, int t2x, const double *__restrict__ Ja, const double *__restrict__ Jac,
          double *__restrict__ G, double *__restrict__ qdot_out, double a_k, double c_k, int update, hxk::DtArgs dta,
          int K, long S, long ES, hxk::Ops ops, GaussOps go, Phys ph)
{
    constexpr int n1 = N + 1, nf = n1 * n1, ne = nf * n1, NFN = 6 * nf;
    constexpr int TPB = gauss_tpb<N>(), P = (NFN + TPB - 1) / TPB;
    __shared__ double sF[3 * NV * ne];   // contravariant fluxes [d][v][ne]; then the new state [v][ne]
    __shared__ double sE[NV * NFN];      // the element's face fluxes [v][6 nf] (element-face order)
    __shared__ double sHat[n1 * n1], sDt;
    const int e = hxk::xcd_block(blockIdx.x, gridDim.x), t = threadIdx.x;
    if (e >= K) return;   // uniform per block
    const bool active = t < ne;
    const int n = active ? t : 0;
    const int i = n % n1, j = (n / n1) % n1, k = n / nf;
    const unsigned g = (unsigned)e * ne + n;
    int code[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int f = t + p * TPB;
        code[p] = ldg(nbx, (unsigned)e * NFN + (f < NFN ? f : 0));
    }
    const double hop = hxk::operator_entry<n1>(ops.hatD, t);
    double q[NV], ja[9], vf[9];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = ldg(Q + v * S, g);
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = ldg(Ja + c * S, g);
    if (!ph.euler) {
#pragma unroll
        for (int c = 0; c < 9; ++c) vf[c] = ldg(visc + c * S, g);
    } else {
#pragma unroll
        for (int c = 0; c < 9; ++c) vf[c] = 0.0;
    }
    const double jg = ldg(Jac, g);
    double dtl0, dtl1;   // this step's dt limits (first wave)
    if (update && t < 64) hxk::load_dt(dta, 0, t, dtl0, dtl1);
    // What round p's face flux reads; round 0's is asked for here, to arrive during the node fluxes
    double qo[NV], qn[NV], nrm[3], jac, t1[3], fo[9], fn[9];
    auto load_face = [&](int p) {
        const int f = t + p * TPB;
        const unsigned x = (unsigned)e * NFN + (f < NFN ? f : 0), xn = (unsigned)code[p] >> 1;
#pragma unroll
        for (int v = 0; v < NV; ++v) { qo[v] = ldg(Qtr + v * ES, x); qn[v] = ldg(Qtr + v * ES, xn); }
#pragma unroll
        for (int c = 0; c < 3; ++c) nrm[c] = ldg(egeo + c * ES, x);
        jac = ldg(egeo + 3 * ES, x);
        if (!ph.euler) {
#pragma unroll
            for (int c = 0; c < 9; ++c) { fo[c] = ldg(fvis + c * ES, x); fn[c] = ldg(fvis + c * ES, xn); }
        }
        if (LXF) {
#pragma unroll
            for (int c = 0; c < 3; ++c) t1[c] = ldg(egeo + (4 + c) * ES, x);
        }
    };
    load_face(0);
    if (active) {
        double Fi[3][NV];
        hx::euler_contravariant(ph, q, ja, Fi);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            sF[(d * NV) * ne + n] = Fi[d][0] - 0.0;
#pragma unroll
            for (int v = 1; v < NV; ++v) {   // BR1_ComputeInnerFluxes (EllipticBR1.f90:740-814)
                const double Fv = vf[hx::viscous_entry(v, 0)] * ja[3 * d] + vf[hx::viscous_entry(v, 1)] * ja[3 * d + 1] +
                                  vf[hx::viscous_entry(v, 2)] * ja[3 * d + 2];
                sF[(d * NV + v) * ne + n] = Fi[d][v] - Fv;
            }
        }
    }
    if (t < n1 * n1) sHat[t] = hop;
    hxk::sched_fence();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int f = t + p * TPB;
        if (p) load_face(p);
        if (f < NFN) {
            const bool right = code[p] & 1;
            double qL[NV], qR[NV], vn[NV], inv[NV];
            vn[0] = 0.0;
            if (!ph.euler) {
                // BR1_RiemannSolver (EllipticBR1.f90:816-868): the average of both sides' tensors,
                // summed in either order with the same bits, and its product with the normal
#pragma unroll
                for (int c = 0; c < 9; ++c) fn[c] = 0.5 * (fo[c] + fn[c]);
#pragma unroll
                for (int v = 1; v < NV; ++v) {
                    vn[v] = fn[hx::viscous_entry(v, 0)] * nrm[0] + fn[hx::viscous_entry(v, 1)] * nrm[1] +
                            fn[hx::viscous_entry(v, 2)] * nrm[2];
                    hxk::hold(vn[v]);
                }
            } else {
#pragma unroll
                for (int v = 1; v < NV; ++v) vn[v] = 0.0;
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) { qL[v] = right ? qn[v] : qo[v]; qR[v] = right ? qo[v] : qn[v]; }
            if (LXF) {
                double t2[3];
                if (!t2x) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) t2[c] = ldg(egeo + (7 + c) * ES, (unsigned)e * NFN + f);
                } else {   // n x t1, see hxk::k_volume
                    t2[0] = nrm[1] * t1[2] - t1[1] * nrm[2];
                    t2[1] = nrm[2] * t1[0] - t1[2] * nrm[0];
                    t2[2] = nrm[0] * t1[1] - t1[0] * nrm[1];
                }
                hx::lxf_flux(ph, qL, qR, nrm, t1, t2, inv);
            } else {
                hx::roe_flux(ph, qL, qR, nrm, inv);
            }
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double fl = (inv[v] - vn[v]) * jac;
                sE[v * NFN + f] = right ? -fl : fl;
            }
        }
    }
    if (update && t < 64) hxk::reduce_dt(dta, 0, e == 0, t, dtl0, dtl1, sDt);
    double gk[NV];
    if (update && a_k != 0.0) {
#pragma unroll
        for (int v = 0; v < NV; ++v) gk[v] = ldg(G + v * S, g);
    } else {
#pragma unroll
        for (int v = 0; v < NV; ++v) gk[v] = 0.0;
    }
    __syncthreads();
    if (active) {
        // surface integral (ScalarWeakIntegrals_StdFace): L, R, FR, BK, BOT, T with the node's b
        double xs[NV];
        {
            const int xl = 5 * nf + j + n1 * k, xr = 3 * nf + j + n1 * k;
            const int xf = 0 * nf + i + n1 * k, xb = 1 * nf + i + n1 * k;
            const int xo = 2 * nf + i + n1 * j, xt = 4 * nf + i + n1 * j;
            const double bl = go.bL[i], br = go.bR[i], bf = go.bL[j], bb = go.bR[j], bo = go.bL[k], bt = go.bR[k];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double *fv = sE + v * NFN;
                double x = fv[xl] * bl;
                x = x + fv[xr] * br;
                x = x + fv[xf] * bf;
                x = x + fv[xb] * bb;
                x = x + fv[xo] * bo;
                x = x + fv[xt] * bt;
                xs[v] = x;
            }
        }
        double qd[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) qd[v] = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int own = d == 0 ? i : (d == 1 ? j : k);
            const int stride = d == 0 ? 1 : (d == 1 ? n1 : nf);
            const int base = n - own * stride;
#pragma unroll
            for (int l = 0; l < n1; ++l) {
                const double hh = sHat[own * n1 + l];
                const int m = base + l * stride;
#pragma unroll
                for (int v = 0; v < NV; ++v) qd[v] = qd[v] + hh * sF[(d * NV + v) * ne + m];
            }
        }
        const double ijg = 1.0 / jg;
#pragma unroll
        for (int v = 0; v < NV; ++v) qd[v] = (qd[v] - xs[v]) * ijg;
        if (qdot_out) {
#pragma unroll
            for (int v = 0; v < NV; ++v) stg(qdot_out + v * S, g, qd[v]);
        }
        if (update) {
            const double dt = sDt;
            if (dta.time && e == 0 && t == 0) dta.time[0] += dt;
            const double cdt = c_k * dt;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double gv = a_k * gk[v] + qd[v];
                stg(G + v * S, g, gv);
                q[v] = q[v] + cdt * gv;
                stg(Q + v * S, g, q[v]);
            }
            if (dta.nan && (isnan(q[0]) || isnan(q[1]) || isnan(q[2]) || isnan(q[3]) || isnan(q[4])))
                atomicOr(dta.nan, 1);
        }
    }
    if (update) {   // uniform: the new state's traces for the next stage
        __syncthreads();   // the fluxes have been read
        if (active) {
#pragma unroll
            for (int v = 0; v < NV; ++v) sF[v * ne + n] = q[v];
        }
        __syncthreads();
        write_traces<N, NV>(sF, Qtn, ES, e, go, t, blockDim.x);
    }
}

}  // namespace hxg
