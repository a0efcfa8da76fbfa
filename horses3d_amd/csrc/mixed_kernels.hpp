// Mixed-order stage kernels of the hx3d engine: elements with their own orders (Nx, Ny, Nz)
// and conforming faces between mismatched orders through the reference's mortar operators
// (Face_AdaptSolutionToFace / Face_AdaptGradientsToFace, FaceClass.f90:281-512, and
// Face_ProjectFluxToElements / Face_ProjectGradientFluxToElements, FaceClass.f90:597-700,
// 865-964).  Included by hx3d_engine.hip after stage_kernels.hpp.
//
// One stage = km_face_grad -> km_grad -> km_face -> km_volume:
//   km_face_grad  one wave per face (or two small faces of one shape, see face_lane): both Q
//                 traces to the face order, BR1 unStar there,
//                 projected back onto each side's element face (lift[15][ES]);
//   km_grad       element tiles: local gradient + lifting -> grad Q (15 values); in a step's
//                 first stage, the dt limits;
//   km_face       as km_face_grad: Q and grad Q traces to the face order, Riemann + BR1
//                 fluxes there, projected back (right side negated) and scaled by the
//                 receiving element's surface weight -> fe[5][ES];
//   km_volume     element tiles: volume integral, surface integral, 1/J and RK update.
// The element kernels are persistent: one launch per stage sweeps every element, each block
// taking tiles (elements packed into at most 512 nodes, one thread per node) in turn, each
// thread reading what it works on from the tiles' node map.
// The same kernels run Gauss-node cases (GAUSS template flag, one order or per-element
// orders): the traces are the Lagrange basis at the face's end applied along the normal
// direction, and the BR1 lift and the surface integral reach every node with b = v(+-1)/w.
#pragma once
#include <hip/hip_runtime.h>

#include "physics.hpp"
#include "stage_kernels.hpp"

namespace hxm {

using hx::NV;
using hx::Phys;
using hxk::DtArgs;

constexpr int MAXN1 = 8;   // orders 1..7

// Operators of every order N (row i, column j at [N][i*8 + j]) and the mortar matrices
// Tset(N -> M) ((M+1) x (N+1), row-major with row length N+1), InterpolationMatrices.f90:42-108.
struct OpsAll {
    double D[MAXN1][64], hatD[MAXN1][64], sharpD[MAXN1][64];
    double b0[MAXN1];     // 1/w_0 = 1/w_N, the GL surface weight
    double dcsi[MAXN1];   // 1/|x_1 - x_0|, MaxTimeStep (DGSEMClass.f90:948-959)
    double T[MAXN1][MAXN1][64];
    // the Lagrange basis at -1 and +1 and b = v / w (NodalStorageClass.f90:257-273): the face
    // values and surface weights of Gauss nodes, on which no node lies on a face
    double vL[MAXN1][8], vR[MAXN1][8], bL[MAXN1][8], bR[MAXN1][8];
};

// Face record (Face_LinkWithElements, FaceClass.f90:187-278), with every index the kernels form of a
// face laid out on the host as an affine map of the face coordinates (i, j), the right side's
// rotation (leftIndexes2Right, MeshTypes.f90:70-108) included.  The face kernels are bound by latency
// (one wave per face, three or four waves per SIMD): their traces start after two dependent loads
// (wave, record) instead of five through element, order and offset tables, the shape's loops count
// in scalar registers and the node arrays are addressed in 32 bits.  20^3 elements, orders 2..7:
// km_face_grad 104.7 -> 79.5 us, km_face 176.4 -> 129.7 us; 10^3 Gauss, orders 2..5: 20.1 -> 16.2 us and
// 39.9 -> 34.5 us.
struct __align__(16) FaceRec {
    int g0[2], gi[2], gj[2];   // side s's node at (i, j), at the face's end of the normal axis
    int x0[2], xi[2], xj[2];   // side s's element face node at (i, j)
    int gn[2];                 // node step along side s's normal axis, from the face inwards
    int foff;                  // first face node (face order) of this face
    int na;                    // order along the normal axis, side s in bits 8s..; bit 16 + s: the plus end
};
// What the faces of a wave share: the face orders Nf and each side's orders Ns in the face
// orientation (three bits each), from which the projection types follow.
struct Shape {
    int Nf0, Nf1, N0[2], N1[2];
};
__host__ __device__ inline int pack_shape(int Nf0, int Nf1, int L0, int L1, int R0, int R1)
{
    return Nf0 | Nf1 << 3 | L0 << 6 | L1 << 9 | R0 << 12 | R1 << 15;
}
__device__ __forceinline__ Shape unpack_shape(int c)
{
    return Shape{c & 7, (c >> 3) & 7, {(c >> 6) & 7, (c >> 12) & 7}, {(c >> 9) & 7, (c >> 15) & 7}};
}
// 0 no projection, 1 along the first face index, 2 along the second, 3 along both
__device__ __forceinline__ int projection(const Shape &r, int side)
{
    return (r.N0[side] != r.Nf0 ? 1 : 0) + (r.N1[side] != r.Nf1 ? 2 : 0);
}
// node (i, j) of a grid of rows of d nodes, 2 <= d <= 8, from q < 64: (q + 1/2)/d lies at least 1/16
// from a whole number, far more than the reciprocal's error
__device__ __forceinline__ void grid_ij(int q, int d, int &i, int &j)
{
    j = (int)(((float)q + 0.5f) * __builtin_amdgcn_rcpf((float)d));
    i = q - j * d;
}

// A tile of elements for the persistent element kernels (host side): up to TILE_MAXE elements
// whose nodes, one thread each, fill at most TILE threads; thread t works on node t - off[s] of
// elem[s], off[s] <= t < off[s + 1] (threads from off[count] on are idle).  Which elements share
// a tile (the packing) is chosen on the host (hx3d_autotune); every packing gives the same
// results.  The kernels read the tiles through their node map (NodeMap).
// Tiles of two sizes, each swept by a launch of its own: 256 threads (two independent blocks
// per CU, whose loads and barriers do not wait for each other) for elements of at most 256
// nodes, 512 threads for larger elements (up to 8 x 8 x 8 nodes).  The host picks the sizes.
constexpr int TILE = 512, TILE_SMALL = 256, TILE_MAXE = 30;
struct Tile {
    int count;
    int elem[TILE_MAXE];
    int off[TILE_MAXE + 1];
};

// What thread t of a tile works on, built on the host with the tiles (one entry per thread of
// every tile, at [tile * T + t] for tiles of T threads): node g of element e, and code = i | j << 3 | k << 6 |
// Nx << 9 | Ny << 12 | Nz << 15 | (first thread of the element in the tile) << 18 | active << 27.
// One load gives a thread everything the tile table, the orders and the node offsets would
// give through three dependent ones; the element kernels load the next tile's entry while
// they work on the current one.  Idle threads (active = 0) carry node 0 of the tile's last
// element, so that their unconditional loads stay in bounds.
struct __align__(16) NodeMap {
    int g, e, code;
    int ef0;   // the element's first element face node
};
template <int T>
__device__ __forceinline__ NodeMap load_map(const NodeMap *__restrict__ map, int tile, int t)
{
    return map[(long)tile * T + t];
}

// Element face node of the element's node (i, j, k) on the face of slot s: the element's six faces
// follow one another in slot order 0..5 = EFRONT, EBACK, EBOTTOM, ERIGHT, ETOP, ELEFT (axes y, y, z,
// x, z, x), each (first coordinate fastest) at the element's orders.
struct ElemFaces {
    int s[6];
};
__device__ __forceinline__ ElemFaces elem_faces(int ef0, int nx, int ny, int nz)
{
    const int xz = nx * nz, xy = nx * ny, yz = ny * nz;
    return ElemFaces{{ef0, ef0 + xz, ef0 + 2 * xz, ef0 + 2 * xz + xy, ef0 + 2 * xz + xy + yz, ef0 + 2 * xz + 2 * xy + yz}};
}

// Face_AdaptSolutionToFace (side trace -> face order Nf) and Face_ProjectFluxToElements (face ->
// the side's element face) at face node (i, j).  Projection type pt: 0 the orders agree (a
// copy), 1 Tset along the first face index, 2 along the second, 3 along both, accumulated as
// acc += T0[i][m] * T1[j][l] * value in the loop order l (outer), m (inner) of the reference.

// The face's mortar matrices in LDS.  Along each face index d at most one side interpolates
// (the face order is the larger of the two sides' orders, so the other side's order is the face
// order): m[d] = Tset(N_s -> n_d) (side to face) and m[2 + d] = Tset(n_d -> N_s) (face to side)
// of that side serve both sides, one entry per lane.  The interpolation loops then read them at
// LDS latency instead of through the cache from the operator table.  (Reading them from the
// operator table instead measured 19% slower in km_face.)
struct Mort {
    const double *a0, *a1, *p0, *p1;   // side to face along the two face indices, face to side
};
__device__ __forceinline__ Mort mort_lds(const double (*m)[64]) { return Mort{m[0], m[1], m[2], m[3]}; }

__device__ __forceinline__ void stage_mortar(const OpsAll &ops, const Shape &r, double (*m)[64], int lane)
{
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        const int n = d ? r.Nf1 : r.Nf0;
        const int a = d ? r.N1[0] : r.N0[0], b = d ? r.N1[1] : r.N0[1], Ns = a < n ? a : b;
        if (Ns < n) {
            m[d][lane] = ops.T[Ns][n][lane];
            m[2 + d][lane] = ops.T[n][Ns][lane];
        }
    }
}

// Face_AdaptSolutionToFace for K values at once (values k at tr[k*64 + q], the side's trace in
// the face orientation, q = m + (Ns0+1) l), with the matrices staged by stage_mortar: each
// source node's weight is formed once, and every value accumulates in the reference's order
// with the reference's products.
template <int K>
__device__ __forceinline__ void adapt_k(const Mort &m, const Shape &r, int side, const double *tr,
                                        int i, int j, double *out)
{
    const int N0 = r.N0[side], N1 = r.N1[side], n0 = r.Nf0;
    const int pt = projection(r, side);
    if (pt == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = tr[k * 64 + i + (n0 + 1) * j];
        return;
    }
    const double *T0 = m.a0, *T1 = m.a1;
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = 0.0;
    if (pt == 1) {
        for (int l = 0; l <= N0; ++l) {
            const double w = T0[i * (N0 + 1) + l];
            const int q = l + (N0 + 1) * j;
#pragma unroll
            for (int k = 0; k < K; ++k) out[k] += w * tr[k * 64 + q];
        }
    } else if (pt == 2) {
        for (int l = 0; l <= N1; ++l) {
            const double w = T1[j * (N1 + 1) + l];
            const int q = i + (N0 + 1) * l;
#pragma unroll
            for (int k = 0; k < K; ++k) out[k] += w * tr[k * 64 + q];
        }
    } else {
        for (int l = 0; l <= N1; ++l)
            for (int mm = 0; mm <= N0; ++mm) {
                const double w = T0[i * (N0 + 1) + mm] * T1[j * (N1 + 1) + l];
                const int q = mm + (N0 + 1) * l;
#pragma unroll
                for (int k = 0; k < K; ++k) out[k] += w * tr[k * 64 + q];
            }
    }
}

// Face_ProjectFluxToElements for K values at once (values k at fl[k*64 + q], q = m + (Nf0+1) l)
template <int K>
__device__ __forceinline__ void project_k(const Mort &m, const Shape &r, int side, const double *fl,
                                          int i, int j, double *out)
{
    const int n0 = r.Nf0, n1 = r.Nf1;
    const int pt = projection(r, side);
    if (pt == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = fl[k * 64 + i + (n0 + 1) * j];
        return;
    }
    const double *T0 = m.p0, *T1 = m.p1;
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = 0.0;
    if (pt == 1) {
        for (int l = 0; l <= n0; ++l) {
            const double w = T0[i * (n0 + 1) + l];
            const int q = l + (n0 + 1) * j;
#pragma unroll
            for (int k = 0; k < K; ++k) out[k] += w * fl[k * 64 + q];
        }
    } else if (pt == 2) {
        for (int l = 0; l <= n1; ++l) {
            const double w = T1[j * (n1 + 1) + l];
            const int q = i + (n0 + 1) * l;
#pragma unroll
            for (int k = 0; k < K; ++k) out[k] += w * fl[k * 64 + q];
        }
    } else {
        for (int l = 0; l <= n1; ++l)
            for (int mm = 0; mm <= n0; ++mm) {
                const double w = T0[i * (n0 + 1) + mm] * T1[j * (n1 + 1) + l];
                const int q = mm + (n0 + 1) * l;
#pragma unroll
                for (int k = 0; k < K; ++k) out[k] += w * fl[k * 64 + q];
            }
    }
}

// The two-direction case (projection type 3) of adapt_k / project_k, factorised: along the
// first index into tmp (lanes (a, l) of the half-interpolated grid), then along the second.
// Each pass is the reference's interpolation along one index; the pair does (N0 + N1 + 2) K
// multiply-adds per node instead of (N0 + 1)(N1 + 1) K, in a different rounding order (within
// the 1e-12 parity bar).  Every lane of the wave calls it (it passes two block barriers);
// lanes without a node get 0.  src: K values at src[k*64 + m + (S0+1) l] of a grid of
// (S0+1) x (S1+1) nodes; out: the node (i, j) of the (D0+1) x (D1+1) grid; T0 (D0+1) x (S0+1),
// T1 (D1+1) x (S1+1); tmp: K x 64 doubles of LDS.
template <int K>
__device__ __forceinline__ void interp2_k(const double *T0, const double *T1, int S0, int S1, int D0, int D1,
                                          const double *src, double *tmp, int lane, int i, int j, bool on,
                                          double *out)
{
    if (lane < (D0 + 1) * (S1 + 1)) {
        int a, l;
        grid_ij(lane, D0 + 1, a, l);
        double acc[K];
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] = 0.0;
        for (int m = 0; m <= S0; ++m) {
            const double w = T0[a * (S0 + 1) + m];
            const int q = m + (S0 + 1) * l;
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] += w * src[k * 64 + q];
        }
#pragma unroll
        for (int k = 0; k < K; ++k) tmp[k * 64 + lane] = acc[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = 0.0;
    if (on) {
        for (int l = 0; l <= S1; ++l) {
            const double w = T1[j * (S1 + 1) + l];
            const int q = i + (D0 + 1) * l;
#pragma unroll
            for (int k = 0; k < K; ++k) out[k] += w * tmp[k * 64 + q];
        }
    }
    __syncthreads();   // tmp read: the next call may overwrite it
}

// Face_AdaptSolutionToFace / Face_ProjectFluxToElements at node (i, j) of the destination grid,
// lanes without a node (on = false) giving 0.  FACT: faces interpolated along both indices take
// the factorised pair of passes.  That is for the values that only reach the viscous terms (the
// BR1 traces and lifting of the gradient, the gradients at the face): there the different
// rounding order stays far inside the parity bar.  The state traces of the Riemann solver and
// the projected face fluxes keep the reference's order: the surface integral cancels against the
// volume integral, and factorising those measured 1.7e-12 on the 20^3 p-anisotropic case.
// Uniform per face: every lane of the wave calls it.
template <int K, bool FACT>
__device__ __forceinline__ void adapt_face(const Mort &m, const Shape &r, int side, const double *tr,
                                           double *tmp, int lane, int i, int j, bool on, double *out)
{
    if (FACT && projection(r, side) == 3) {
        interp2_k<K>(m.a0, m.a1, r.N0[side], r.N1[side], r.Nf0, r.Nf1, tr, tmp, lane, i, j, on, out);
    } else if (on) {
        adapt_k<K>(m, r, side, tr, i, j, out);
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = 0.0;
    }
}

template <int K, bool FACT>
__device__ __forceinline__ void project_face(const Mort &m, const Shape &r, int side, const double *fl,
                                             double *tmp, int lane, int i, int j, bool on, double *out)
{
    if (FACT && projection(r, side) == 3) {
        interp2_k<K>(m.p0, m.p1, r.Nf0, r.Nf1, r.N0[side], r.N1[side], fl, tmp, lane, i, j, on, out);
    } else if (on) {
        project_k<K>(m, r, side, fl, i, j, out);
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = 0.0;
    }
}

// A lane's part of a side's element trace: its node of the trace (at the side's orders, in the face
// orientation) and whether it has one; lanes without read the side's first node and discard it, so
// that every load is unconditional.
struct TraceLane {
    bool on;
    unsigned g;
};
__device__ __forceinline__ TraceLane trace_lane(const FaceRec &f, const Shape &r, int side, int ql)
{
    int i, j;
    grid_ij(ql, r.N0[side] + 1, i, j);
    const bool on = j <= r.N1[side];
    return TraceLane{on, (unsigned)(f.g0[side] + (on ? i * f.gi[side] + j * f.gj[side] : 0))};
}

// Gauss-Lobatto nodes: the trace is the face's row of nodes, K values of the node arrays src[c*S + g]
// in registers; put_trace stores them.
template <int K>
__device__ __forceinline__ void load_trace(const TraceLane &tl, const double *src, long S, double *v)
{
#pragma unroll
    for (int c = 0; c < K; ++c) v[c] = hxk::ldg(src + c * S, tl.g);
}
template <int K>
__device__ __forceinline__ void put_trace(const TraceLane &tl, const double *v, double *tr, int ql)
{
    if (tl.on) {
#pragma unroll
        for (int c = 0; c < K; ++c) tr[c * 64 + ql] = v[c];
    }
}

// Gauss nodes: the trace is the Lagrange basis at the face's end of the normal direction applied along
// it, acc = acc + value * v(l) for l = 0..N (HexElement_ProlongSolutionToFaces,
// HexElementClass.f90:233-302, and _ProlongGradientsToFaces, :304-372), into tr.  The line's loads are
// all in flight before the sum; past a short line's end the load repeats the last node and adds
// nothing.
template <int K>
__device__ __forceinline__ void prolong_trace(const FaceRec &f, int side, const TraceLane &tl, const double *src,
                                              long S, const OpsAll &ops, double *tr, int ql)
{
    const int Na = (f.na >> (8 * side)) & 7;
    const bool plus = (f.na >> (16 + side)) & 1;
    const double *vv = plus ? ops.vR[Na] : ops.vL[Na];
    const int step = plus ? -f.gn[side] : f.gn[side];   // towards larger l
    const unsigned g0 = tl.g - (plus ? Na * step : 0);
    if (tl.on) {
        double w[MAXN1];
#pragma unroll
        for (int l = 0; l < MAXN1; ++l) w[l] = l <= Na ? vv[l] : 0.0;
#pragma unroll
        for (int c = 0; c < K; ++c) {
            double x[MAXN1];
#pragma unroll
            for (int l = 0; l < MAXN1; ++l) x[l] = l <= Na ? hxk::ldg(src + c * S, g0 + l * step) : 0.0;
            double acc = 0.0;
#pragma unroll
            for (int l = 0; l < MAXN1; ++l)
                if (l <= Na) acc = acc + x[l] * w[l];
            tr[c * 64 + ql] = acc;
        }
    }
}

// The faces of one wave of the face kernels: sched[w] = (face, -1, shape) puts one face on all 64
// lanes; (face a, face b, shape) puts two faces of one shape (the same orders on both sides, so the
// same projection types and mortar matrices, at most 32 face nodes) on the two half-waves, so that
// small faces do not leave most of a wave idle.  Each half works in its own 32 columns of the
// per-face LDS rows (every grid of such a face, and every half-interpolated grid, has at most
// 32 nodes); the mortar matrices are shared.  Both halves take the same branches at every
// barrier: the shape comes with the schedule, in scalar registers, so that the interpolation loops
// count there.
struct FaceLane {
    int f;     // the lane's face
    int q;     // the lane's index within its face
    int col;   // first LDS column of its face
};
__device__ __forceinline__ FaceLane face_lane(const int4 s, int lane)
{
    const bool two = s.y >= 0;
    const int h = two ? lane >> 5 : 0;
    return FaceLane{h ? s.y : s.x, two ? (lane & 31) : lane, 32 * h};
}

// ------------------------------------------------------------------------------------
// km_face_grad: BR1 unStar = 1/2 (U_R - U_L) |Ja| n at the face nodes
// (BR1_ComputeElementInterfaceAverage, EllipticBR1.f90:571-627), projected onto both sides:
// lift[(3v + d)... laid out as lift[(d*5 + v)*ES + x].
// ------------------------------------------------------------------------------------
template <bool GAUSS>
__global__ void __launch_bounds__(64)
km_face_grad(const double *__restrict__ Q, const FaceRec *__restrict__ faces, const int4 *__restrict__ sched,
             const double *__restrict__ fgeo, int fc, const OpsAll *__restrict__ opsp, double *__restrict__ lift, int W,
             long S, long ES, long FSm)
{
    // LDS: both sides' Q traces, then one direction's unStar in their place; the mortar
    // matrices; the half-interpolated grid of a factorised interpolation (9.5 KB)
    __shared__ double sT[2][NV * 64];
    __shared__ double sM[4][64];
    __shared__ double sTmp[NV * 64];
    // waves in XCD-contiguous ranges (the grid is a multiple of 8): faces that share elements
    // mostly run on one XCD and find the elements' traces in its L2
    const int w = hxk::xcd_block(blockIdx.x, gridDim.x), lane = threadIdx.x;
    if (w >= W) return;   // uniform per block
    const int4 sc = sched[w];
    const Shape r = unpack_shape(sc.z);
    const FaceLane fl = face_lane(sc, lane);
    const int ql = fl.q;
    double *const tL = sT[0] + fl.col, *const tR = sT[1] + fl.col, *const tmp = sTmp + fl.col;
    double *const sU = tL;   // [NV][64], once both traces are at the face order
    const FaceRec f = faces[fl.f];
    double qL[NV], qR[NV];
    {
        const TraceLane a = trace_lane(f, r, 0, ql), b = trace_lane(f, r, 1, ql);
        if (GAUSS) {
            stage_mortar(*opsp, r, sM, lane);
            prolong_trace<NV>(f, 0, a, Q, S, *opsp, tL, ql);
            prolong_trace<NV>(f, 1, b, Q, S, *opsp, tR, ql);
        } else {
            load_trace<NV>(a, Q, S, qL);
            load_trace<NV>(b, Q, S, qR);
            stage_mortar(*opsp, r, sM, lane);
            put_trace<NV>(a, qL, tL, ql);
            put_trace<NV>(b, qR, tR, ql);
        }
    }
    const Mort M = mort_lds(sM);
    int i, j;
    grid_ij(ql, r.Nf0 + 1, i, j);
    const bool on = j <= r.Nf1;
    if (!on) { i = 0; j = 0; }
    const long fq = fc ? (long)fl.f : f.foff + (on ? ql : 0);
    double nrm[3];
    nrm[0] = fgeo[fq];
    nrm[1] = fgeo[FSm + fq];
    nrm[2] = fgeo[2 * FSm + fq];
    const double jac = fgeo[9 * FSm + fq];
    __syncthreads();
    double uS[NV];
    adapt_face<NV, true>(M, r, 0, tL, tmp, ql, i, j, on, qL);
    adapt_face<NV, true>(M, r, 1, tR, tmp, ql, i, j, on, qR);
#pragma unroll
    for (int v = 0; v < NV; ++v) uS[v] = 0.5 * (qR[v] - qL[v]) * jac;
    // each side's node of this lane in the projection
    bool son[2];
    int si[2], sj[2];
    unsigned sx[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        grid_ij(ql, r.N0[side] + 1, si[side], sj[side]);
        son[side] = sj[side] <= r.N1[side];
        if (!son[side]) { si[side] = 0; sj[side] = 0; }
        sx[side] = (unsigned)(f.x0[side] + si[side] * f.xi[side] + sj[side] * f.xj[side]);
    }
    // unStar(v) n_d, one direction at a time, projected onto both sides: lift[(5d + v)*ES + x]
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        __syncthreads();   // the traces (d = 0), the previous direction's unStar (d > 0) have been read
        if (on) {
#pragma unroll
            for (int v = 0; v < NV; ++v) sU[v * 64 + ql] = uS[v] * nrm[d];
        }
        __syncthreads();
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            double lv[NV];
            project_face<NV, true>(M, r, side, sU, tmp, ql, si[side], sj[side], son[side], lv);
            if (son[side]) {
#pragma unroll
                for (int v = 0; v < NV; ++v) hxk::stg(lift + (d * NV + v) * ES, sx[side], lv[v]);
            }
        }
    }
}

// ------------------------------------------------------------------------------------
// km_grad: local gradient (HexElement_ComputeLocalGradient, HexElementClass.f90:427-531) and
// BR1 lifting (BR1_GradientFaceLoop, EllipticBR1.f90:531-569, with the weights b of
// VectorWeakIntegrals_StdFace): grad Q at every node, U[(5d + v)*S + g].
// Bound by memory: 176 bytes a node (256 where the metrics are by node) and 120 an element face node; 440 MB
// on 20^3 elements of orders 2..7, 3.8 TB/s, 115 us (154.9 before what follows and before the metrics were
// read once per element).  What keeps the registers under 128 and two large tiles on a CU:
// the nodes of a tile lie together in LDS (one address per node with constant offsets, instead of one
// per value; the odd stride keeps a line's nodes in distinct banks), derivative loops that are
// not unrolled, and the lifting a direction at a time.  10^3 Gauss elements of orders 2..5: 29.6 -> 13.3 us.
// ------------------------------------------------------------------------------------
template <bool GAUSS, int T>
__global__ void __launch_bounds__(T)
km_grad(const NodeMap *__restrict__ tmap, int ntiles, const double *__restrict__ Q, hxk::Metric mt,
        const double *__restrict__ lift, const OpsAll *__restrict__ opsp,
        double *__restrict__ U, long S, long ES, Phys ph, hxk::DtLimits dtl, int pbase)
{
    HIP_DYNAMIC_SHARED(double, smem)
    const OpsAll &ops = *opsp;
    const int t = threadIdx.x;
    double *sD = smem;                   // D of every order, [MAXN1][64] (visible after the first barrier)
    double *sQall = smem + MAXN1 * 64;   // [node of the tile][NV]
    for (int x = t; x < MAXN1 * 64; x += blockDim.x) sD[x] = ops.D[x / 64][x % 64];
    double tc = INFINITY, tv = INFINITY;   // MaxTimeStep limits of this thread's nodes (stage 1)
    NodeMap nm = load_map<T>(tmap, blockIdx.x < ntiles ? blockIdx.x : 0, t);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int code = nm.code, ef0 = nm.ef0;
    const unsigned g = nm.g;   // loads are unconditional (see k_volume)
    const int i = code & 7, j = (code >> 3) & 7, k = (code >> 6) & 7;
    const int Nx = (code >> 9) & 7, Ny = (code >> 12) & 7, Nz = (code >> 15) & 7;
    const int nx = Nx + 1, ny = Ny + 1, nz = Nz + 1;
    const int first = (code >> 18) & 511;
    const bool active = (code >> 27) & 1;
    const int n = i + nx * (j + ny * k);
    double q[NV], ja[9];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = hxk::ldg(Q + v * S, g);
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = hxk::ldg(mt.Ja + c * mt.S, mt.node(nm.e, g));
    const double jg = hxk::ldg(mt.J, mt.node(nm.e, g));
    if (tile + (int)gridDim.x < ntiles) nm = load_map<T>(tmap, tile + gridDim.x, t);   // the next tile's
    const double iJ = 1.0 / jg;   // the same bits as a stored 1/J
    const bool onx = i == 0 || i == Nx, ony = j == 0 || j == Ny, onz = k == 0 || k == Nz;
    const ElemFaces ef = elem_faces(ef0, nx, ny, nz);
    const unsigned xx = (i == 0 ? ef.s[5] : ef.s[3]) + j + ny * k, xy = (j == 0 ? ef.s[0] : ef.s[1]) + i + nx * k,
                   xz = (k == 0 ? ef.s[2] : ef.s[4]) + i + nx * j;
    double *sQ = sQall + NV * first;   // [ne][NV]
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) sQ[NV * n + v] = q[v];
    }
    __syncthreads();
    if (active) {
    // Gauss-Lobatto: the lifting values of the node's faces (slots 5/3, 0/1, 2/4), a direction of the
    // gradient at a time (all at once they took 60 registers more); the first direction's are asked
    // for ahead of the derivatives
    double h[3][NV];
    auto ask = [&](int d) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double *lc = lift + (long)(d * NV + v) * ES;
            h[0][v] = hxk::ldg(lc, xx);
            h[1][v] = hxk::ldg(lc, xy);
            h[2][v] = hxk::ldg(lc, xz);
        }
        hxk::sched_fence();
    };
    if (!GAUSS) ask(0);
    const double *Dx = sD + 64 * Nx, *Dy = sD + 64 * Ny, *Dz = sD + 64 * Nz;
    double uxi[NV], ueta[NV], uzeta[NV];
    auto line = [](const double *a, int step, const double *w, int len, double *u) {
#pragma unroll
        for (int v = 0; v < NV; ++v) u[v] = 0.0;
#pragma unroll 1
        for (int l = 0; l < len; ++l) {
#pragma unroll
            for (int v = 0; v < NV; ++v) u[v] = u[v] + a[l * step + v] * w[l];
        }
    };
    line(sQ + NV * (nx * (j + ny * k)), NV, Dx + i * 8, nx, uxi);
    line(sQ + NV * (i + nx * ny * k), NV * nx, Dy + j * 8, ny, ueta);
    line(sQ + NV * (i + nx * j), NV * nx * ny, Dz + k * 8, nz, uzeta);
    if (GAUSS) {
        // every node takes the lifting values of all six faces with its surface weights b,
        // in the order L, R (xi), FR, BK (eta), BOT, T (zeta) of VectorWeakIntegrals_StdFace
        // (DGIntegrals.f90:365-443); slots 5, 3, 0, 1, 2, 4
        const unsigned xl = ef.s[5] + j + ny * k, xr = ef.s[3] + j + ny * k;
        const unsigned xf = ef.s[0] + i + nx * k, xb = ef.s[1] + i + nx * k;
        const unsigned xo = ef.s[2] + i + nx * j, xt = ef.s[4] + i + nx * j;
        const double bl = ops.bL[Nx][i], br = ops.bR[Nx][i], bf = ops.bL[Ny][j], bb = ops.bR[Ny][j];
        const double bo = ops.bL[Nz][k], bt = ops.bR[Nz][k];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double gr[3];
            gr[0] = (uxi[v] * ja[0] + ueta[v] * ja[3] + uzeta[v] * ja[6]) * iJ;
            gr[1] = (uxi[v] * ja[1] + ueta[v] * ja[4] + uzeta[v] * ja[7]) * iJ;
            gr[2] = (uxi[v] * ja[2] + ueta[v] * ja[5] + uzeta[v] * ja[8]) * iJ;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double *lc = lift + (long)(d * NV + v) * ES;
                double fi = hxk::ldg(lc, xl) * bl;
                fi = fi + hxk::ldg(lc, xr) * br;
                fi = fi + hxk::ldg(lc, xf) * bf;
                fi = fi + hxk::ldg(lc, xb) * bb;
                fi = fi + hxk::ldg(lc, xo) * bo;
                fi = fi + hxk::ldg(lc, xt) * bt;
                hxk::stg(U + (d * NV + v) * S, g, gr[d] + fi * iJ);
            }
        }
    } else {
        const double bx = ops.b0[Nx], by = ops.b0[Ny], bz = ops.b0[Nz];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (d) ask(d);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double gr = (uxi[v] * ja[d] + ueta[v] * ja[3 + d] + uzeta[v] * ja[6 + d]) * iJ;
                // absent faces give 0
                const double ax = onx ? h[0][v] * bx : 0.0;
                const double ay = ony ? h[1][v] * by : 0.0;
                const double az = onz ? h[2][v] * bz : 0.0;
                const double fi = ((0.0 + ax) + ay) + az;
                hxk::stg(U + (d * NV + v) * S, g, (onx || ony || onz) ? gr + fi * iJ : gr);
            }
            hxk::sched_fence();
        }
    }
    if (dtl.part) {
        double c0, c1;
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = sQ[NV * n + v];   // again: not held through the derivatives
        hx::dt_limits(ph, q, ja, jg, ops.dcsi[Nx], ops.dcsi[Ny], ops.dcsi[Nz], dtl.cfl, dtl.dcfl, c0, c1);
        tc = fmin(tc, c0);
        tv = fmin(tv, c1);
    }
    }
    __syncthreads();   // the tile's sQ has been read: the next tile overwrites it
    }
    if (dtl.part) hxk::block_min_pair(tc, tv, dtl.part, t, pbase + blockIdx.x);
}

// ------------------------------------------------------------------------------------
// km_face: computeElementInterfaceFlux (SD.f90:1710-1799) at the face order with the face
// viscosities of compute_viscosity_at_faces (SD.f90:1345-1398), projected back
// (FaceClass.f90:597-700) and scaled by the receiving element's surface weight:
// fe[v*ES + x] = (+/-) projected flux * b.
// ------------------------------------------------------------------------------------
template <bool GAUSS, bool LES>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
km_face(const double *__restrict__ Q, const double *__restrict__ U, const FaceRec *__restrict__ faces,
        const int4 *__restrict__ sched, const double *__restrict__ fgeo, int fc, const double *__restrict__ fdelta,
        const OpsAll *__restrict__ opsp, double *__restrict__ fe, int W, long S, long ES, long FSm, Phys ph,
        hxk::DtReduce dtr)
{
    // LDS: both sides' Q traces (rows 0-4, 5-9), then one side's grad Q trace at a time, then
    // the face flux, in one space; the mortar matrices; the half-interpolated grid of a
    // factorised interpolation (12.25 KB: three waves per SIMD)
    __shared__ double sR[3 * NV * 64];
    __shared__ double sM[4][64];
    __shared__ double sTmp[NV * 64];
    // waves in XCD-contiguous ranges (the grid is a multiple of 8): faces that share elements
    // mostly run on one XCD and find the elements' traces in its L2
    const int w = hxk::xcd_block(blockIdx.x, gridDim.x), lane = threadIdx.x;
    if (dtr.bits && w == 0) hxk::reduce_dt_partials(dtr.part, dtr.n, dtr.bits, lane);
    if (w >= W) return;   // uniform per block
    const int4 sc = sched[w];
    const Shape r = unpack_shape(sc.z);
    const FaceLane fl = face_lane(sc, lane);
    const int ql = fl.q;
    double *const qLt = sR + fl.col, *const qRt = sR + NV * 64 + fl.col, *const gT = sR + fl.col,
                  *const tmp = sTmp + fl.col;
    const FaceRec f = faces[fl.f];
    const TraceLane tl[2] = {trace_lane(f, r, 0, ql), trace_lane(f, r, 1, ql)};
    double qs[2][NV];
    // Gauss-Lobatto: the left side's gradients are asked for with the state traces, the right side's
    // while the left's are interpolated.  (Without the LES model as a template flag these 30 registers
    // would spill at three waves per SIMD.)
    double gv[3 * NV];
    if (!GAUSS) {
        load_trace<NV>(tl[0], Q, S, qs[0]);
        load_trace<NV>(tl[1], Q, S, qs[1]);
        if (!ph.euler) load_trace<3 * NV>(tl[0], U, S, gv);
    }
    stage_mortar(*opsp, r, sM, lane);
    const Mort M = mort_lds(sM);
    if (GAUSS) {
        prolong_trace<NV>(f, 0, tl[0], Q, S, *opsp, qLt, ql);
        prolong_trace<NV>(f, 1, tl[1], Q, S, *opsp, qRt, ql);
    } else {
        put_trace<NV>(tl[0], qs[0], qLt, ql);
        put_trace<NV>(tl[1], qs[1], qRt, ql);
    }
    // lanes past the face's nodes work on node (0, 0) and discard the result (every index stays
    // inside the face's arrays)
    int i, j;
    grid_ij(ql, r.Nf0 + 1, i, j);
    const bool on = j <= r.Nf1;
    if (!on) { i = 0; j = 0; }
    const long fq = fc ? (long)fl.f : f.foff + (on ? ql : 0);
    double nrm[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) nrm[c] = fgeo[c * FSm + fq];
    const double jac = fgeo[9 * FSm + fq];
    const double fd = LES ? fdelta[fl.f] : 0.0;
    __syncthreads();
    adapt_face<NV, false>(M, r, 0, qLt, tmp, ql, i, j, on, qs[0]);
    adapt_face<NV, false>(M, r, 1, qRt, tmp, ql, i, j, on, qs[1]);
    __syncthreads();   // the Q traces are read: the space takes a grad Q trace or the face flux
    double visc[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (!ph.euler) {
        // BR1_RiemannSolver (EllipticBR1.f90:816-868): each side's viscous flux from its
        // gradients at the face order, the sides one after the other through the trace space; the
        // gradients (15 values) are interpolated five at a time (the size of sTmp)
        auto side_grad = [&](int s, double *g) {
#pragma unroll
            for (int c = 0; c < 3; ++c) adapt_face<NV, true>(M, r, s, gT + c * NV * 64, tmp, ql, i, j, on, g + c * NV);
        };
        auto side_flux = [&](int s, const double *g, double *ft) {
            double vg[12], sh[6], mu, kappa;
            hx::viscous_state(ph, qs[s], g, g + NV, g + 2 * NV, vg);
            hx::laminar_mu_kappa(ph, qs[s], mu, kappa);
            if (LES) {
                const double mt = hx::les_mu(ph, fd, qs[s][0], hx::les_factor(ph, qs[s], g, g + NV, g + 2 * NV));
                mu = mu + mt;
                kappa = kappa + mt * ph.mu_to_kappa;
            }
            const double ir = 1.0 / qs[s][0];
            hx::stress_shape(vg, sh);
            hx::viscous_tensor(mu, kappa, qs[s][1] * ir, qs[s][2] * ir, qs[s][3] * ir, sh, vg + 9, ft);
        };
        double fa[9], fb[9], g[3 * NV];
        if (GAUSS) {
            prolong_trace<3 * NV>(f, 0, tl[0], U, S, *opsp, gT, ql);
        } else {
            put_trace<3 * NV>(tl[0], gv, gT, ql);
            load_trace<3 * NV>(tl[1], U, S, gv);
        }
        __syncthreads();
        side_grad(0, g);
        if (on) side_flux(0, g, fa);
        __syncthreads();   // side 0's gradients consumed
        if (GAUSS) prolong_trace<3 * NV>(f, 1, tl[1], U, S, *opsp, gT, ql);
        else put_trace<3 * NV>(tl[1], gv, gT, ql);
        __syncthreads();
        side_grad(1, g);
        if (on) {
            side_flux(1, g, fb);
#pragma unroll
            for (int c = 0; c < 9; ++c) fa[c] = 0.5 * (fa[c] + fb[c]);
#pragma unroll
            for (int v = 1; v < NV; ++v)
                visc[v] = fa[hx::viscous_entry(v, 0)] * nrm[0] + fa[hx::viscous_entry(v, 1)] * nrm[1] +
                          fa[hx::viscous_entry(v, 2)] * nrm[2];
        }
        __syncthreads();   // the space takes the face flux next
    }
    double *const sF = gT;   // face flux [NV][64]
    if (on) {
        double inv[NV];
        if (ph.riemann == 1) {
            double t1[3], t2[3];   // the tangents: the Lax-Friedrichs flux alone reads them
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                t1[c] = fgeo[(3 + c) * FSm + fq];
                t2[c] = fgeo[(6 + c) * FSm + fq];
            }
            hx::lxf_flux(ph, qs[0], qs[1], nrm, t1, t2, inv);
        } else {
            hx::roe_flux(ph, qs[0], qs[1], nrm, inv);
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) sF[v * 64 + ql] = (inv[v] - visc[v]) * jac;
    }
    __syncthreads();
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        int si, sj;
        grid_ij(ql, r.N0[side] + 1, si, sj);
        const bool son = sj <= r.N1[side];
        if (!son) { si = 0; sj = 0; }
        double a[NV];
        project_face<NV, false>(M, r, side, sF, tmp, ql, si, sj, son, a);
        if (son) {
            const unsigned x = (unsigned)(f.x0[side] + si * f.xi[side] + sj * f.xj[side]);
            // Gauss nodes: the surface weights b(i) of every node are applied by the volume kernel
            const double b = GAUSS ? 1.0 : opsp->b0[(f.na >> (8 * side)) & 7];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double x0 = side == 0 ? a[v] : -1.0 * a[v];
                hxk::stg(fe + v * ES, x, GAUSS ? x0 : x0 * b);
            }
        }
    }
}

// ------------------------------------------------------------------------------------
// km_volume: as hxk::k_volume with the element's own orders per direction, the viscous
// state formed from grad Q (ViscousFlux_STATE), and MaxTimeStep's 1/|x_1 - x_0| per direction.
// LDS (dynamic): hatD and sharpD of every order [2][MAXN1][64], then each node's fluxes and data
// together (see km_grad).
// Bound by memory: 296 bytes a node (376 where the metrics are by node) and 40 an element face node; 493 MB
// on 20^3 elements of orders 2..7, standard form, 5.0 TB/s, 99 us (158.3 before what follows and before the
// metrics were read once per element).  That takes two large tiles per CU (four waves per SIMD,
// 128 registers): the surface integral is summed as its loads arrive, the fluxes go to LDS a direction
// at a time.  The split form's LDS admits one large tile.  Gauss nodes, with six faces' loads in
// flight per node, are faster with the registers (10^3 elements of orders 2..5: 12.7 us against 18.5 at
// four waves), and so is LES, which takes 164 of them (20^3, orders 2..7, Smagorinsky 113.8 us against 117.6,
// WALE 118.1 against 157.1; 20^3 of order 3 but for one element 38.6 against 42.8 and 39.4 against 58.9).
// ------------------------------------------------------------------------------------
template <int FORM>
constexpr int mvolume_per_node()
{
    // odd: the nodes of a wave's line lie in distinct banks
    return (3 * (FORM >= 0 ? 4 : 5) + (FORM >= 0 ? hx::node_data_size(FORM) + 3 : 0)) | 1;
}

template <int FORM, bool GAUSS, bool LES, int T>
__global__ void __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(FORM < 0 && !GAUSS && !LES ? 4 : 2)))
km_volume(const NodeMap *__restrict__ tmap, int ntiles, double *__restrict__ Q, const double *__restrict__ U,
          hxk::Metric mt, const double *__restrict__ edelta,
          const double *__restrict__ fe, const OpsAll *__restrict__ opsp, double *__restrict__ G,
          double *__restrict__ qdot_out, double a_k, double c_k, int update, DtArgs dta, long S, long ES,
          Phys ph)
{
    constexpr bool SPLIT = FORM >= 0;
    constexpr int AVG = SPLIT ? FORM : 0;
    constexpr int ND = hx::node_data_size(AVG);
    constexpr bool SYM = hx::two_point_symmetric(AVG);
    constexpr int NF = SPLIT ? 4 : 5, V0 = SPLIT ? 1 : 0;
    constexpr int PER_NODE = mvolume_per_node<FORM>();
    HIP_DYNAMIC_SHARED(double, smem)
    const OpsAll &ops = *opsp;
    const int t = threadIdx.x;
    // hatD and sharpD of every order (read at LDS latency in the contractions below; visible
    // after the first barrier of the direction loop)
    double *sOp = smem;
    for (int x = t; x < 2 * MAXN1 * 64; x += blockDim.x)
        sOp[x] = x < MAXN1 * 64 ? ops.hatD[x / 64][x % 64] : ops.sharpD[(x / 64) - MAXN1][x % 64];
    double *chunk0 = smem + 2 * MAXN1 * 64;
    NodeMap nm = load_map<T>(tmap, blockIdx.x < ntiles ? blockIdx.x : 0, t);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int e = nm.e, code = nm.code, ef0 = nm.ef0;
    const unsigned g = nm.g;
    const int i = code & 7, j = (code >> 3) & 7, k = (code >> 6) & 7;
    const int Nx = (code >> 9) & 7, Ny = (code >> 12) & 7, Nz = (code >> 15) & 7;
    const int nx = Nx + 1, ny = Ny + 1, nz = Nz + 1;
    const int first = (code >> 18) & 511;
    const bool active = (code >> 27) & 1;
    const int n = i + nx * (j + ny * k);
    const bool onx = i == 0 || i == Nx, ony = j == 0 || j == Ny, onz = k == 0 || k == Nz;
    // this node's values: the fluxes [3][NF] (the split form: viscous fluxes), the two-point data
    // [ND], the metric row [3]; the node at distance m along an axis lies m * PER_NODE further
    double *mine = chunk0 + PER_NODE * (first + n);
    constexpr int ON = 3 * NF, OJ = ON + ND;
    // loads, unconditional (see hxk::k_volume)
    double q[NV], ja[9], gq[3][NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) q[v] = hxk::ldg(Q + v * S, g);
#pragma unroll
    for (int c = 0; c < 9; ++c) ja[c] = hxk::ldg(mt.Ja + c * mt.S, mt.node(e, g));
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int v = 0; v < NV; ++v) gq[d][v] = hxk::ldg(U + (d * NV + v) * S, g);
    const double dl = hxk::ldg(edelta, (unsigned)e);
    const double jg = hxk::ldg(mt.J, mt.node(e, g));
    if (tile + (int)gridDim.x < ntiles) nm = load_map<T>(tmap, tile + gridDim.x, t);   // the next tile's
    double xs[NV];   // the node's surface integral
    const ElemFaces ef = elem_faces(ef0, nx, ny, nz);
    if (GAUSS) {
        // surface integral on every node: the face fluxes of all six faces with the node's
        // surface weights, L, R, FR, BK, BOT, T (ScalarWeakIntegrals_StdFace, DGIntegrals.f90:
        // 214-273)
        const unsigned xl = ef.s[5] + j + ny * k, xr = ef.s[3] + j + ny * k;
        const unsigned xf = ef.s[0] + i + nx * k, xb = ef.s[1] + i + nx * k;
        const unsigned xo = ef.s[2] + i + nx * j, xt = ef.s[4] + i + nx * j;
        const double bl = ops.bL[Nx][i], br = ops.bR[Nx][i], bf = ops.bL[Ny][j], bb = ops.bR[Ny][j];
        const double bo = ops.bL[Nz][k], bt = ops.bR[Nz][k];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double *fv = fe + (long)v * ES;
            double x = hxk::ldg(fv, xl) * bl;
            x = x + hxk::ldg(fv, xr) * br;
            x = x + hxk::ldg(fv, xf) * bf;
            x = x + hxk::ldg(fv, xb) * bb;
            x = x + hxk::ldg(fv, xo) * bo;
            x = x + hxk::ldg(fv, xt) * bt;
            xs[v] = x;
        }
    } else {
        const unsigned xx = (i == 0 ? ef.s[5] : ef.s[3]) + j + ny * k, xy = (j == 0 ? ef.s[0] : ef.s[1]) + i + nx * k,
                       xz = (k == 0 ? ef.s[2] : ef.s[4]) + i + nx * j;
        double sx[NV], sy[NV], sz[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const double a = hxk::ldg(fe + v * ES, xx), b = hxk::ldg(fe + v * ES, xy), c = hxk::ldg(fe + v * ES, xz);
            sx[v] = onx ? a : 0.0;
            sy[v] = ony ? b : 0.0;
            sz[v] = onz ? c : 0.0;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) xs[v] = ((0.0 + sx[v]) + sy[v]) + sz[v];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) hxk::hold(xs[v]);
    hxk::sched_fence();
    if (active) {
        double ft[9];   // the viscous tensor (hx::viscous_entry)
        if (!ph.euler) {
            double vg[12], sh[6], mu, kappa;
            hx::viscous_state(ph, q, gq[0], gq[1], gq[2], vg);
            hx::laminar_mu_kappa(ph, q, mu, kappa);
            if (LES) {
                const double mut = hx::les_mu(ph, dl, q[0], hx::les_factor(ph, q, gq[0], gq[1], gq[2]));
                mu = mu + mut;
                kappa = kappa + mut * ph.mu_to_kappa;
            }
            const double ir = 1.0 / q[0];
            hx::stress_shape(vg, sh);
            hx::viscous_tensor(mu, kappa, q[1] * ir, q[2] * ir, q[3] * ir, sh, vg + 9, ft);
        } else {
#pragma unroll
            for (int c = 0; c < 9; ++c) ft[c] = 0.0;
        }
#pragma unroll
        for (int c = 0; c < 9; ++c) hxk::hold(ft[c]);
        double pu, pv, pw, pp;
        hx::euler_primitives(ph, q, pu, pv, pw, pp);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double fi[NV];
            if (!SPLIT) hx::euler_contravariant_row(q, pu, pv, pw, pp, &ja[3 * d], fi);
#pragma unroll
            for (int v = V0; v < NV; ++v) {
                const double fv = v == 0 ? 0.0
                                         : ft[hx::viscous_entry(v, 0)] * ja[3 * d] + ft[hx::viscous_entry(v, 1)] * ja[3 * d + 1] +
                                               ft[hx::viscous_entry(v, 2)] * ja[3 * d + 2];
                mine[d * NF + v - V0] = SPLIT ? fv : fi[v] - fv;
            }
            hxk::sched_fence();
        }
        if (SPLIT) {
            double a[ND];
            hx::node_data<AVG>(ph, q, a);
#pragma unroll
            for (int c = 0; c < ND; ++c) mine[ON + c] = a[c];
        }
    }
    double qd[NV], gk[NV], dt0 = 0.0, dt1 = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v) qd[v] = 0.0;
    for (int d = 0; d < 3; ++d) {
        double jh[3];   // this node's metric row times metric_scale
#pragma unroll
        for (int c = 0; c < 3; ++c) jh[c] = hx::metric_scale(AVG) * ja[3 * d + c];
        if (SPLIT) {
            if (d) __syncthreads();
            if (active) {
#pragma unroll
                for (int c = 0; c < 3; ++c) mine[OJ + c] = jh[c];
            }
        }
        if (SPLIT || d == 0) __syncthreads();
        if (d == 2) {
#pragma unroll
            for (int v = 0; v < NV; ++v) gk[v] = hxk::ldg(G + v * S, g);
            dt0 = hxk::bits_to_double(dta.in[0]);
            dt1 = hxk::bits_to_double(dta.in[1]);
        }
        if (!active) continue;
        const int own = d == 0 ? i : (d == 1 ? j : k);
        const int Nd = d == 0 ? Nx : (d == 1 ? Ny : Nz);
        const int stride = d == 0 ? 1 : (d == 1 ? nx : nx * ny);
        const double *line = mine - own * stride * PER_NODE;   // node 0 of this node's line
        const double *hatD = sOp + 64 * Nd + own * 8, *sharpD = hatD + MAXN1 * 64;
        if (!SPLIT) {
#pragma unroll(GAUSS ? 2 : 1)
            for (int l = 0; l <= Nd; ++l) {
                const double *m = line + l * stride * PER_NODE;
                const double hh = hatD[l];
#pragma unroll
                for (int v = 0; v < NV; ++v) qd[v] = qd[v] + hh * m[d * NF + v];
            }
        } else {
            double fi[NV], pu, pv, pw, pp;
            hx::euler_primitives(ph, q, pu, pv, pw, pp);
            hx::euler_contravariant_row(q, pu, pv, pw, pp, &ja[3 * d], fi);
#pragma unroll 1
            for (int l = 0; l <= Nd; ++l) {
                const double sh = sharpD[l], hh = hatD[l];
                const double *m = line + l * stride * PER_NODE;
                double a[ND], b[ND], jb[3], fs[NV];
#pragma unroll
                for (int c = 0; c < ND; ++c) { a[c] = mine[ON + c]; b[c] = m[ON + c]; }
#pragma unroll
                for (int c = 0; c < 3; ++c) jb[c] = m[OJ + c];
                if (SYM) {
                    hx::two_point<AVG>(a, jh, b, jb, fs);
                } else {
                    const bool lo = own < l;
                    double x1[ND], x2[ND], j1[3], j2[3];
#pragma unroll
                    for (int c = 0; c < ND; ++c) { x1[c] = lo ? a[c] : b[c]; x2[c] = lo ? b[c] : a[c]; }
#pragma unroll
                    for (int c = 0; c < 3; ++c) { j1[c] = lo ? jh[c] : jb[c]; j2[c] = lo ? jb[c] : jh[c]; }
                    hx::two_point<AVG>(x1, j1, x2, j2, fs);
                }
                qd[0] = qd[0] + sh * (l == own ? fi[0] : fs[0]);
#pragma unroll
                for (int v = 1; v < NV; ++v)
                    qd[v] = qd[v] + sh * (l == own ? fi[v] : fs[v]) + hh * m[d * NF + v - V0];
            }
        }
    }
    if (active) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if (SPLIT) qd[v] = -qd[v];
            hxk::hold(xs[v]);
            qd[v] = qd[v] - xs[v];
        }
        const double ijg = 1.0 / jg;
#pragma unroll
        for (int v = 0; v < NV; ++v) qd[v] = qd[v] * ijg;
        if (qdot_out) {
#pragma unroll
            for (int v = 0; v < NV; ++v) hxk::stg(qdot_out + v * S, g, qd[v]);
        }
        if (update) {
            hxk::hold(dt0);
            hxk::hold(dt1);
            const double dt = fmin(dt0, dt1);
            if (dta.time && tile == 0 && t == 0) dta.time[0] += dt;   // the host passes the time to one launch per stage
            const double cdt = c_k * dt;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                hxk::hold(gk[v]);
                const double gv = a_k * gk[v] + qd[v];
                hxk::stg(G + v * S, g, gv);
                q[v] = q[v] + cdt * gv;
                hxk::stg(Q + v * S, g, q[v]);
            }
            if (dta.nan && (isnan(q[0]) || isnan(q[1]) || isnan(q[2]) || isnan(q[3]) || isnan(q[4])))
                atomicOr(dta.nan, 1);
        }
    }
    __syncthreads();   // the tile's LDS has been read: the next tile overwrites it
    }
}

// MaxTimeStep of the resident state for mixed orders: one thread per node, the element of each
// node from eofn (DGSEMClass.f90:870-1035); block minima to part (see k_dt_reduce).
__global__ void __launch_bounds__(256)
km_maxdt(const double *__restrict__ Q, const double *__restrict__ Ja, const double *__restrict__ Jac,
         const int *__restrict__ eofn, const int *__restrict__ N3, const OpsAll *__restrict__ opsp,
         long nodes, long S, double cfl, double dcfl, Phys ph, double *__restrict__ part)
{
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double tc = INFINITY, tv = INFINITY;
    if (g < nodes) {
        const int e = eofn[g];
        const double dc = opsp->dcsi[N3[3 * e]], de = opsp->dcsi[N3[3 * e + 1]], dz = opsp->dcsi[N3[3 * e + 2]];
        double q[NV], ja[9];
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = Q[v * S + g];
#pragma unroll
        for (int c = 0; c < 9; ++c) ja[c] = Ja[c * S + g];
        hx::dt_limits(ph, q, ja, Jac[g], dc, de, dz, cfl, dcfl, tc, tv);
    }
    hxk::block_min_pair(tc, tv, part, threadIdx.x, blockIdx.x);
}

}  // namespace hxm
