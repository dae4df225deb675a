// Quadrilaterals and hexahedra that the sum-factorised tensor kernels of
// tensor.hip do not take: elements whose map is not affine (the bilinear /
// trilinear map of MappingToPhysHypercubeLinear, kernel/Geometry/Mappings/
// MappingToPhysHypercubeLinear.cpp:222-304) and neighbours that meet across a
// face rotated against them or through another local face (FaceGeometry.cpp:
// 148-155, the face maps of ReferenceSquare/ReferenceCube).
//
// Gauss-point form. hpGEM integrates an order-p element with its rule of
// order 2p+1, the (p+1)-point Gauss rule per direction, so with B = B1 (x) B1
// (x) B1, B1(q,a) = psi_a(x_q) square and invertible, the mass matrix it
// factorises on every call is M_e = B^T W B (W = diag(w_q |det J(x_q)|)) and
// has the exact inverse B^{-1} W^{-1} B^{-T}. With U = B u the point values:
//   advection  k = B^{-1} W^{-1} [ sum_r C_r^T (W ahat_r U) + sum_f lam_f (x) c_f ],
//              ahat = J^{-1} a at each point, C_r = C along direction r
//              (C = derivative of the interpolant of point values);
//   acoustic   k_v = B^{-1} [ div s + W^{-1} sum_f lam_f (x) c_f^v ],
//              k_s = B^{-1} [ grad v + W^{-1} sum_f lam_f (x) c_f^s ] / c_inv,
// where c_f holds, at the face's Gauss points, the flux integrand times the
// face weight and area element, and lam_f = B1^{-T} e_side (Lagrange
// polynomials of the points at +-1) lifts it to the element's points. This
// is hpGEM's operator with hpGEM's quadrature (element and face integrals of
// HpgemAPILinear::createStiffnessMatrices with the integrands of
// 080AdvectionLinear_SelfTest.cpp:108-170 and AcousticWaveLinear_Impl.h:
// 102-283, mass solve of HpgemAPILinear_Impl.h:143-156), evaluated in another
// order: results agree with it to rounding.
//
// Faces: hpGEM evaluates every face integrand at the face rule's points p
// (face coordinates of the left element L, the lower-numbered one), takes
// L's trace at L's point of p and the right element's trace at R's point of
// map(p), where map is the square's orientation map that the reference picks
// from the two faces' node lists; normal and area element come from L's map at
// p. Each element here loops over its own face points and pairs them the same
// way; for faces where it is R, it evaluates L's normal from L's vertices at
// L's point, so both sides use the same normal, as in hpGEM.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <string>
#include <unordered_map>
#include <vector>

#include "context.hpp"

namespace hgdg {

namespace {

constexpr int kGenTarget = 256;  // threads per workgroup aimed at

__host__ __device__ constexpr int ipow(int b, int e) { return e == 0 ? 1 : b * ipow(b, e - 1); }

template <int DIM, int N1>
struct GenShape {
    static constexpr int NP = ipow(N1, DIM);       // points = coefficients per field
    static constexpr int NFP = ipow(N1, DIM - 1);  // points per face
    static constexpr int NV = 1 << DIM;
    static constexpr int NFACE = 2 * DIM;
    static constexpr int EPB = NP >= kGenTarget ? 1 : kGenTarget / NP;
    static constexpr int THREADS = EPB * NP;
};

// Offsets in the packed NodalOps table of order N1 - 1.
template <int N1>
struct NodalTab {
    static constexpr int X = 0, W = N1, B = 2 * N1, BINV = B + N1 * N1, C = BINV + N1 * N1, LAM0 = C + N1 * N1,
                         LAM1 = LAM0 + N1, X2 = LAM1 + N1, W2 = X2 + N1 + 1, B2 = W2 + N1 + 1,
                         SIZE = B2 + N1 * (N1 + 1);
};

// Local faces of the reference square (0: y = -1, 1: x = -1, 2: x = 1, 3: y = 1)
// and cube (0: z = -1, 1: y = -1, 2: x = -1, 3: x = 1, 4: y = 1, 5: z = 1); a
// face's coordinates are the element coordinates other than its axis, in
// increasing order (MappingToRefLineToSquare, MappingToRefSquareToCube).
__host__ __device__ constexpr int face_axis(int dim, int f) {
    return dim == 2 ? ((f == 1 || f == 2) ? 0 : 1) : ((f == 2 || f == 3) ? 0 : (f == 1 || f == 4) ? 1 : 2);
}
__host__ __device__ constexpr int face_side(int dim, int f) { return dim == 2 ? (f >= 2 ? 1 : 0) : (f >= 3 ? 1 : 0); }
// the k-th face coordinate axis (k = 0, 1)
__host__ __device__ constexpr int face_coord_axis(int dim, int f, int k) {
    return face_axis(dim, f) <= k ? k + 1 : k;
}
// Sign that turns the wedge product of the face tangents into the outward
// normal for a positively oriented element (the same sign per face in both
// shapes: odd faces +1, even faces -1).
__host__ __device__ constexpr double face_sign(int f) { return (f & 1) ? 1.0 : -1.0; }

// Point x(xi) and Jacobian J[r][d] = dx_r / dxi_d of the multilinear map of
// the element with vertices X[v][r] (vertex v at the corner whose coordinate
// d is -1 / +1 by bit d of v).
template <int DIM>
__device__ inline void multilinear(const double* X, const double* xi, double (&J)[DIM][DIM], double* x) {
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
        if (x) x[r] = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) J[r][d] = 0;
    }
#pragma unroll
    for (int v = 0; v < (1 << DIM); ++v) {
        double f[DIM], g[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const bool hi = (v >> d) & 1;
            f[d] = hi ? 0.5 * (1 + xi[d]) : 0.5 * (1 - xi[d]);
            g[d] = hi ? 0.5 : -0.5;
        }
        double prod = 1;
#pragma unroll
        for (int d = 0; d < DIM; ++d) prod *= f[d];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            double dd = g[d];
#pragma unroll
            for (int k = 0; k < DIM; ++k)
                if (k != d) dd *= f[k];
#pragma unroll
            for (int r = 0; r < DIM; ++r) J[r][d] += X[v * DIM + r] * dd;
        }
        if (x) {
#pragma unroll
            for (int r = 0; r < DIM; ++r) x[r] += X[v * DIM + r] * prod;
        }
    }
}

template <int DIM>
__device__ inline double det_inv(const double (&J)[DIM][DIM], double (&Ji)[DIM][DIM]) {
    if constexpr (DIM == 2) {
        const double det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
        Ji[0][0] = J[1][1] / det;
        Ji[0][1] = -J[0][1] / det;
        Ji[1][0] = -J[1][0] / det;
        Ji[1][1] = J[0][0] / det;
        return det;
    } else {
        const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                           J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                           J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int r1 = (c + 1) % 3, r2 = (c + 2) % 3, c1 = (r + 1) % 3, c2 = (r + 2) % 3;
                Ji[r][c] = (J[r1][c1] * J[r2][c2] - J[r1][c2] * J[r2][c1]) / det;
            }
        return det;
    }
}

// Outward normal scaled by the area element at face point (qa, qb) of face f
// of the element with vertices X (hpGEM's PhysicalFace normal: wedge product
// of the mapped face tangents, signed per face and by the orientation of the
// element map).
template <int DIM, int N1>
__device__ inline void face_normal(const double* X, int f, int qa, int qb, const double* tab, double (&n)[DIM]) {
    double xi[DIM];
    xi[face_axis(DIM, f)] = face_side(DIM, f) ? 1.0 : -1.0;
    xi[face_coord_axis(DIM, f, 0)] = tab[NodalTab<N1>::X + qa];
    if constexpr (DIM == 3) xi[face_coord_axis(DIM, f, 1)] = tab[NodalTab<N1>::X + qb];
    double J[DIM][DIM], Ji[DIM][DIM];
    multilinear<DIM>(X, xi, J, nullptr);
    const double det = det_inv<DIM>(J, Ji);
    const double s = face_sign(f) * (det > 0 ? 1.0 : -1.0);
    const int a0 = face_coord_axis(DIM, f, 0);
    if constexpr (DIM == 2) {
        n[0] = -J[1][a0] * s;
        n[1] = J[0][a0] * s;
    } else {
        const int a1 = face_coord_axis(DIM, f, 1);
        n[0] = (J[1][a0] * J[2][a1] - J[2][a0] * J[1][a1]) * s;
        n[1] = (J[2][a0] * J[0][a1] - J[0][a0] * J[2][a1]) * s;
        n[2] = (J[0][a0] * J[1][a1] - J[1][a0] * J[0][a1]) * s;
    }
}

// sum_m M(i, m) in[t with its index along `ax` set to m], i = t's index along
// ax, M row-major N1 x N1 (or its transpose); `along` does it for NF fields of
// NP values each, into out[f][t].
template <int N1, bool TRANSPOSE>
__device__ inline double along_val(const double* M, int ax, int t, const double* in) {
    const int st = ax == 0 ? 1 : ax == 1 ? N1 : N1 * N1;
    const int i = (t / st) % N1;
    const int t0 = t - i * st;
    double s = 0;
#pragma unroll
    for (int m = 0; m < N1; ++m) s = fma(TRANSPOSE ? M[m * N1 + i] : M[i * N1 + m], in[t0 + m * st], s);
    return s;
}

template <int N1, int NP, int NF, bool TRANSPOSE>
__device__ inline void along(const double* M, int ax, int t, const double* in, double* out) {
#pragma unroll
    for (int f = 0; f < NF; ++f) out[f * NP + t] = along_val<N1, TRANSPOSE>(M, ax, t, in + f * NP);
}

// Per (element, face): the neighbour (or -1) and packed data: bits 0-2 the
// neighbour's local face, bits 3-5 the map of this element's face point
// indices onto the neighbour's (bit 3: swap the two face coordinates first,
// bits 4/5: reverse the first / second), bit 6: this element is the face's
// left element.
__host__ __device__ __forceinline__ void partner_point(int code, int ka, int kb, int n1, int& pa, int& pb) {
    pa = (code & 1) ? kb : ka;
    pb = (code & 1) ? ka : kb;
    if (code & 2) pa = n1 - 1 - pa;
    if (code & 4) pb = n1 - 1 - pb;
}

struct GenParams {
    int64_t n_elem;
    int64_t first, end;    // the elements of this launch
    StageIO io;
    const int32_t* nbr;    // [NFACE][E]
    const int32_t* info;   // [NFACE][E]
    const double* tab;     // NodalOps of the order, packed
    const double* geo;     // per point, GenRhs::GP numbers [E][GP][NP] (where those
    const double* fgeo;    // of element 0 would be); per face point, GF [E][NFACE][GF][NFP]
    const double* cinv;    // [E] (acoustic)
};

// One thread per point. Threads of a workgroup: the smallest of 64, 128 and
// 256 that whole elements fill to 15/16, or as many elements as 256 hold.
template <int DIM, int N1, bool ACOUSTIC>
struct GenRhs {
    using S = GenShape<DIM, N1>;
    static constexpr int kDim = DIM, kN1 = N1;
    static constexpr bool kAcoustic = ACOUSTIC;
    static constexpr int NF = ACOUSTIC ? DIM + 1 : 1;
    static constexpr int NP = S::NP, NFP = S::NFP, NFACE = S::NFACE;
    static constexpr int EPB = (64 % NP) * 16 <= 64 ? 64 / NP : (128 % NP) * 16 <= 128 ? 128 / NP : 256 / NP;
    static constexpr int THREADS = EPB * NP;
    // stored geometry. Per point: acoustic J^{-1} and 1/W; advection W ahat_r
    // and 1/W (W the point's weight times |det J|). Per face point: acoustic
    // the own outward normal times the face's weight and area element;
    // advection the two factors of the own and the neighbour's trace in the
    // flux, upwinding included.
    static constexpr int GP = (ACOUSTIC ? DIM * DIM : DIM) + 1;
    static constexpr int GF = ACOUSTIC ? DIM : 2;
    // face values of all fields per element, and how many a thread loads
    static constexpr int NI = NFACE * NF * NFP;
    static constexpr int KI = (NI + NP - 1) / NP;
    static constexpr int KF = (NFACE * NFP + NP - 1) / NP;  // face points per thread
    // LDS per element, in doubles: two work arrays, the advection fluxes, the
    // neighbours' face coefficients, and (3D) those with the first face
    // coordinate at points; the face integrands overlay the coefficients in 3D
    static constexpr int A = 0, B = NF * NP, F = 2 * NF * NP, NBC = F + (ACOUSTIC ? 0 : DIM * NP), NBT = NBC + NI,
                         PER = NBT + NI;
    static constexpr int FC = DIM == 3 ? NBC : NBT;
};

// The geometry a mesh and an operator fix, once per operator (or slab by slab
// before each use, tensor_general_in_slabs): thread t of element e takes point t
// and the face points t, t + NP, ..
struct GenGeoParams {
    int64_t n_elem;
    int64_t first, count;
    const double* X;       // [E][NV][DIM] vertex coordinates
    const int32_t* nbr;
    const int32_t* info;
    const double* tab;
    double a[3];           // advection velocity
    double* geo;
    double* fgeo;
};

template <int DIM, int N1, bool ACOUSTIC>
__global__ __launch_bounds__(kGenTarget) void tensor_general_geometry(const GenGeoParams p) {
    using G = GenRhs<DIM, N1, ACOUSTIC>;
    using T = NodalTab<N1>;
    constexpr int NP = G::NP, NFP = G::NFP, NV = G::S::NV, NFACE = G::NFACE;
    const int t = threadIdx.x % NP;
    const int64_t at = int64_t(blockIdx.x) * G::EPB + threadIdx.x / NP, e = p.first + at;
    if (at >= p.count) return;
    const double* tab = p.tab;
    const double* X = p.X + e * NV * DIM;
    const int ii[3] = {t % N1, (t / N1) % N1, DIM == 3 ? t / (N1 * N1) : 0};
    double xi[DIM], J[DIM][DIM], Ji[DIM][DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xi[d] = tab[T::X + ii[d]];
    multilinear<DIM>(X, xi, J, nullptr);
    double W = fabs(det_inv<DIM>(J, Ji));
#pragma unroll
    for (int d = 0; d < DIM; ++d) W *= tab[T::W + ii[d]];
    double* geo = p.geo + at * G::GP * NP + t;
#pragma unroll
    for (int r = 0; r < DIM; ++r) {
        double ah = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            if constexpr (ACOUSTIC) geo[(r * DIM + d) * NP] = Ji[r][d];
            else ah += Ji[r][d] * p.a[d];
        }
        if constexpr (!ACOUSTIC) geo[r * NP] = W * ah;
    }
    geo[(G::GP - 1) * NP] = 1.0 / W;
    for (int it = t; it < NFACE * NFP; it += NP) {
        const int f = it / NFP, k = it % NFP;
        const int ka = k % N1, kb = DIM == 3 ? k / N1 : 0;
        const int32_t nb = p.nbr[f * p.n_elem + e];
        const int32_t info = p.info[f * p.n_elem + e];
        const bool inner = nb >= 0;
        const bool left = !inner || ((info >> 6) & 1);
        // the left element's normal and area element at its point
        int qa = ka, qb = kb;
        if (!left) partner_point((info >> 3) & 7, ka, kb, N1, qa, qb);
        double n[DIM];
        face_normal<DIM, N1>(left ? X : p.X + int64_t(nb) * NV * DIM, left ? f : (info & 7), qa, qb, tab, n);
        double area = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) area += n[d] * n[d];
        area = sqrt(area);
        double wf = tab[T::W + qa];
        if constexpr (DIM == 3) wf *= tab[T::W + qb];
        const double sgn = left ? 1.0 : -1.0;  // own normal = sgn n
        double* out = p.fgeo + ((at * NFACE + f) * G::GF) * NFP + k;
        if constexpr (ACOUSTIC) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) out[d * NFP] = sgn * n[d] * wf;
        } else {
            double An = 0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) An += p.a[d] * (n[d] / area);
            // the trace of the flux: left, right (none on a boundary), or half of each
            double cl = 0, cr = 0;
            if (An > 1e-12) cl = 1;
            else if (An < -1e-12) cr = 1;
            else if (fabs(An) < 1e-12) cl = cr = 0.5;
            const double flux = -(An * sgn) * (wf * area);
            out[0] = flux * (left ? cl : cr);
            out[NFP] = inner ? flux * (left ? cr : cl) : 0.0;
        }
    }
}

// Bound by the LDS reads and barriers of its one-dimensional contractions:
// every operand but a row of the matrix comes from LDS. The geometry comes
// from memory (3.5 KB an element at p = 2 in 3D, where a vector has 0.9): formed
// from the vertices at every point and face point of every launch, it took 256
// registers, a third of the LDS for the vertices and most of the time (FP64
// acoustic, 22x18x20 p = 2: 114 us then, 24 now; 14x12x13 p = 3 70 and 14;
// advection 22x18x20 p = 2 31.5 and 8.1). A face's traces at its points cost
// N1 products each: the own one from the point values, the neighbour's one
// face coordinate after the other. form_here on the volume sums takes the
// acoustic p = 2 kernel from 208 to 108 registers.
template <int DIM, int N1, bool ACOUSTIC>
__global__ __launch_bounds__((GenRhs<DIM, N1, ACOUSTIC>::THREADS)) void tensor_general_rhs(const GenParams p) {
    using G = GenRhs<DIM, N1, ACOUSTIC>;
    using T = NodalTab<N1>;
    constexpr int NP = G::NP, NFP = G::NFP, NFACE = G::NFACE, NF = G::NF;
    __shared__ double lds[G::EPB * G::PER];
    __shared__ double tab[T::SIZE];
    const int tid = threadIdx.x;
    const int le = tid / NP;
    const int t = tid % NP;
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t e = p.first + blk * G::EPB + le;
    const bool ok = e < p.end;
    const int64_t E = p.n_elem;
    double* sA = lds + le * G::PER + G::A;
    double* sB = lds + le * G::PER + G::B;
    double* snb = lds + le * G::PER + G::NBC;
    double* sc = lds + le * G::PER + G::FC;
    for (int k = tid; k < T::SIZE; k += G::THREADS) tab[k] = p.tab[k];

    // ---- stage input, neighbours' face coefficients, geometry
    const int64_t base = e * NF * NP;
    double gp[G::GP], gf[G::KF][G::GF];
    int32_t fnb[G::KF], finfo[G::KF];
    if (ok) {
        int64_t at[G::KI];
#pragma unroll
        for (int i = 0; i < G::KI; ++i) {
            const int it = t + i * NP < G::NI ? t + i * NP : 0;
            const int f = it / (NF * NFP), r = it % (NF * NFP), fld = r / NFP, k = r % NFP;
            const int32_t nb = p.nbr[f * E + e];
            const int fn = p.info[f * E + e] & 7;
            int idx = face_side(DIM, fn) * ipow(N1, face_axis(DIM, fn)) +
                      (k % N1) * ipow(N1, face_coord_axis(DIM, fn, 0));
            if constexpr (DIM == 3) idx += (k / N1) * ipow(N1, face_coord_axis(DIM, fn, 1));
            at[i] = (nb >= 0 ? int64_t(nb) * NF * NP : base) + fld * NP + idx;
        }
        int64_t own[NF];
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) own[fld] = base + fld * NP + t;
        double u[NF], v[G::KI];
        combine_n<NF>(p.io, own, u);
        combine_n<G::KI>(p.io, at, v);
#pragma unroll
        for (int c = 0; c < G::GP; ++c) gp[c] = p.geo[(e * G::GP + c) * NP + t];
#pragma unroll
        for (int i = 0; i < G::KF; ++i) {
            const int it = t + i * NP < NFACE * NFP ? t + i * NP : 0;
            const int f = it / NFP;
            fnb[i] = p.nbr[f * E + e];
            finfo[i] = p.info[f * E + e];
#pragma unroll
            for (int c = 0; c < G::GF; ++c)
                gf[i][c] = p.fgeo[((e * NFACE + f) * G::GF + c) * NFP + it % NFP];
        }
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) sA[fld * NP + t] = u[fld];
#pragma unroll
        for (int i = 0; i < G::KI; ++i)
            if (t + i * NP < G::NI) snb[t + i * NP] = v[i];
    }
    __syncthreads();

    // ---- point values U = B u, one direction after the other; the first face
    // coordinate of the neighbours' traces with the first of them
    along<N1, NP, NF, false>(tab + T::B, 0, t, sA, sB);
    if constexpr (DIM == 3) {
        double* st = lds + le * G::PER + G::NBT;
#pragma unroll
        for (int i = 0; i < G::KI; ++i) {
            const int it = t + i * NP;
            if (it < G::NI) {
                const int q = it % N1, row = it - q;
                double s = 0;
#pragma unroll
                for (int a = 0; a < N1; ++a) s = fma(tab[T::B + q * N1 + a], snb[row + a], s);
                st[it] = s;
            }
        }
    }
    __syncthreads();
    along<N1, NP, NF, false>(tab + T::B, 1, t, sB, sA);
    __syncthreads();
    const double* Up = sA;
    if constexpr (DIM == 3) {
        along<N1, NP, NF, false>(tab + T::B, 2, t, sA, sB);
        __syncthreads();
        Up = sB;
    }

    // ---- volume terms at the point
    double res[NF];
    if constexpr (!ACOUSTIC) {
        double* sF = lds + le * G::PER + G::F;
        const double u = Up[t];
#pragma unroll
        for (int r = 0; r < DIM; ++r) sF[r * NP + t] = gp[r] * u;
    } else {
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) res[fld] = 0.0;
#pragma unroll
        for (int r = 0; r < DIM; ++r) {
            const double gv = along_val<N1, false>(tab + T::C, r, t, Up);
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const double Jrd = gp[r * DIM + d];
                res[1 + d] = fma(Jrd, gv, res[1 + d]);
                res[0] = fma(Jrd, along_val<N1, false>(tab + T::C, r, t, Up + (1 + d) * NP), res[0]);
            }
        }
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) form_here(res[fld]);
    }

    // ---- face integrands at the face points
    if (ok) {
#pragma unroll
        for (int i = 0; i < G::KF; ++i) {
            const int it = t + i * NP;
            if (it >= NFACE * NFP) continue;
            const int f = it / NFP, k = it % NFP;
            const int ka = k % N1, kb = DIM == 3 ? k / N1 : 0;
            const int ax = face_axis(DIM, f), a0 = face_coord_axis(DIM, f, 0);
            const int stf = ax == 0 ? 1 : ax == 1 ? N1 : N1 * N1;
            const int st0 = a0 == 0 ? 1 : N1;  // the first face coordinate is x or y,
            const int st1 = face_coord_axis(DIM, f, 1) == 1 ? N1 : N1 * N1;  // the second y or z
            const double* lam = tab + (face_side(DIM, f) ? T::LAM1 : T::LAM0);
            const double* uf = Up + ka * st0 + (DIM == 3 ? kb * st1 : 0);
            const bool inner = fnb[i] >= 0;
            int pa = ka, pb = kb;
            if (inner) partner_point((finfo[i] >> 3) & 7, ka, kb, N1, pa, pb);
            double own[NF], nbv[NF];
#pragma unroll
            for (int fld = 0; fld < NF; ++fld) {
                double s = 0, q = 0;
#pragma unroll
                for (int m = 0; m < N1; ++m) {
                    s = fma(lam[m], uf[fld * NP + m * stf], s);
                    const double* nf = lds + le * G::PER + (DIM == 3 ? G::NBT : G::NBC) + (f * NF + fld) * NFP;
                    q = DIM == 3 ? fma(tab[T::B + pb * N1 + m], nf[pa + N1 * m], q)
                                 : fma(tab[T::B + pa * N1 + m], nf[m], q);
                }
                own[fld] = s;
                nbv[fld] = q;
            }
            double* out = sc + f * NF * NFP + k;
            if constexpr (!ACOUSTIC) {
                // a trace the flux does not take is left out, not multiplied by
                // its factor of zero: it may be infinite or not a number
                const double fn = inner && gf[i][1] != 0.0 ? gf[i][1] * nbv[0] : 0.0;
                out[0] = gf[i][0] != 0.0 ? fma(gf[i][0], own[0], fn) : fn;
            } else {
                // -1/2 n.(s_own - s_nbr) and -1/2 n (v_own - v_nbr), n the own
                // normal; -n.s_own and nothing on a wall
                double jn = 0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) jn = fma(gf[i][d], inner ? own[1 + d] - nbv[1 + d] : own[1 + d], jn);
                out[0] = inner ? -0.5 * jn : -jn;
                const double jv = inner ? -0.5 * (own[0] - nbv[0]) : 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) out[(1 + d) * NFP] = inner ? gf[i][d] * jv : 0.0;
            }
        }
    }
    __syncthreads();

    // ---- lift the face integrands to the points, divide by the point weight
    const int ii[3] = {t % N1, (t / N1) % N1, DIM == 3 ? t / (N1 * N1) : 0};
    const double wi = gp[G::GP - 1];
    const double ci = ACOUSTIC && ok ? 1.0 / p.cinv[e] : 1.0;
    double lift[NF];
#pragma unroll
    for (int fld = 0; fld < NF; ++fld) lift[fld] = 0.0;
#pragma unroll
    for (int f = 0; f < NFACE; ++f) {
        const int a0 = face_coord_axis(DIM, f, 0), a1 = DIM == 3 ? face_coord_axis(DIM, f, 1) : 0;
        const int k = ii[a0] + (DIM == 3 ? N1 * ii[a1] : 0);
        const double lam = tab[(face_side(DIM, f) ? T::LAM1 : T::LAM0) + ii[face_axis(DIM, f)]];
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) lift[fld] = fma(lam, sc[(f * NF + fld) * NFP + k], lift[fld]);
    }
    if constexpr (!ACOUSTIC) {
        const double* sF = lds + le * G::PER + G::F;
        double v = lift[0];
#pragma unroll
        for (int r = 0; r < DIM; ++r) v += along_val<N1, true>(tab + T::C, r, t, sF + r * NP);
        sA[t] = v * wi;
    } else {
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) sA[fld * NP + t] = fma(lift[fld], wi, res[fld]) * (fld > 0 ? ci : 1.0);
    }
    __syncthreads();

    // ---- back to coefficients: k = B^{-1} (point values)
    along<N1, NP, NF, false>(tab + T::BINV, 0, t, sA, sB);
    __syncthreads();
    const double* Kp = sB;
    if constexpr (DIM == 3) {
        along<N1, NP, NF, false>(tab + T::BINV, 1, t, sB, sA);
        __syncthreads();
        Kp = sA;
    }
    if (ok) {
        double kept[NF];  // the values as stored
#pragma unroll
        for (int fld = 0; fld < NF; ++fld) {
            const double v = along_val<N1, false>(tab + T::BINV, DIM - 1, t, Kp + fld * NP);
            if (p.io.out_f32) {
                const float vf = float(v);
                static_cast<float*>(p.io.out)[base + fld * NP + t] = vf;
                kept[fld] = double(vf);
            } else {
                static_cast<double*>(p.io.out)[base + fld * NP + t] = v;
                kept[fld] = v;
            }
        }
        if (p.io.upd.u != nullptr) {  // the RK update fused into a step's last stage (StageIO::upd)
#pragma unroll
            for (int fld = 0; fld < NF; ++fld) {
                const double own[1] = {kept[fld]};
                rk_update_run<1>(p.io.upd, base + fld * NP + t, own);
            }
        }
    }
}

// v = M v or M^{-1} v in place (FP64), M = B^T W B per element and field
// (c_inv W on the acoustic s-fields).
struct GenMassParams {
    int64_t n_elem;
    int32_t nf, inverse;
    double* v;
    const double* X;
    const double* tab;
    const double* cinv;  // NULL: advection
};

template <int DIM, int N1>
__global__ __launch_bounds__(kGenTarget) void tensor_general_mass(const GenMassParams p) {
    using S = GenShape<DIM, N1>;
    using T = NodalTab<N1>;
    constexpr int NP = S::NP, NV = S::NV;
    __shared__ double sXs[S::EPB][NV * DIM];
    __shared__ double sbuf[S::EPB][2][NP];
    __shared__ double tab[T::SIZE];
    const int tid = threadIdx.x, le = tid / NP, t = tid % NP;
    const int64_t e = int64_t(blockIdx.x) * S::EPB + le;
    const bool ok = e < p.n_elem;
    for (int k = tid; k < T::SIZE; k += blockDim.x) tab[k] = p.tab[k];
    if (ok)
        for (int k = t; k < NV * DIM; k += NP) sXs[le][k] = p.X[e * NV * DIM + k];
    __syncthreads();
    const int ii[3] = {t % N1, (t / N1) % N1, DIM == 3 ? t / (N1 * N1) : 0};
    double Wq;
    {
        double xi[DIM], J[DIM][DIM], Ji[DIM][DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xi[d] = tab[T::X + ii[d]];
        multilinear<DIM>(sXs[le], xi, J, nullptr);
        Wq = fabs(det_inv<DIM>(J, Ji));
#pragma unroll
        for (int d = 0; d < DIM; ++d) Wq *= tab[T::W + ii[d]];
    }
    double* b0 = sbuf[le][0];
    double* b1 = sbuf[le][1];
    for (int fld = 0; fld < p.nf; ++fld) {
        const int64_t o = (e * p.nf + fld) * NP + t;
        const double scale = (p.cinv && fld > 0 && ok) ? p.cinv[e] : 1.0;
        b0[t] = ok ? p.v[o] : 0.0;
        __syncthreads();
        // M: B^T (W (B x)); M^{-1}: B^{-1} (W^{-1} (B^{-T} x))
        const double* M1 = tab + (p.inverse ? T::BINV : T::B);
        double* src = b0;
        double* dst = b1;
#pragma unroll
        for (int ax = 0; ax < DIM; ++ax) {
            if (p.inverse) along<N1, NP, 1, true>(M1, ax, t, src, dst);
            else along<N1, NP, 1, false>(M1, ax, t, src, dst);
            __syncthreads();
            double* tmp = src;
            src = dst;
            dst = tmp;
        }
        src[t] = p.inverse ? src[t] / (Wq * scale) : src[t] * (Wq * scale);
        __syncthreads();
#pragma unroll
        for (int ax = 0; ax < DIM; ++ax) {
            if (p.inverse) along<N1, NP, 1, false>(M1, ax, t, src, dst);
            else along<N1, NP, 1, true>(M1, ax, t, src, dst);
            __syncthreads();
            double* tmp = src;
            src = dst;
            dst = tmp;
        }
        if (ok) p.v[o] = src[t];
        __syncthreads();
    }
}

// L2 projection of sine modes or a Gaussian pulse with the element rule (order
// 2p+1): M^{-1} int f phi = B^{-1} (f at the points).
struct GenProjParams {
    int64_t n_elem;
    int32_t nf, field;
    void* out;
    int32_t out_f32;
    int32_t n_modes;
    const double* modes;  // [n_modes][4]: amp, k
    int32_t gaussian;
    double g[5];          // centre, width, amplitude
    const double* X;
    const double* tab;
};

__device__ inline double source_value(const GenProjParams& p, const double* x, int dim) {
    if (p.gaussian) {
        double r2 = 0;
        for (int d = 0; d < dim; ++d) r2 += (x[d] - p.g[d]) * (x[d] - p.g[d]);
        return p.g[4] * exp(-r2 / (p.g[3] * p.g[3]));
    }
    double v = 0;
    for (int m = 0; m < p.n_modes; ++m) {
        double arg = 0;
        for (int d = 0; d < dim; ++d) arg += p.modes[4 * m + 1 + d] * x[d];
        v += p.modes[4 * m] * sin(2 * M_PI * arg);
    }
    return v;
}

template <int DIM, int N1>
__global__ __launch_bounds__(kGenTarget) void tensor_general_project(const GenProjParams p) {
    using S = GenShape<DIM, N1>;
    using T = NodalTab<N1>;
    constexpr int NP = S::NP, NV = S::NV;
    __shared__ double sXs[S::EPB][NV * DIM];
    __shared__ double sbuf[S::EPB][2][NP];
    __shared__ double tab[T::SIZE];
    const int tid = threadIdx.x, le = tid / NP, t = tid % NP;
    const int64_t e = int64_t(blockIdx.x) * S::EPB + le;
    const bool ok = e < p.n_elem;
    for (int k = tid; k < T::SIZE; k += blockDim.x) tab[k] = p.tab[k];
    if (ok)
        for (int k = t; k < NV * DIM; k += NP) sXs[le][k] = p.X[e * NV * DIM + k];
    __syncthreads();
    const int ii[3] = {t % N1, (t / N1) % N1, DIM == 3 ? t / (N1 * N1) : 0};
    double xi[DIM], J[DIM][DIM], x[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) xi[d] = tab[T::X + ii[d]];
    multilinear<DIM>(sXs[le], xi, J, x);
    sbuf[le][0][t] = ok ? source_value(p, x, DIM) : 0.0;
    __syncthreads();
    double* src = sbuf[le][0];
    double* dst = sbuf[le][1];
#pragma unroll
    for (int ax = 0; ax < DIM; ++ax) {
        along<N1, NP, 1, false>(tab + T::BINV, ax, t, src, dst);
        __syncthreads();
        double* tmp = src;
        src = dst;
        dst = tmp;
    }
    if (!ok) return;
    for (int fld = 0; fld < p.nf; ++fld) {
        if (p.field >= 0 && fld != p.field) continue;
        const int64_t o = (e * p.nf + fld) * NP + t;
        if (p.out_f32) static_cast<float*>(p.out)[o] = float(src[t]);
        else static_cast<double*>(p.out)[o] = src[t];
    }
}

// computeTotalError (rule 2p+2, HpgemAPISimplified_Impl.h:339-401) and
// computeMaxError (the element rule, :403-530) against shifted sine modes,
// or the mass-weighted L2 of a difference x - y (modes = 0, y set): one
// thread per element, per-block partial sums [blocks][2] (sum, max).
struct GenNormParams {
    int64_t n_elem;
    int32_t nf, field;
    const void* u;
    int32_t u_f32;
    const void* y;        // difference mode: the vector subtracted
    int32_t y_f32;
    int32_t n_modes;
    const double* modes;
    double shift[3];
    const double* X;
    const double* tab;
    double* partial;
};

template <int DIM, int N1>
__global__ __launch_bounds__(kBlock) void tensor_general_norm(const GenNormParams p) {
    using S = GenShape<DIM, N1>;
    using T = NodalTab<N1>;
    constexpr int NP = S::NP, NV = S::NV;
    __shared__ double s_red[2][kBlock];
    const int64_t e = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    double sum = 0, mx = 0;
    auto coef = [&](const void* v, int32_t f32, int64_t i) {
        return f32 ? double(static_cast<const float*>(v)[i]) : static_cast<const double*>(v)[i];
    };
    if (e < p.n_elem) {
        const double* X = p.X + e * NV * DIM;
        for (int fld = 0; fld < p.nf; ++fld) {
            if (p.field >= 0 && fld != p.field) continue;
            const int64_t base = (e * p.nf + fld) * NP;
            if (p.y) {
                for (int i = 0; i < NP; ++i)
                    mx = fmax(mx, fabs(coef(p.u, p.u_f32, base + i) - coef(p.y, p.y_f32, base + i)));
            }
            // pass 0: the L2 integral (difference: the element rule, so that it
            // is x^T M x; modes: rule 2p+2); pass 1: max error at the element rule's points
            for (int pass = 0; pass < (p.y ? 1 : 2); ++pass) {
                const bool l2rule = pass == 0 && !p.y;
                const int NQ = l2rule ? N1 + 1 : N1;
                const double* xq = p.tab + (l2rule ? T::X2 : T::X);
                const double* wq = p.tab + (l2rule ? T::W2 : T::W);
                const int nz = DIM == 3 ? NQ : 1;
                for (int qz = 0; qz < nz; ++qz)
                    for (int qy = 0; qy < NQ; ++qy)
                        for (int qx = 0; qx < NQ; ++qx) {
                            const int q[3] = {qx, qy, qz};
                            auto psi = [&](int a, int qq) {
                                return l2rule ? p.tab[T::B2 + a * (N1 + 1) + qq] : p.tab[T::B + qq * N1 + a];
                            };
                            double val = 0;
                            for (int c = 0; c < (DIM == 3 ? N1 : 1); ++c) {
                                double vy = 0;
                                for (int b = 0; b < N1; ++b) {
                                    double vx = 0;
                                    for (int a = 0; a < N1; ++a) {
                                        const int64_t i = base + a + N1 * (b + N1 * c);
                                        double cf = coef(p.u, p.u_f32, i);
                                        if (p.y) cf -= coef(p.y, p.y_f32, i);
                                        vx += cf * psi(a, qx);
                                    }
                                    vy += vx * psi(b, qy);
                                }
                                val += DIM == 3 ? vy * psi(c, qz) : vy;
                            }
                            double xi[DIM], J[DIM][DIM], Ji[DIM][DIM], x[DIM];
                            for (int d = 0; d < DIM; ++d) xi[d] = xq[q[d]];
                            multilinear<DIM>(X, xi, J, x);
                            double err = val;
                            if (!p.y) {
                                double ex = 0;
                                for (int m = 0; m < p.n_modes; ++m) {
                                    double arg = 0;
                                    for (int d = 0; d < DIM; ++d) arg += p.modes[4 * m + 1 + d] * (x[d] - p.shift[d]);
                                    ex += p.modes[4 * m] * sin(2 * M_PI * arg);
                                }
                                err = ex - val;
                            }
                            if (pass == 0) {
                                double w = fabs(det_inv<DIM>(J, Ji));
                                for (int d = 0; d < DIM; ++d) w *= wq[q[d]];
                                sum += w * err * err;
                            } else {
                                mx = fmax(mx, fabs(err));
                            }
                        }
            }
        }
    }
    s_red[0][threadIdx.x] = sum;
    s_red[1][threadIdx.x] = mx;
    __syncthreads();
    for (int h = kBlock / 2; h > 0; h /= 2) {
        if (int(threadIdx.x) < h) {
            s_red[0][threadIdx.x] += s_red[0][threadIdx.x + h];
            s_red[1][threadIdx.x] = fmax(s_red[1][threadIdx.x], s_red[1][threadIdx.x + h]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        p.partial[2 * blockIdx.x] = s_red[0][0];
        p.partial[2 * blockIdx.x + 1] = s_red[1][0];
    }
}

template <typename F>
void dispatch_general(int dim, int n1, F&& f) {
    auto go = [&](auto D) {
        constexpr int DIMc = decltype(D)::value;
        switch (n1) {
            case 2: f(D, std::integral_constant<int, 2>{}); return;
            case 3: f(D, std::integral_constant<int, 3>{}); return;
            case 4: f(D, std::integral_constant<int, 4>{}); return;
            case 5: f(D, std::integral_constant<int, 5>{}); return;
            case 6: f(D, std::integral_constant<int, 6>{}); return;
        }
        (void)DIMc;
        throw Failure(HGDG_ERR_UNSUPPORTED, "no general tensor kernel for this order");
    };
    if (dim == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 3>{});
}

// Face orientation as hpGEM pairs the face points: the map of the left
// element's face coordinates onto the right element's is the square symmetry
// that sends the left face's corners onto the right face's corners with the
// same node ids, except that for the two quarter turns hpGEM's index lookup
// (ReferenceSquare::getCodim0MappingIndex) selects the opposite quarter turn
// (MappingToRefSquareToSquare1/3): the map actually applied is the inverse of
// the corner map. Returned as the index code of partner_point (swap, reverse
// first, reverse second).
int left_to_right_code(int dim, const int64_t* lnodes, const int64_t* rnodes) {
    if (dim == 2) return lnodes[0] == rnodes[0] ? 0 : 2;  // a line: identity or reversed
    // corner k of a face has face coordinates (2 (k & 1) - 1, 2 (k >> 1) - 1)
    for (int code = 0; code < 8; ++code) {
        bool all = true;
        for (int k = 0; k < 4 && all; ++k) {
            int pa, pb;
            partner_point(code, k & 1, k >> 1, 2, pa, pb);
            all = lnodes[k] == rnodes[pa + 2 * pb];
        }
        if (!all) continue;
        const bool swap = code & 1, ra = code & 2, rb = code & 4;
        if (swap && ra != rb) return 1 | (ra ? 4 : 0) | (rb ? 2 : 0);  // quarter turn: the opposite one
        return code;
    }
    throw Failure(HGDG_ERR_ARG, "a shared face whose corners do not match");
}

// Inverse of a partner_point code (maps the right element's face point indices back).
int inverse_code(int code) {
    if (!(code & 1)) return code;
    return 1 | ((code & 2) ? 4 : 0) | ((code & 4) ? 2 : 0);
}

}  // namespace

void tensor_general_upload(hgdg_ctx* c, const hgdg_mesh_desc* m) {
    const int dim = shape_dim(m->shape);
    const int64_t ne = m->n_elements;
    const int nv = 1 << dim, nfaces = 2 * dim, fverts = 1 << (dim - 1);
    TensorMesh& tm = c->tm;
    tm.general = true;
    tm.structured = false;
    tm.gX.assign(m->coords, m->coords + size_t(ne) * nv * dim);
    tm.gnbr.assign(size_t(nfaces) * ne, -1);
    tm.ginfo.assign(size_t(nfaces) * ne, 0);
    // every element must map with a nonzero Jacobian determinant at its points
    // (checked at the element rule's points on the host)
    const NodalOps ops = nodal_ops(tm.p);
    for (int64_t e = 0; e < ne; ++e) {
        const double* X = m->coords + size_t(e) * nv * dim;
        const int npts = dim == 3 ? tm.n1 * tm.n1 * tm.n1 : tm.n1 * tm.n1;
        for (int q = 0; q < npts; ++q) {
            const int ii[3] = {q % tm.n1, (q / tm.n1) % tm.n1, q / (tm.n1 * tm.n1)};
            double J[3][3] = {{0}};
            for (int v = 0; v < nv; ++v)
                for (int d = 0; d < dim; ++d) {
                    double dd = ((v >> d) & 1) ? 0.5 : -0.5;
                    for (int k = 0; k < dim; ++k)
                        if (k != d) dd *= ((v >> k) & 1) ? 0.5 * (1 + ops.x[ii[k]]) : 0.5 * (1 - ops.x[ii[k]]);
                    for (int r = 0; r < dim; ++r) J[r][d] += X[v * dim + r] * dd;
                }
            const double det = dim == 2 ? J[0][0] * J[1][1] - J[0][1] * J[1][0]
                                        : J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                                              J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                                              J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
            require(det != 0.0 && std::isfinite(det), HGDG_ERR_ARG, "degenerate element " + std::to_string(e));
        }
    }
    // faces: hpGEM's face search visits elements in order, so the first
    // element to reach a face is its left element; a face's node list follows
    // the face's corner order (corner k: bit 0 of k along the first face
    // coordinate, bit 1 along the second)
    auto face_node = [&](int64_t e, int f, int k) {
        const int ax = face_axis(dim, f);
        int v = face_side(dim, f) << ax;
        v |= (k & 1) << face_coord_axis(dim, f, 0);
        if (dim == 3) v |= ((k >> 1) & 1) << face_coord_axis(dim, f, 1);
        return m->node_ids[size_t(e) * nv + v];
    };
    std::unordered_map<std::string, std::pair<int64_t, int>> open;
    open.reserve(size_t(ne) * nfaces);
    int64_t n_internal = 0, n_total = 0;
    for (int64_t e = 0; e < ne; ++e) {
        for (int f = 0; f < nfaces; ++f) {
            std::array<int64_t, 4> key{};
            for (int k = 0; k < fverts; ++k) key[k] = face_node(e, f, k);
            std::sort(key.begin(), key.begin() + fverts);
            std::string kstr(reinterpret_cast<const char*>(key.data()), sizeof(int64_t) * fverts);
            auto it = open.find(kstr);
            if (it == open.end()) {
                open.emplace(std::move(kstr), std::make_pair(e, f));
                continue;
            }
            const int64_t l = it->second.first;
            const int fl = it->second.second;
            require(l != e, HGDG_ERR_UNSUPPORTED, "element " + std::to_string(e) + " meets itself across a face");
            require(tm.gnbr[size_t(fl) * ne + l] < 0, HGDG_ERR_ARG, "a face is bounded by more than two elements");
            int64_t ln[4], rn[4];
            for (int k = 0; k < fverts; ++k) {
                ln[k] = face_node(l, fl, k);
                rn[k] = face_node(e, f, k);
            }
            const int code = left_to_right_code(dim, ln, rn);
            tm.gnbr[size_t(fl) * ne + l] = int32_t(e);
            tm.ginfo[size_t(fl) * ne + l] = f | (code << 3) | (1 << 6);
            tm.gnbr[size_t(f) * ne + e] = int32_t(l);
            tm.ginfo[size_t(f) * ne + e] = fl | (inverse_code(code) << 3);
            open.erase(it);
            ++n_internal;
            ++n_total;
        }
    }
    n_total += int64_t(open.size());
    c->n_faces = n_total;
    c->n_internal = n_internal;
    c->n_fields = 1;
    c->dof = ne * tm.nb;
    tm.d_gX.upload(tm.gX, c->stream);
    std::vector<int32_t> fi(tm.gnbr);
    fi.insert(fi.end(), tm.ginfo.begin(), tm.ginfo.end());
    tm.d_gface.upload(fi, c->stream);
    tm.d_gtab.upload(ops.packed(), c->stream);
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

namespace {

constexpr int64_t kGeoSlab = 4096;

// f(GenRhs) of the mesh and an operator of this kind
template <typename F>
void with_shape(const hgdg_ctx* c, int kind, F&& f) {
    dispatch_general(c->dim, c->tm.n1, [&](auto D, auto N) {
        if (kind == HGDG_OP_ACOUSTIC_CENTRAL) f(GenRhs<decltype(D)::value, decltype(N)::value, true>{});
        else f(GenRhs<decltype(D)::value, decltype(N)::value, false>{});
    });
}

void alloc_geometry(hgdg_ctx* c, int kind, int64_t elements) {
    with_shape(c, kind, [&](auto G_) {
        using G = decltype(G_);
        c->tm.d_ggeo.alloc(size_t(elements) * G::GP * G::NP);
        c->tm.d_gfgeo.alloc(size_t(elements) * G::NFACE * G::GF * G::NFP);
    });
}

// The geometry of elements [first, first + count), to the buffers' start.
void launch_geometry(hgdg_ctx* c, int kind, const double* velocity, int64_t first, int64_t count) {
    GenGeoParams p{};
    p.n_elem = c->n_elem;
    p.first = first;
    p.count = count;
    p.X = c->tm.d_gX.ptr;
    p.nbr = c->tm.d_gface.ptr;
    p.info = c->tm.d_gface.ptr + size_t(2 * c->dim) * c->n_elem;
    p.tab = c->tm.d_gtab.ptr;
    for (int d = 0; d < 3; ++d) p.a[d] = kind == HGDG_OP_ADVECTION_UPWIND && d < c->dim ? velocity[d] : 0.0;
    p.geo = c->tm.d_ggeo.ptr;
    p.fgeo = c->tm.d_gfgeo.ptr;
    with_shape(c, kind, [&](auto G_) {
        using G = decltype(G_);
        hipLaunchKernelGGL((tensor_general_geometry<G::kDim, G::kN1, G::kAcoustic>),
                           dim3(unsigned((count + G::EPB - 1) / G::EPB)), dim3(G::THREADS), 0, c->stream, p);
    });
    HGDG_HIP(hipGetLastError());
}

}  // namespace

void tensor_general_operator_set(hgdg_ctx* c, const hgdg_op_desc* op) {
    const int64_t ne = c->n_elem;
    if (op->kind == HGDG_OP_ACOUSTIC_CENTRAL) {
        c->tm.d_gcinv.upload(std::vector<double>(op->c_inv, op->c_inv + ne), c->stream);
        c->n_fields = c->dim + 1;
    } else {
        c->n_fields = 1;
    }
    c->dof = ne * c->tm.nb * c->n_fields;
    c->tm.geo_slab = 0;
    try {
        alloc_geometry(c, op->kind, ne);
    } catch (const Failure&) {
        (void)hipGetLastError();
        c->tm.geo_slab = std::min(ne, kGeoSlab);
        alloc_geometry(c, op->kind, c->tm.geo_slab);
        return;
    }
    launch_geometry(c, op->kind, op->velocity, 0, ne);
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

// Gives the stored geometry back but for `elements` at a time, whose geometry
// each right-hand side forms anew. Of a mesh that nearly fills the card: it takes
// more than a state vector (3D acoustics 3.5 KB an element against 0.9 at p = 2,
// 22 against 6.9 at p = 5).
void tensor_general_in_slabs(hgdg_ctx* c, int64_t elements) {
    HGDG_HIP(hipStreamSynchronize(c->stream));
    c->drop_graph();
    c->tm.d_ggeo.reset();
    c->tm.d_gfgeo.reset();
    c->tm.geo_slab = std::min(c->n_elem, elements > 0 ? elements : kGeoSlab);
    alloc_geometry(c, c->op.kind, c->tm.geo_slab);
}

void tensor_general_rhs(hgdg_ctx* c, const StageIO& io) {
    GenParams p{};
    p.n_elem = c->n_elem;
    p.io = io;
    p.nbr = c->tm.d_gface.ptr;
    p.info = c->tm.d_gface.ptr + size_t(2 * c->dim) * c->n_elem;
    p.tab = c->tm.d_gtab.ptr;
    const bool acoustic = c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL;
    p.cinv = acoustic ? c->tm.d_gcinv.ptr : nullptr;
    const int64_t slab = c->tm.geo_slab > 0 ? c->tm.geo_slab : c->n_elem;
    for (p.first = 0; p.first < c->n_elem; p.first += slab) {
        p.end = std::min(p.first + slab, c->n_elem);
        if (c->tm.geo_slab > 0) launch_geometry(c, c->op.kind, c->op.velocity, p.first, p.end - p.first);
        with_shape(c, c->op.kind, [&](auto G_) {
            using G = decltype(G_);
            p.geo = c->tm.d_ggeo.ptr - p.first * G::GP * G::NP;
            p.fgeo = c->tm.d_gfgeo.ptr - p.first * G::NFACE * G::GF * G::NFP;
            hipLaunchKernelGGL((tensor_general_rhs<G::kDim, G::kN1, G::kAcoustic>),
                               dim3(unsigned((p.end - p.first + G::EPB - 1) / G::EPB)), dim3(G::THREADS), 0, c->stream, p);
        });
        HGDG_HIP(hipGetLastError());
    }
}

void tensor_general_mass_apply(hgdg_ctx* c, Vec& v, bool inverse) {
    require(!v.is_f32, HGDG_ERR_UNSUPPORTED, "mass apply/solve needs a vector stored in FP64");
    GenMassParams p{};
    p.n_elem = c->n_elem;
    p.nf = c->n_fields;
    p.inverse = inverse ? 1 : 0;
    p.v = v.f64->ptr;
    p.X = c->tm.d_gX.ptr;
    p.tab = c->tm.d_gtab.ptr;
    p.cinv = c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL ? c->tm.d_gcinv.ptr : nullptr;
    dispatch_general(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = GenShape<DIMc, N1c>;
        const int64_t grid = (c->n_elem + S::EPB - 1) / S::EPB;
        hipLaunchKernelGGL((tensor_general_mass<DIMc, N1c>), dim3(unsigned(grid)), dim3(S::THREADS), 0, c->stream, p);
    });
    HGDG_HIP(hipGetLastError());
}

void tensor_general_project(hgdg_ctx* c, Vec& v, int field, int n_modes, const double* amp, const double* k,
                            const double* gauss) {
    std::vector<double> modes;
    for (int m = 0; m < n_modes; ++m) {
        modes.push_back(amp[m]);
        for (int d = 0; d < 3; ++d) modes.push_back(k[3 * m + d]);
    }
    modes.push_back(0.0);  // never empty
    DevBuf<double> d_modes;
    d_modes.upload(modes, c->stream);
    GenProjParams p{};
    p.n_elem = c->n_elem;
    p.nf = c->n_fields;
    p.field = field;
    p.out = v.ptr();
    p.out_f32 = v.is_f32;
    p.n_modes = n_modes;
    p.modes = d_modes.ptr;
    if (gauss) {
        p.gaussian = 1;
        for (int q = 0; q < 5; ++q) p.g[q] = gauss[q];
    }
    p.X = c->tm.d_gX.ptr;
    p.tab = c->tm.d_gtab.ptr;
    dispatch_general(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = GenShape<DIMc, N1c>;
        const int64_t grid = (c->n_elem + S::EPB - 1) / S::EPB;
        hipLaunchKernelGGL((tensor_general_project<DIMc, N1c>), dim3(unsigned(grid)), dim3(S::THREADS), 0, c->stream,
                           p);
    });
    HGDG_HIP(hipGetLastError());
    HGDG_HIP(hipStreamSynchronize(c->stream));  // before the temporary modes go
}

namespace {

void general_norm(hgdg_ctx* c, GenNormParams& p, double* l2, double* max_abs) {
    p.n_elem = c->n_elem;
    p.nf = c->n_fields;
    p.X = c->tm.d_gX.ptr;
    p.tab = c->tm.d_gtab.ptr;
    const int64_t grid = (c->n_elem + kBlock - 1) / kBlock;
    if (c->d_partial.n < size_t(2 * grid)) c->d_partial.alloc(size_t(2 * grid));
    p.partial = c->d_partial.ptr;
    dispatch_general(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        hipLaunchKernelGGL((tensor_general_norm<DIMc, N1c>), dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, p);
    });
    HGDG_HIP(hipGetLastError());
    std::vector<double> h(size_t(2 * grid));
    HGDG_HIP(hipMemcpyAsync(h.data(), c->d_partial.ptr, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HGDG_HIP(hipStreamSynchronize(c->stream));
    double s = 0, m = 0;
    for (int64_t i = 0; i < grid; ++i) {
        s += h[2 * i];
        m = std::max(m, h[2 * i + 1]);
    }
    *l2 = std::sqrt(std::max(s, 0.0));
    *max_abs = m;
}

}  // namespace

void tensor_general_error_modes(hgdg_ctx* c, const Vec& v, int field, int n_modes, const double* amp,
                                const double* k, const double* shift, double* l2, double* max_abs) {
    std::vector<double> modes;
    for (int m = 0; m < n_modes; ++m) {
        modes.push_back(amp[m]);
        for (int d = 0; d < 3; ++d) modes.push_back(k[3 * m + d]);
    }
    modes.push_back(0.0);
    DevBuf<double> d_modes;
    d_modes.upload(modes, c->stream);
    GenNormParams p{};
    p.field = field;
    p.u = v.ptr();
    p.u_f32 = v.is_f32;
    p.n_modes = n_modes;
    p.modes = d_modes.ptr;
    for (int d = 0; d < 3; ++d) p.shift[d] = shift ? shift[d] : 0.0;
    general_norm(c, p, l2, max_abs);
}

void tensor_general_state_diff(hgdg_ctx* c, const Vec& x, const Vec& y, double* l2, double* max_abs) {
    GenNormParams p{};
    p.field = -1;
    p.u = x.ptr();
    p.u_f32 = x.is_f32;
    p.y = y.ptr();
    p.y_f32 = y.is_f32;
    general_norm(c, p, l2, max_abs);
}

}  // namespace hgdg
