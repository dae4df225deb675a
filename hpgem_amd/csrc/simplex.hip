// Tetrahedral elements with per-element order p = 1..4 (hp meshes): the
// first-order acoustic wave system of hpGEM's AcousticWaveLinear
// (applications/ExampleMultipleVariableProblem/AcousticWaveLinear_Impl.h:
// 102-283): fields v and s_1..s_3, mass blocks M (v) and c_inv M (s),
//   r_v   = int phi grad.s  - 1/2 int_f phi n_L.(s_L - s_R)   (internal faces)
//   r_s_d = int phi d_d v   - 1/2 int_f phi n_L,d (v_L - v_R)
// and on reflecting walls r_v gets - int_f phi n.s and r_s nothing.
//
// On an affine tetrahedron the inverse-mass apply turns the volume terms into
// exact reference derivative matrices Dr_e (d/dxi_e in P_p) combined with
// J^{-1}, and each face term into a lifting, M_ref^{-1} int_f phi psi_m, of the
// flux's coefficients in the face functions psi_m: the traces of the
// hierarchical element functions that do not vanish on the face. A neighbour's
// traces are the same functions up to order and signs, through hpGEM's
// orientation map (FaceGeometry.h:372-393), so both sides are gathered from the
// stage input itself and one launch does the whole stage: elements are grouped
// by order on the device, each block working on elements of one order.
#include <algorithm>
#include <array>
#include <cmath>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <utility>

#include "context.hpp"

namespace hgdg {

namespace {

// int32 table index: per order (p-1) the offsets of its tables in the table
// array; then, of the order-4 set (whose first functions are those of the
// lower orders), the face functions of each local face (the element functions
// whose trace there does not vanish) and how a neighbour's meet ours.
constexpr int kTixM = 0;       // [nb][nb]: M_ref
constexpr int kTixDrP = 1;     // [3][4 ceil(nb/4) k][16 ceil(nb/16) i]: Dr_r(i, k), zeros outside nb x nb
constexpr int kTixLift = 2;    // [4 f][16 m][16 ceil(nb/16) i]: (M_ref^{-1} int_f phi psi_m)_i, zeros for m = 15
constexpr int kTixStride = 3;
constexpr int kTixCols = 4 * kTixStride;  // [4 f][16 m]: the element function of face function m
// [4 f][4 neighbour's face][6 relative orientation][16 m]: bits 0-5 the
// neighbour's function loaded for m, bits 6-7 its coefficient in ours, bits
// 8-9 the coefficient of the one loaded for 27 - m (0: none, 1: +1, 2: -1)
constexpr int kTixFace = kTixCols + 4 * 16;
constexpr int kTixSize = kTixFace + 4 * 4 * 6 * 16;

// packed per-face info
__host__ __device__ constexpr int info_lf(int v) { return v & 3; }
__host__ __device__ constexpr int info_oown(int v) { return (v >> 2) & 7; }
__host__ __device__ constexpr int info_onbr(int v) { return (v >> 5) & 7; }
__host__ __device__ constexpr int info_pn(int v) { return (v >> 8) & 7; }
// the orientation that maps the neighbour's face coordinates onto ours,
// o_nbr o o_own^{-1} (bits set once the orientation group table is built)
__host__ __device__ constexpr int info_rel(int v) { return (v >> 11) & 7; }
constexpr int info_pack(int lf, int oown, int onbr, int pn) { return lf | (oown << 2) | (onbr << 5) | (pn << 8); }

struct RefTetRule {
    int order, n;
    const double* pts;  // [n][3] on the reference tetrahedron
    const double* w;
};
#include "tet_rules.inc"
}  // namespace

struct SimplexParams {
    StageIO io;
    int64_t n_elem;
    int64_t group_start[5];
    int64_t group_dof[5];
    const double* jinv;       // [9][E]: (J^{-1})_{e,d} at [(3e + d) E + elem]
    const double* cinv;       // [E]
    const uint2* frec;        // [E][4]: the neighbours (simplex_faces)
    const uint8_t* fcode;     // [E][4][16]: their face functions
    const double* tab;
    int32_t tab_dr[4], tab_lift[4];  // per order: offsets in tab
    const int32_t* cols;      // [4 f][16]: the element function of each face function
    const int4* blocks;       // per block: order, first device element, element count, face functions met
};

__host__ __device__ constexpr int simplex_nb(int p) { return (p + 1) * (p + 2) * (p + 3) / 6; }
__host__ __device__ constexpr int simplex_ncol(int p) { return (p + 1) * (p + 2) / 2; }
// Elements per workgroup of the RHS kernel, two candidates per order, for met =
// the face functions the order's elements meet (their own or a neighbour's).
// The first fills a workgroup: one basis function per thread, and LDS for five
// workgroups a CU; the second makes more workgroups, which small meshes need.
// The library times both per order when the operator is set; results do not
// depend on the choice (a column's sums do not depend on its tile). The
// interface names the choices by thread counts per element.
__host__ __device__ constexpr int simplex_tpe(int p) { return p == 1 ? 8 : p == 2 ? 12 : p == 3 ? 32 : simplex_nb(p); }
__host__ __device__ constexpr int simplex_tpe_alt(int p) { return p == 1 ? 16 : p == 2 ? 32 : 64; }
__host__ __device__ constexpr int simplex_tpe_of(int p, int variant) { return variant ? simplex_tpe_alt(p) : simplex_tpe(p); }
__host__ __device__ constexpr int simplex_face_lanes(int met) { return met <= 3 ? 4 : met <= 6 ? 8 : 16; }
constexpr int kSimplexLds = 3968;  // doubles
constexpr int kTile = 8;           // elements per column tile of the matrix cores

template <int P>
struct SimplexShape {
    static constexpr int NB = simplex_nb(P);
    static constexpr int NC = simplex_ncol(P);
    static constexpr int NTM = (NB + 15) / 16;           // row tiles
    static constexpr int KS = (NB + 3) / 4;              // steps of a derivative
    static constexpr int NBP = 16 * NTM, KP = 4 * KS;    // padded tables: [3][KP][NBP] and [4][16][NBP]
    // LDS per element, in doubles: v and g_r ([4][NB]); the face integrands
    // ([4 f][v, s][lanes]); J^{-1} and minus the sum of its rows ([4][3]) and
    // 1/c_inv. The first two strides are odd multiples of four doubles, so that
    // the eight elements of a tile lie in different banks.
    static constexpr int ES = NB % 2 ? 4 * NB : 4 * NB + 4;
    static constexpr int JS = 13;
    static constexpr int fs(int lanes) { return 8 * lanes + 4; }
};

__host__ __device__ constexpr int simplex_elem_lds(int p, int lanes) {
    return 4 * simplex_nb(p) + (simplex_nb(p) % 2 ? 0 : 4) + 8 * lanes + 4 + 13;
}
__host__ __device__ constexpr int simplex_epb(int p, int variant, int met) {
    const int full = kBlock / simplex_nb(p), room = kSimplexLds / simplex_elem_lds(p, simplex_face_lanes(met));
    const int n = full < room ? full : room;
    return variant == 0 ? (n > kTile ? n / 4 * 4 : n) : p == 4 ? 4 : kTile;
}

typedef double mfma_d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mfma_d4 mfma_step(double a, double b, mfma_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One workgroup takes `count` consecutive device elements of order P.
//
// With g_r = sum_d (J^{-1})_{r,d} s_d, and grad lambda_o the gradient of the
// barycentric coordinate of the vertex opposite face f (rows of J^{-1}; for
// vertex 0 minus their sum), sigma_f n_f = -grad lambda_o (n_f the outward
// normal, sigma_f area over volume). The first three local faces are opposite
// vertices 1..3, so both equations share one operator per direction r:
//   k_v   =             sum_r [ Dr_r g_r + L_r A_r ] + L_3 A_3
//   k_s_d = (1/c_inv) sum_r (J^{-1})_{r,d} [ Dr_r v + L_r B_r + L_3 B_3 ]
// with the face integrands (sigma_f times the flux of the v equation, and
// minus / plus half the jump of v) as coefficients of the face functions,
//   A_f = 1/2 grad lambda_o.(s_own - s_nbr),  B_f = 1/2 (v_own - v_nbr)  (f < 3; minus that for f = 3)
// on internal faces and A_f = grad lambda_o.s_own, B_f = 0 on walls.
//
// The face functions of f are the traces of the order-4 element functions
// that do not vanish there (hierarchical: order p has the first (p+1)(p+2)/2
// of them), so an own trace is the element's coefficients of those functions,
// and L_f = M_ref^{-1} int_f phi_i psi_m lifts them. A neighbour's traces in
// our face coordinates are its coefficients of its face's functions, up to
// their order and signs: the vertex, edge and degree-3 face functions of the
// two sides match one to one, and the two degree-4 face functions are
// combinations with coefficients 0, +-1 of the other side's two (checked when
// the table is built). So a face function m needs one of the neighbour's
// functions, of every field, gathered from the stage input itself.
//
// Phases: (1) own stage input as v and g_r to LDS, the neighbours' values in
// registers, one face function per lane; (2) face integrands to LDS; (3) on
// the matrix cores, per row tile and tile of eight elements, four
// accumulators (r = 0..2 and the fourth face) over 16 columns [g_r or A | v
// or B]: A(i, k) from lane i + 16 k, B(k, j) from lane j + 16 k, output q of
// lane l holds D(4 q + l / 16, l % 16). A lane then holds k_v, or the brackets
// of k_s, of its element and rows; (4) k goes back through LDS, so that stores
// and the fused update's reads are in order.
//
// Bound by latency, not by a unit: at 24^3 x 5 elements of order 1..4 a launch
// takes 72 to 78 us in FP64, as the choice of elements per workgroup turns out
// (100.7 before: a launch of 28 us that wrote projected traces of every face, and
// one of 73 that gathered them, with the matrix units for the derivatives of
// orders 3 and 4 alone), 70 to 76 with FP32 stage values (81.1). Of 78 us the
// matrix instructions keep their units busy for 15, LDS takes 15, the issue of
// vector instructions 26; the 125 MB of vectors and geometry take 18 to 23 at a
// copy's rate (165 MB with what is read more than once, 24 to 31).
// Whole orders: 31.8 -> 23.3, 53 -> 39.7, 113 -> 66.2 and 179 -> 102.8 us for
// p = 1..4; 13 x 11 x 9 cells of order 2 (launch-bound, two before) 14.7 ->
// 10.1 us. Arithmetic is FP64 whatever the stage values' type: the matrix units
// are not what bounds this, and it leaves the FP32 path the rounding of its
// stored values as its only error. Five workgroups a CU, at the price of a few spilled
// registers, beat four without (77.9 us) and three (102 registers and 32
// accumulation registers, 78.4).
template <int P, int KIND, bool UPD>
__device__ __forceinline__ void simplex_block(const SimplexParams& p, int64_t first, int count, int met, double* lds) {
    using S = SimplexShape<P>;
    constexpr int NB = S::NB;
    constexpr int NI = 2;  // face functions a thread has in flight
    const int tid = threadIdx.x;
    const int64_t E = p.n_elem;
    const int64_t base0 = p.group_dof[P - 1] + (first - p.group_start[P - 1]) * 4 * NB;
    const int lg = met <= 3 ? 2 : met <= 6 ? 3 : 4;  // lanes per face: 4, 8 or 16
    const int FL = 1 << lg, FS = S::fs(FL);
    double* sG = lds;
    double* sF = sG + count * S::ES;
    double* sJ = sF + count * FS;
    const int lane = tid % 64, wave = tid / 64;

    // ---- phase 1: geometry, own values and what the faces meet; then the
    // neighbours' values
    const int n_items = count << (2 + lg);
    const int f = (tid >> lg) & 3, m = tid & (FL - 1);  // the same for all of a thread's items
    uint2 rec[NI];
    int code[NI];
    auto fetch_faces = [&](int i0) {
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            const int it = i0 + tid + k * kBlock;
            rec[k] = make_uint2(0, 0);
            code[k] = 0;
            if (it < n_items) {
                rec[k] = p.frec[first * 4 + (it >> lg)];
                code[k] = p.fcode[(first * 4 + (it >> lg)) * 16 + m];
            }
        }
    };
    int64_t nbr_at[4 * NI];
    double w[4 * NI], w1[4 * NI];  // per face function the neighbour's v and s
    auto fetch_neighbours = [&] {
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            const int nbn = rec[k].y & 63;
            const int64_t b = code[k] != 0 ? int64_t(rec[k].x) * 4 + (code[k] & 63) : base0;
#pragma unroll
            for (int q = 0; q < 4; ++q) nbr_at[4 * k + q] = b + (code[k] != 0 ? q * nbn : 0);
        }
        load_two<KIND>(p.io, nbr_at, w, w1);
    };
    fetch_faces(0);
    const int own_fn = p.cols[f * 16 + m];
    const bool row_ok = tid < count * NB;
    const int row_le = tid / NB;
    int64_t own_at[4];
    double u[4], u1[4];
    {
        const int64_t b = base0 + (row_ok ? row_le * 4 * NB + tid % NB : 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) own_at[q] = b + q * NB;
    }
    load_two<KIND>(p.io, own_at, u, u1);
    for (int k = tid; k < count * S::JS; k += kBlock) {
        const int le = k / S::JS, c = k % S::JS;
        const double* Jp = p.jinv + first + le;
        sJ[k] = c < 9 ? Jp[c * E] : c < 12 ? -(Jp[(c - 9) * E] + Jp[(c - 6) * E] + Jp[(c - 3) * E])
                                  : 1.0 / p.cinv[first + le];
    }
    __syncthreads();
    fetch_neighbours();
    mix_two<KIND>(p.io, own_at, u, u1);
    if (row_ok) {
        double* g = sG + row_le * S::ES + tid % NB;
        const double* J = sJ + row_le * S::JS;
        g[0] = u[0];
#pragma unroll
        for (int r = 0; r < 3; ++r) g[(1 + r) * NB] = fma(J[3 * r + 2], u[3], fma(J[3 * r + 1], u[2], J[3 * r] * u[1]));
    }

    // ---- the matrix cores' first task of this wave (phase 3) and its first
    // table values: the values of one direction, or of two faces, are loaded
    // while the previous ones are multiplied
    const int col = lane % 16, kk = lane / 16;
    const bool vcol = col >= kTile;
    const int tasks = S::NTM * ((count + kTile - 1) / kTile);  // (row tile fast, column tile slow)
    const int rt = wave % S::NTM;
    const double* Dr = p.tab + p.tab_dr[P - 1] + kk * S::NBP + 16 * rt + col;
    const double* L = p.tab + p.tab_lift[P - 1] + kk * S::NBP + 16 * rt + col;
    constexpr int AG = S::KS > 8 ? S::KS : 8;
    double av[2][AG];
    auto fetch = [&](int g, double (&a)[AG]) {
        if (g < 3) {
#pragma unroll
            for (int s = 0; s < S::KS; ++s) a[s] = Dr[(g * S::KP + 4 * s) * S::NBP];
        } else {
#pragma unroll
            for (int s = 0; s < 8; ++s) a[s] = L[(((g - 3) * 2 + s / 4) * 16 + 4 * (s % 4)) * S::NBP];
        }
    };
    fetch(0, av[0]);
    mix_two<KIND>(p.io, nbr_at, w, w1);
    __syncthreads();

    // ---- phase 2: the face integrands
    for (int i0 = 0;;) {
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            const int it = i0 + tid + k * kBlock, le = it >> (lg + 2);
            const bool in = it < n_items;
            double Jf[3] = {0, 0, 0};
            if (in) {
#pragma unroll
                for (int d = 0; d < 3; ++d) Jf[d] = sJ[le * S::JS + 3 * f + d];
            }
            const double nv = w[4 * k], ng = fma(Jf[2], w[4 * k + 3], fma(Jf[1], w[4 * k + 2], Jf[0] * w[4 * k + 1]));
            // the other of the two degree-4 face functions sits in the lane of 27 - m
            const int partner = m >= 13 && m < 15 ? lane + 27 - 2 * m : lane;
            const double pv = __shfl(nv, partner, 64), pg = __shfl(ng, partner, 64);
            if (!in) continue;
            double bv = 0, bg = 0;
            // 1: +, 2: - (m = 15 is no face function: what such a lane has loaded is nobody's)
            const int c1 = code[k] >> 6, c2 = m >= 13 && m < 15 ? (rec[k].y >> (m == 13 ? 8 : 10)) & 3 : 0;
            if (c1 == 1 || c1 == 2) {
                bv = c1 == 1 ? nv : -nv;
                bg = c1 == 1 ? ng : -ng;
            }
            if (c2 != 0) {
                bv += c2 == 1 ? pv : -pv;
                bg += c2 == 1 ? pg : -pg;
            }
            double ov = 0, og = 0;
            if (m < S::NC) {
                const double* g = sG + le * S::ES + own_fn;
                ov = g[0];
                og = f < 3 ? g[(1 + f) * NB] : -(g[NB] + g[2 * NB] + g[3 * NB]);
            }
            const bool inner = (rec[k].y & 64) != 0;
            double* out = sF + le * FS + f * 2 * FL + m;
            out[0] = inner ? 0.5 * (og - bg) : og;
            out[FL] = inner ? (f < 3 ? 0.5 : -0.5) * (ov - bv) : 0.0;
        }
        i0 += NI * kBlock;
        if (i0 >= n_items) break;
        fetch_faces(i0);
        fetch_neighbours();
        mix_two<KIND>(p.io, nbr_at, w, w1);
    }
    __syncthreads();

    // ---- phase 3: derivatives and lifts on the matrix cores; the results
    // take the place of v and g_r. Orders 1 and 2 have one row tile: the wave
    // is the only reader of its column tile's values. Orders 3 and 4 have one
    // task per wave, whose results wait for the other waves' reads.
    const int fsteps = (met + 3) / 4;
    static_assert(S::NTM == 1 || S::NTM * 2 <= 4 || P == 4, "one task per wave");
    mfma_d4 acc[4];
    auto multiply = [&](int ct) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = mfma_d4{0, 0, 0, 0};
        const int le = ct * kTile + col % kTile < count ? ct * kTile + col % kTile : count - 1;
        const double* gB = sG + le * S::ES + kk;
        const double* fB = sF + le * FS + (vcol ? FL : 0) + kk;
#pragma unroll
        for (int g = 0; g < 5; ++g) {
            if (g < 4) fetch(g + 1, av[(g + 1) % 2]);
            const double (&a)[AG] = av[g % 2];
            if (g < 3) {
#pragma unroll
                for (int s = 0; s < S::KS; ++s) {
                    // (the table is zero beyond NB, but zero times a stray infinity is not)
                    const double b = 4 * s + 3 < NB || 4 * s + kk < NB ? gB[(vcol ? 0 : 1 + g) * NB + 4 * s] : 0.0;
                    acc[g] = mfma_step(a[s], b, acc[g]);
                }
            } else {
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const int q = (g - 3) * 2 + s / 4;
                    if (s % 4 < fsteps) acc[q] = mfma_step(a[s], fB[q * 2 * FL + 4 * (s % 4)], acc[q]);
                }
            }
        }
    };
    auto keep = [&](int ct) {
        const int le = ct * kTile + col % kTile;
        if (le >= count) return;
        const double* J = sJ + le * S::JS;
        const double ci = J[12];
        double* out = sG + le * S::ES;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = 16 * rt + 4 * q + kk;
            if (row >= NB) continue;
            if (!vcol) {
                out[row] = acc[0][q] + acc[1][q] + acc[2][q] + acc[3][q];
            } else {
                double b[3];
#pragma unroll
                for (int r = 0; r < 3; ++r) b[r] = acc[r][q] + acc[3][q];
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    out[(1 + d) * NB + row] = fma(J[6 + d], b[2], fma(J[3 + d], b[1], J[d] * b[0])) * ci;
            }
        }
    };
    if constexpr (S::NTM == 1) {
        for (int t = wave; t < tasks; t += kBlock / 64) {
            if (t != wave) fetch(0, av[0]);
            multiply(t);
            keep(t);
        }
    } else {
        if (wave < tasks) multiply(wave / S::NTM);
        __syncthreads();
        if (wave < tasks) keep(wave / S::NTM);
    }
    __syncthreads();

    // ---- phase 4: the block's values are stored (and the update read) in order
    constexpr int NO = 4;  // outputs a thread has in flight
    const int n_out = count * 4 * NB;
    for (int i0 = tid; i0 < n_out; i0 += NO * kBlock) {
        int64_t at[NO];
        double k[NO];
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int i = i0 + j * kBlock < n_out ? i0 + j * kBlock : i0;  // (past the end: the first once more)
            at[j] = base0 + i;
            k[j] = sG[i / (4 * NB) * S::ES + i % (4 * NB)];
            if (p.io.out_f32) {
                const float v = float(k[j]);
                static_cast<float*>(p.io.out)[at[j]] = v;
                k[j] = double(v);
            } else {
                static_cast<double*>(p.io.out)[at[j]] = k[j];
            }
        }
        if constexpr (UPD) rk_update_n(p.io.upd, at, k);  // the RK update fused into a step's last stage
    }
}

// What a face's lanes need of its neighbour, from the faces and the matching
// table, once per mesh: per (element, face) the neighbour's first DOF / 4 and,
// packed, its functions (bits 0-5), whether there is one (6) and the
// coefficients of the partners of face functions 13 (8-9) and 14 (10-11); per
// face function a byte: the neighbour's function (bits 0-5) and 64 times its
// coefficient's code, or 192 if only the partner takes it; 0: nothing there.
struct SimplexFaceParams {
    int64_t n_elem;
    const int32_t* nbr;
    const int32_t* info;
    const int64_t* elem_off;
    const int32_t* tix;
    uint2* frec;
    uint8_t* fcode;
};

__global__ __launch_bounds__(kBlock) void simplex_faces(const SimplexFaceParams p) {
    const int64_t it = int64_t(blockIdx.x) * kBlock + threadIdx.x;  // (element, face)
    if (it >= 4 * p.n_elem) return;
    const int64_t e = it / 4;
    const int f = int(it % 4);
    const int32_t nb = p.nbr[f * p.n_elem + e], info = p.info[f * p.n_elem + e];
    uint2 rec = make_uint2(0, 0);
    for (int m = 0; m < 16; ++m) {
        int byte = 0;
        if (nb >= 0) {
            const int nbn = simplex_nb(info_pn(info));
            rec.x = uint32_t(p.elem_off[nb] / 4);
            rec.y |= uint32_t(nbn) | 64u;
            const int code = p.tix[kTixFace + ((f * 4 + info_lf(info)) * 6 + info_rel(info)) * 16 + m];
            if (m < kFaceBasis && (code & 63) < nbn) {
                const int c1 = (code >> 6) & 3;
                byte = (code & 63) | ((c1 == 0 ? 3 : c1) << 6);
                if (m >= 13) rec.y |= uint32_t((code >> 8) & 3) << (m == 13 ? 8 : 10);
            }
        }
        p.fcode[it * 16 + m] = uint8_t(byte);
    }
    p.frec[it] = rec;
}

// All orders in one launch, one kernel for each way the stage values are stored
// and counted (StageKind): deciding that inside costs registers. Blocks follow a schedule built on the host: the
// mesh is cut into slabs of consecutive elements and, slab after slab, each
// order's elements of the slab fill blocks of that order. With the XCD
// renumbering an XCD works through neighbouring slabs, so the values an
// element gathers from neighbours of every order are read while they are
// still in that XCD's L2.
template <int KIND, bool UPD>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5))) void simplex_acoustic_rhs(const SimplexParams p) {
    __shared__ double lds[kSimplexLds];
    const int4 bl = p.blocks[xcd_block(blockIdx.x, gridDim.x)];
    switch (bl.x) {  // the same order for the whole block
        case 1: simplex_block<1, KIND, UPD>(p, bl.y, bl.z, bl.w, lds); break;
        case 2: simplex_block<2, KIND, UPD>(p, bl.y, bl.z, bl.w, lds); break;
        case 3: simplex_block<3, KIND, UPD>(p, bl.y, bl.z, bl.w, lds); break;
        default: simplex_block<4, KIND, UPD>(p, bl.y, bl.z, bl.w, lds); break;
    }
}

// Per-element |det J| sum_f dx_f^T M_ref dx_f (plain L2 of all fields) and
// max |dx|, one partial per block.
struct SimplexDiffParams {
    int64_t n_elem;
    int64_t group_start[5];
    int64_t group_dof[5];
    int32_t group_block[5];
    const void* x;
    const void* y;
    int32_t x_f32, y_f32;
    const double* absdet;
    const double* tab;
    const int32_t* tix;
    double* partial;
};

template <int P>
struct SimplexRows {
    static constexpr int NB = simplex_nb(P), TPE = simplex_tpe(P), EPB = kBlock / TPE;
};

template <int P>
__device__ void simplex_diff_block(const SimplexDiffParams& p, int blk, double* sd, double* red) {
    using S = SimplexRows<P>;
    constexpr int NB = S::NB;
    const int tid = threadIdx.x;
    const int le = tid / S::TPE;
    const int i = tid % S::TPE;
    const int64_t e = p.group_start[P - 1] + int64_t(blk) * S::EPB + le;
    const bool row_ok = (le < S::EPB) && (e < p.group_start[P]) && (i < NB);
    const int64_t base = p.group_dof[P - 1] + (e - p.group_start[P - 1]) * 4 * NB;
    double* d = sd + le * 4 * NB;
    double v = 0, m = 0;
    if (row_ok)
        for (int f = 0; f < 4; ++f) {
            const int64_t k = base + f * NB + i;
            const double xv = p.x_f32 ? double(static_cast<const float*>(p.x)[k]) : static_cast<const double*>(p.x)[k];
            const double yv = p.y_f32 ? double(static_cast<const float*>(p.y)[k]) : static_cast<const double*>(p.y)[k];
            d[f * NB + i] = xv - yv;
            m = fmax(m, fabs(xv - yv));
        }
    __syncthreads();
    if (row_ok) {
        const double* M = p.tab + p.tix[(P - 1) * kTixStride + kTixM] + i * NB;
        for (int f = 0; f < 4; ++f) {
            double s = 0;
            for (int j = 0; j < NB; ++j) s += M[j] * d[f * NB + j];
            v += s * d[f * NB + i];
        }
        v *= p.absdet[e];
    }
    red[tid] = v;
    red[kBlock + tid] = m;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (tid < w) {
            red[tid] += red[tid + w];
            red[kBlock + tid] = fmax(red[kBlock + tid], red[kBlock + tid + w]);
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void simplex_diff_norm(const SimplexDiffParams p) {
    constexpr int n1 = SimplexRows<1>::EPB * 4 * SimplexRows<1>::NB, n2 = SimplexRows<2>::EPB * 4 * SimplexRows<2>::NB;
    constexpr int n3 = SimplexRows<3>::EPB * 4 * SimplexRows<3>::NB, n4 = SimplexRows<4>::EPB * 4 * SimplexRows<4>::NB;
    constexpr int n12 = n1 > n2 ? n1 : n2, n34 = n3 > n4 ? n3 : n4;
    __shared__ double sd[n12 > n34 ? n12 : n34];  // [EPB][4][NB] of the largest order group
    __shared__ double red[2 * kBlock];
    const int b = blockIdx.x;
    if (b < p.group_block[1]) simplex_diff_block<1>(p, b - p.group_block[0], sd, red);
    else if (b < p.group_block[2]) simplex_diff_block<2>(p, b - p.group_block[1], sd, red);
    else if (b < p.group_block[3]) simplex_diff_block<3>(p, b - p.group_block[2], sd, red);
    else simplex_diff_block<4>(p, b - p.group_block[3], sd, red);
    if (threadIdx.x == 0) {
        p.partial[2 * b] = red[0];
        p.partial[2 * b + 1] = red[kBlock];
    }
}

// The block-diagonal mass matrix of the acoustic system
// (AcousticWaveLinear_Impl.h:102-129: |det J| M_ref on v, c_inv |det J| M_ref
// on each s_d) applied to a vector or solved against it, in place. One
// wavefront per element; the element's four fields are staged in LDS.
struct SimplexMassParams {
    const int64_t* elem_off;  // [n_elem + 1]
    const int32_t* order;     // [n_elem]
    const double* tab;        // per order: M_ref, then M_ref^{-1}
    int32_t tab_off[2][4];    // [apply / solve][order - 1]
    int32_t inverse;
    double* v;
    const double* absdet;     // [n_elem]
    const double* cinv;       // [n_elem]
};

__global__ __launch_bounds__(64) void simplex_mass(const SimplexMassParams p) {
    __shared__ double s[4 * SimplexShape<4>::NB];
    const int64_t e = blockIdx.x;
    const int P = p.order[e];
    const int nb = (P + 1) * (P + 2) * (P + 3) / 6;
    const int n = 4 * nb;
    const int64_t off = p.elem_off[e];
    for (int i = threadIdx.x; i < n; i += 64) s[i] = p.v[off + i];
    __syncthreads();
    const double* A = p.tab + p.tab_off[p.inverse][P - 1];
    const double w0 = p.absdet[e];
    const double ws = w0 * p.cinv[e];
    for (int r = threadIdx.x; r < n; r += 64) {
        const int f = r / nb, i = r - f * nb;
        double acc = 0;
        for (int j = 0; j < nb; ++j) acc += A[i * nb + j] * s[f * nb + j];
        const double w = f > 0 ? ws : w0;
        p.v[off + r] = p.inverse ? acc / w : acc * w;
    }
}

// Quadrature tables of the on-device projection and error norms, per order
// (index p - 1), as offsets into one table array: the element rule of order
// 2p+1 (points; the projection operator R = M_ref^{-1} [w_q phi_i(x_q)], [nb][nq];
// the basis at its points, [nq][nb], for the maximum error) and the rule of
// order 2p+2 (points, weights and the basis at its points, for the L2 error),
// all hpGEM's tetrahedral rules.
struct SimplexQuadTab {
    int32_t nb[4], nq_p[4], nq_e[4];
    int32_t pts_p[4], R[4], phi_p[4], pts_e[4], w_e[4], phi_e[4];
};

struct SimplexFnParams {
    const double* tab;
    SimplexQuadTab t;
    const double* xj;         // [E][12]: vertex 0, then J row-major (device order)
    const int64_t* elem_off;  // [E + 1]
    const int32_t* order;     // [E]
    int32_t n_fields, field;  // field < 0: every field
    int32_t n_modes;
    const double* modes;      // [n_modes][4]: amplitude, k
    int32_t gaussian;         // 1: f = g[4] exp(-|x - g[0..2]|^2 / g[3]^2) instead of the modes
    double g[5];
    double shift[3];          // error: f(x - shift)
    void* u;                  // projection: output; error: input
    int32_t u_f32;
    const double* absdet;
    double* partial;          // error: [E][2] (squared L2, max)
};

__device__ __forceinline__ void tet_point(const double* xj, const double* xi, double (&x)[3]) {
#pragma unroll
    for (int r = 0; r < 3; ++r) x[r] = xj[r] + xj[3 + r * 3] * xi[0] + xj[3 + r * 3 + 1] * xi[1] + xj[3 + r * 3 + 2] * xi[2];
}

__device__ __forceinline__ double tet_fn(const SimplexFnParams& p, const double (&x)[3]) {
    if (p.gaussian) {
        const double r2 = (x[0] - p.g[0]) * (x[0] - p.g[0]) + (x[1] - p.g[1]) * (x[1] - p.g[1]) +
                          (x[2] - p.g[2]) * (x[2] - p.g[2]);
        return p.g[4] * exp(-r2 / (p.g[3] * p.g[3]));
    }
    double f = 0;
    for (int m = 0; m < p.n_modes; ++m) {
        const double* md = p.modes + 4 * m;
        f += md[0] * sin(2 * M_PI * (md[1] * (x[0] - p.shift[0]) + md[2] * (x[1] - p.shift[1]) +
                                     md[3] * (x[2] - p.shift[2])));
    }
    return f;
}

// L2 projection (HpgemAPISimplified::setInitialSolution with hpGEM's element
// rule of order 2p+1): one wavefront per element, lanes over points, then
// over basis functions.
__global__ __launch_bounds__(64) void simplex_project(const SimplexFnParams p) {
    __shared__ double fq[64];
    const int64_t e = blockIdx.x;
    const int P = p.order[e], nb = p.t.nb[P - 1], nq = p.t.nq_p[P - 1];
    const double* xj = p.xj + 12 * e;
    const int l = threadIdx.x;
    if (l < nq) {
        double x[3];
        tet_point(xj, p.tab + p.t.pts_p[P - 1] + 3 * l, x);
        fq[l] = tet_fn(p, x);
    }
    __syncthreads();
    if (l < nb) {
        const double* R = p.tab + p.t.R[P - 1] + l * nq;
        double s = 0;
        for (int q = 0; q < nq; ++q) s += R[q] * fq[q];
        const int64_t o = p.elem_off[e];
        for (int f = 0; f < p.n_fields; ++f) {
            if (p.field >= 0 && f != p.field) continue;
            if (p.u_f32) static_cast<float*>(p.u)[o + f * nb + l] = float(s);
            else static_cast<double*>(p.u)[o + f * nb + l] = s;
        }
    }
}

// computeTotalError (rule 2p+2) and computeMaxError (the points of the rule
// 2p+1) of one field or all, per element: partial[2e] = |det J| sum_q w_q
// err^2, partial[2e+1] = max |err|.
__global__ __launch_bounds__(64) void simplex_error(const SimplexFnParams p) {
    __shared__ double cf[4 * SimplexShape<4>::NB];
    const int64_t e = blockIdx.x;
    const int P = p.order[e], nb = p.t.nb[P - 1];
    const double* xj = p.xj + 12 * e;
    const int64_t o = p.elem_off[e];
    const int l = threadIdx.x;
    for (int k = l; k < p.n_fields * nb; k += 64)
        cf[k] = p.u_f32 ? double(static_cast<const float*>(p.u)[o + k]) : static_cast<const double*>(p.u)[o + k];
    __syncthreads();
    double s2 = 0, mx = 0;
    for (int pass = 0; pass < 2; ++pass) {
        const int nq = pass == 0 ? p.t.nq_e[P - 1] : p.t.nq_p[P - 1];
        const double* pts = p.tab + (pass == 0 ? p.t.pts_e[P - 1] : p.t.pts_p[P - 1]);
        const double* phi = p.tab + (pass == 0 ? p.t.phi_e[P - 1] : p.t.phi_p[P - 1]);
        for (int q = l; q < nq; q += 64) {
            double x[3];
            tet_point(xj, pts + 3 * q, x);
            const double ex = tet_fn(p, x);
            for (int f = 0; f < p.n_fields; ++f) {
                if (p.field >= 0 && f != p.field) continue;
                double val = 0;
                for (int i = 0; i < nb; ++i) val += cf[f * nb + i] * phi[q * nb + i];
                const double err = ex - val;
                if (pass == 0) s2 += p.tab[p.t.w_e[P - 1] + q] * err * err;
                else mx = fmax(mx, fabs(err));
            }
        }
    }
    for (int w = 32; w > 0; w /= 2) {
        s2 += __shfl_xor(s2, w, 64);
        mx = fmax(mx, __shfl_xor(mx, w, 64));
    }
    if (l == 0) {
        p.partial[2 * e] = s2 * p.absdet[e];
        p.partial[2 * e + 1] = mx;
    }
}

// ---------------------------------------------------------------- host side
namespace {

int epb_of(int p) { return kBlock / simplex_tpe(p); }

void group_blocks(const SimplexMesh& sm, int32_t* gb) {
    gb[0] = 0;
    for (int g = 0; g < 4; ++g) {
        const int64_t n = sm.group_start[g + 1] - sm.group_start[g];
        gb[g + 1] = gb[g] + int32_t((n + epb_of(g + 1) - 1) / epb_of(g + 1));
    }
}

}  // namespace

namespace {

// Processing order of the tetrahedra (the order of the RHS kernel's block
// schedule, and of the device layout inside each order group): the elements'
// centroids are cut into 4 x 4 columns across the two shorter extents of the
// mesh's bounding box and run through column by column, along the longest
// extent inside a column. A face neighbour is then either in the same column,
// at most one column layer (a few hundred elements) away in processing order,
// so its face columns are still in the XCD's L2 when they are gathered, or
// across a column side; in mesh order (x fastest) every neighbour along the
// slowest axis was a whole mesh layer back, beyond the L2.
std::vector<int64_t> locality_rank(const hgdg_mesh_desc* m) {
    const int64_t ne = m->n_elements;
    std::vector<std::array<double, 3>> ctr(static_cast<size_t>(ne));
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t e = 0; e < ne; ++e)
        for (int r = 0; r < 3; ++r) {
            double s = 0;
            for (int v = 0; v < 4; ++v) s += m->coords[(size_t(e) * 4 + v) * 3 + r];
            ctr[size_t(e)][r] = s / 4;
            lo[r] = std::min(lo[r], s / 4);
            hi[r] = std::max(hi[r], s / 4);
        }
    int ax[3] = {0, 1, 2};  // ax[2]: the longest extent (the last of equal ones)
    std::stable_sort(ax, ax + 3, [&](int a, int b) { return hi[a] - lo[a] < hi[b] - lo[b]; });
    constexpr int kCols = 4;
    auto cell = [&](int64_t e, int r) {
        const double ext = hi[r] - lo[r];
        if (!(ext > 0)) return 0;
        return std::min(kCols - 1, int((ctr[size_t(e)][r] - lo[r]) / ext * kCols));
    };
    std::vector<int64_t> idx(static_cast<size_t>(ne));
    for (int64_t e = 0; e < ne; ++e) idx[size_t(e)] = e;
    std::stable_sort(idx.begin(), idx.end(), [&](int64_t a, int64_t b) {
        const int ca = cell(a, ax[1]) * kCols + cell(a, ax[0]), cb = cell(b, ax[1]) * kCols + cell(b, ax[0]);
        if (ca != cb) return ca < cb;
        for (int k = 2; k >= 0; --k)
            if (ctr[size_t(a)][ax[k]] != ctr[size_t(b)][ax[k]]) return ctr[size_t(a)][ax[k]] < ctr[size_t(b)][ax[k]];
        return a < b;
    });
    std::vector<int64_t> rank(static_cast<size_t>(ne));
    for (int64_t k = 0; k < ne; ++k) rank[size_t(idx[size_t(k)])] = k;
    return rank;
}

}  // namespace

namespace {

// P^{-1} Q of two kFaceBasis x kFaceBasis matrices, row-major (Gauss-Jordan in
// long double, partial pivoting).
std::vector<double> face_match(const std::vector<double>& P, const std::vector<double>& Q) {
    constexpr int n = kFaceBasis;
    std::vector<long double> a(P.begin(), P.end()), b(Q.begin(), Q.end());
    for (int k = 0; k < n; ++k) {
        int piv = k;
        for (int i = k + 1; i < n; ++i)
            if (std::fabs(a[i * n + k]) > std::fabs(a[piv * n + k])) piv = i;
        for (int j = 0; j < n; ++j) {
            std::swap(a[k * n + j], a[piv * n + j]);
            std::swap(b[k * n + j], b[piv * n + j]);
        }
        const long double d = a[k * n + k];
        for (int j = 0; j < n; ++j) {
            a[k * n + j] /= d;
            b[k * n + j] /= d;
        }
        for (int i = 0; i < n; ++i) {
            const long double f = a[i * n + k];
            if (i == k || f == 0) continue;
            for (int j = 0; j < n; ++j) {
                a[i * n + j] -= f * a[k * n + j];
                b[i * n + j] -= f * b[k * n + j];
            }
        }
    }
    return std::vector<double>(b.begin(), b.end());
}

// How a neighbour's face functions meet ours (kTixFace), from the order-4 tables
// and the identity among the orientations; the same for every mesh, and made once
// (1.5 ms): P_f O = P_lf,rel in face-basis coefficients.
const std::vector<int32_t>& face_matches(const SimplexOps& top, int ident) {
    static const std::vector<int32_t> table = [&] {
        std::vector<int32_t> match(4 * 4 * 6 * 16, 0);
        for (int f = 0; f < 4; ++f)
            for (int lf = 0; lf < 4; ++lf)
                for (int o = 0; o < 6; ++o) {
                    const std::vector<double> O = face_match(top.proj[f][ident], top.proj[lf][o]);
                    for (int m = 0; m < kFaceBasis; ++m) {
                        int from = m >= 13 ? m : -1, c1 = 0, c2 = 0;
                        for (int q = 0; q < kFaceBasis; ++q) {
                            const double v = O[size_t(m) * kFaceBasis + q];
                            const int r = int(std::lround(v));
                            require(std::fabs(v - r) < 1e-9 && std::abs(r) <= 1, HGDG_ERR_ARG, "face functions do not match");
                            if (r == 0) continue;
                            const int code = r > 0 ? 1 : 2;
                            if (m < 13) {
                                require(from < 0 && q < 13, HGDG_ERR_ARG, "face functions do not match one to one");
                                from = q;
                                c1 = code;
                            } else {
                                require(q >= 13, HGDG_ERR_ARG, "degree-4 face functions mix with others");
                                (q == m ? c1 : c2) = code;
                            }
                        }
                        require(from >= 0, HGDG_ERR_ARG, "a face function without match");
                        match[size_t((f * 4 + lf) * 6 + o) * 16 + m] = top.cols[lf][size_t(from)] | (c1 << 6) | (c2 << 8);
                    }
                }
        return match;
    }();
    return table;
}

}  // namespace

void simplex_mesh_upload(hgdg_ctx* c, const hgdg_mesh_desc* m) {
    SimplexMesh& sm = c->sm;
    const int64_t ne = m->n_elements;
    std::vector<int32_t> order(ne);
    for (int64_t e = 0; e < ne; ++e) {
        order[e] = m->order ? m->order[e] : m->uniform_order;
        require(order[e] >= 1 && order[e] <= kMaxSimplexOrder, HGDG_ERR_UNSUPPORTED,
                "tetrahedral orders must be in 1..4");
    }
    // group by order; inside a group, elements follow the locality rank
    int64_t counts[4] = {0, 0, 0, 0};
    for (int64_t e = 0; e < ne; ++e) ++counts[order[e] - 1];
    sm.group_start[0] = 0;
    for (int g = 0; g < 4; ++g) sm.group_start[g + 1] = sm.group_start[g] + counts[g];
    sm.dev_of.assign(ne, 0);
    sm.mesh_of.assign(ne, 0);
    sm.order.assign(ne, 0);
    sm.rank = locality_rank(m);
    std::vector<int64_t> by_rank(ne);
    for (int64_t e = 0; e < ne; ++e) by_rank[size_t(sm.rank[e])] = e;
    int64_t fill[4] = {sm.group_start[0], sm.group_start[1], sm.group_start[2], sm.group_start[3]};
    for (int64_t e : by_rank) {
        const int64_t d = fill[order[e] - 1]++;
        sm.dev_of[e] = d;
        sm.mesh_of[d] = e;
        sm.order[d] = order[e];
    }
    constexpr int nf = 4;  // fields of the acoustic system
    sm.group_dof[0] = 0;
    for (int g = 0; g < 4; ++g) sm.group_dof[g + 1] = sm.group_dof[g] + counts[g] * nf * tet_nb(g + 1);
    sm.dof_off.assign(ne, 0);
    sm.d_io_off.reset();
    for (int64_t d = 0; d < ne; ++d) {
        const int g = sm.order[d] - 1;
        sm.dof_off[d] = sm.group_dof[g] + (d - sm.group_start[g]) * nf * tet_nb(g + 1);
    }
    c->n_fields = nf;
    c->dof = sm.group_dof[4];
    std::vector<int64_t> elem_off(sm.dof_off);  // lives until the synchronize at the end
    elem_off.push_back(c->dof);
    sm.d_elem_off.upload(elem_off, c->stream);

    // geometry (device order): J column k = X_{k+1} - X_0
    sm.jinv.assign(size_t(ne) * 9, 0.0);
    sm.absdet.assign(ne, 0.0);
    std::vector<double> jinv_soa(9 * size_t(ne)), detJ(ne);
    std::vector<std::array<double, 9>> Jm(ne);
    sm.x0.assign(size_t(ne) * 3, 0.0);
    sm.jac.assign(size_t(ne) * 9, 0.0);
    for (int64_t d = 0; d < ne; ++d) {
        const double* X = m->coords + size_t(sm.mesh_of[d]) * 12;
        for (int r = 0; r < 3; ++r) sm.x0[size_t(d) * 3 + r] = X[r];
        double J[3][3];
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) J[r][k] = X[(k + 1) * 3 + r] - X[r];
        const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                           J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                           J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
        require(det != 0.0 && std::isfinite(det), HGDG_ERR_ARG, "degenerate tetrahedron");
        double inv[3][3];
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) {
                const int r1 = (k + 1) % 3, r2 = (k + 2) % 3, c1 = (r + 1) % 3, c2 = (r + 2) % 3;
                inv[r][k] = (J[r1][c1] * J[r2][c2] - J[r1][c2] * J[r2][c1]) / det;
            }
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < 3; ++k) {
                jinv_soa[(r * 3 + k) * size_t(ne) + d] = inv[r][k];
                Jm[d][r * 3 + k] = J[r][k];
                sm.jac[size_t(d) * 9 + r * 3 + k] = J[r][k];
            }
        detJ[d] = det;
        sm.absdet[d] = std::fabs(det);
    }

    // faces: sorted node triples; the lower mesh index is hpGEM's left element
    sm.nbr_dev.assign(4 * size_t(ne), -1);
    sm.info.assign(4 * size_t(ne), 0);
    struct Open { int64_t e; int f; };
    std::unordered_map<std::string, Open> open;
    open.reserve(size_t(ne) * 2);
    int64_t n_internal = 0, n_total = 0;
    sm.sigma.assign(4 * size_t(ne), 0.0);
    sm.normal.assign(12 * size_t(ne), 0.0);
    static const double V[4][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int64_t e = 0; e < ne; ++e) {
        const int64_t* nid = m->node_ids + size_t(e) * 4;
        const int64_t d = sm.dev_of[e];
        for (int f = 0; f < 4; ++f) {
            // outward normal: sign(det J) (J c1) x (J c2), c = face edges in
            // reference coordinates (FaceGeometry.h:412-459)
            const int* fn = kTetFaceNodes[f];
            double a[3], b[3];
            for (int r = 0; r < 3; ++r) {
                a[r] = 0;
                b[r] = 0;
                for (int k = 0; k < 3; ++k) {
                    a[r] += Jm[d][r * 3 + k] * (V[fn[1]][k] - V[fn[0]][k]);
                    b[r] += Jm[d][r * 3 + k] * (V[fn[2]][k] - V[fn[0]][k]);
                }
            }
            double nrm[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
            const double sg = detJ[d] > 0 ? 1.0 : -1.0;
            const double len = std::sqrt(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
            for (int r = 0; r < 3; ++r) sm.normal[(size_t(r) * 4 + f) * ne + d] = sg * nrm[r] / len;
            sm.sigma[size_t(f) * ne + d] = len / sm.absdet[d];
            sm.info[size_t(f) * ne + d] = info_pack(0, 0, 0, 0);

            std::array<int64_t, 3> key{nid[fn[0]], nid[fn[1]], nid[fn[2]]};
            std::sort(key.begin(), key.end());
            std::string k(reinterpret_cast<const char*>(key.data()), sizeof(key));
            auto it = open.find(k);
            if (it == open.end()) {
                open.emplace(std::move(k), Open{e, f});
                continue;
            }
            const int64_t L = it->second.e;
            const int fL = it->second.f;
            require(L != e, HGDG_ERR_ARG, "tetrahedron meets itself across a face");
            const int64_t* lid = m->node_ids + size_t(L) * 4;
            long long ln[3], rn[3];
            for (int q = 0; q < 3; ++q) {
                ln[q] = lid[kTetFaceNodes[fL][q]];
                rn[q] = nid[fn[q]];
            }
            const int o = tri_orientation_index(ln, rn);
            const int64_t dL = sm.dev_of[L];
            require(sm.nbr_dev[size_t(fL) * ne + dL] < 0, HGDG_ERR_ARG, "a face is bounded by more than two elements");
            sm.nbr_dev[size_t(fL) * ne + dL] = int32_t(d);
            sm.nbr_dev[size_t(f) * ne + d] = int32_t(dL);
            sm.info[size_t(fL) * ne + dL] = info_pack(f, 0, o, sm.order[d]);
            sm.info[size_t(f) * ne + d] = info_pack(fL, o, 0, sm.order[dL]);
            open.erase(it);
            ++n_internal;
            ++n_total;
        }
    }
    n_total += int64_t(open.size());
    c->n_faces = n_total;
    c->n_internal = n_internal;

    int perm[6][kFaceQ];  // face point q after orientation o of the reference triangle
    for (int o = 0; o < 6; ++o)
        for (int qq = 0; qq < kFaceQ; ++qq) {
            const long double tp[2] = {kFaceRulePts[qq][0], kFaceRulePts[qq][1]};
            long double m[2];
            tri_orientation_map(o, tp, m);
            int hit = -1;
            for (int k = 0; k < kFaceQ; ++k)
                if (fabsl(m[0] - kFaceRulePts[k][0]) < 1e-12L && fabsl(m[1] - kFaceRulePts[k][1]) < 1e-12L) hit = k;
            require(hit >= 0, HGDG_ERR_ARG, "face rule is not symmetric under the orientation maps");
            perm[o][qq] = hit;
        }
    // Both sides of a face reach a physical point through their orientation:
    // own coordinates o_own(t), neighbour's o_nbr(t). Seen from the element,
    // the neighbour's face coordinates are o_nbr(o_own^{-1}(s)), itself one
    // of the six orientation maps (they form a group), identified here by
    // its action on the (symmetric) face rule points.
    std::vector<int32_t> tix(size_t(kTixSize), 0);
    int rel_of[6][6];
    int ident = -1;
    for (int o = 0; o < 6 && ident < 0; ++o) {
        bool id = true;
        for (int qq = 0; qq < kFaceQ; ++qq) id = id && perm[o][qq] == qq;
        if (id) ident = o;
    }
    require(ident >= 0, HGDG_ERR_ARG, "no identity among the face orientation maps");
    for (int oo = 0; oo < 6; ++oo) {
        int inv[kFaceQ];
        for (int qq = 0; qq < kFaceQ; ++qq) inv[perm[oo][qq]] = qq;
        for (int on = 0; on < 6; ++on) {
            int rel = -1;
            for (int o = 0; o < 6 && rel < 0; ++o) {
                bool same = true;
                for (int r = 0; r < kFaceQ; ++r) same = same && perm[o][r] == perm[on][inv[r]];
                if (same) rel = o;
            }
            require(rel >= 0, HGDG_ERR_ARG, "face orientation maps do not compose");
            rel_of[oo][on] = rel;
        }
    }
    for (size_t k = 0; k < sm.info.size(); ++k)
        if (sm.nbr_dev[k] >= 0)
            sm.info[k] |= rel_of[info_oown(sm.info[k])][info_onbr(sm.info[k])] << 11;
    sm.ops.clear();
    for (int q = 1; q <= kMaxSimplexOrder; ++q) sm.ops.push_back(simplex_ops(q));
    // reference tables of every order (see the kernel)
    std::vector<double> tab;
    const SimplexOps& top = sm.ops[kMaxSimplexOrder - 1];
    for (int q = 1; q <= kMaxSimplexOrder; ++q) {
        const SimplexOps& ops = sm.ops[q - 1];
        const int nb = ops.nb, kp = 4 * ((nb + 3) / 4), ip = 16 * ((nb + 15) / 16);
        int32_t* t = tix.data() + (q - 1) * kTixStride;
        t[kTixM] = int32_t(tab.size());
        tab.insert(tab.end(), ops.Mref.begin(), ops.Mref.end());
        t[kTixDrP] = int32_t(tab.size());
        for (int r = 0; r < 3; ++r)
            for (int k = 0; k < kp; ++k)
                for (int i = 0; i < ip; ++i)
                    tab.push_back(k < nb && i < nb ? ops.Dr[(size_t(r) * nb + i) * nb + k] : 0.0);
        t[kTixLift] = int32_t(tab.size());
        for (int f = 0; f < 4; ++f) {
            // hierarchical: the order's face functions are the first of the order-4 ones
            const int nc = simplex_ncol(q);
            require(int(ops.cols[f].size()) == nc && int(top.cols[f].size()) == kFaceBasis &&
                        std::equal(ops.cols[f].begin(), ops.cols[f].end(), top.cols[f].begin()),
                    HGDG_ERR_ARG, "unexpected face functions");
            for (int m = 0; m < 16; ++m)
                for (int i = 0; i < ip; ++i) {
                    long double v = 0;
                    if (m < kFaceBasis && i < nb)
                        for (int k = 0; k < kFaceBasis; ++k)
                            v += (long double)ops.lift[f][ident][size_t(i) * kFaceBasis + k] *
                                 top.proj[f][ident][size_t(k) * kFaceBasis + m];
                    tab.push_back(double(v));
                }
        }
    }
    for (int g = 0; g < 4; ++g) {
        sm.tab_dr[g] = tix[size_t(g) * kTixStride + kTixDrP];
        sm.tab_lift[g] = tix[size_t(g) * kTixStride + kTixLift];
    }
    for (int f = 0; f < 4; ++f)
        for (int m = 0; m < kFaceBasis; ++m) tix[size_t(kTixCols) + f * 16 + m] = top.cols[f][size_t(m)];
    const std::vector<int32_t>& match = face_matches(top, ident);
    std::copy(match.begin(), match.end(), tix.begin() + kTixFace);

    for (int g = 0; g < 4; ++g) {
        sm.tpe_variant[g] = sm.tpe_fixed[g] == simplex_tpe_alt(g + 1) ? 1 : 0;
        sm.tpe_ms[g][0] = sm.tpe_ms[g][1] = 0;
    }
    simplex_schedule(c);

    sm.d_tables.upload(tab, c->stream);
    std::vector<double> mass;  // lives until the synchronize below
    for (int q = 1; q <= kMaxSimplexOrder; ++q) mass.insert(mass.end(), sm.ops[q - 1].Mref.begin(), sm.ops[q - 1].Mref.end());
    for (int q = 1; q <= kMaxSimplexOrder; ++q) mass.insert(mass.end(), sm.ops[q - 1].Minv.begin(), sm.ops[q - 1].Minv.end());
    sm.d_mass.upload(mass, c->stream);
    sm.d_order.upload(sm.order, c->stream);
    sm.d_tab_index.upload(tix, c->stream);
    sm.d_absdet.upload(sm.absdet, c->stream);
    std::vector<double> geo(jinv_soa);
    geo.resize(geo.size() + size_t(ne), 1.0);  // c_inv, set with the operator
    sm.d_geo.upload(geo, c->stream);
    std::vector<int32_t> face(sm.nbr_dev);
    face.insert(face.end(), sm.info.begin(), sm.info.end());
    sm.d_face.upload(face, c->stream);
    require(c->dof / 4 <= int64_t(UINT32_MAX), HGDG_ERR_UNSUPPORTED, "more than 2^34 degrees of freedom");
    sm.d_frec.alloc(8 * size_t(ne));
    sm.d_fcode.alloc(64 * size_t(ne));
    SimplexFaceParams fp{ne, sm.d_face.ptr, sm.d_face.ptr + 4 * ne, sm.d_elem_off.ptr, sm.d_tab_index.ptr,
                         reinterpret_cast<uint2*>(sm.d_frec.ptr), sm.d_fcode.ptr};
    hipLaunchKernelGGL(simplex_faces, dim3(unsigned((4 * ne + kBlock - 1) / kBlock)), dim3(kBlock), 0, c->stream, fp);
    HGDG_HIP(hipGetLastError());
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

void simplex_operator_set(hgdg_ctx* c, const hgdg_op_desc* op) {
    require(op->kind == HGDG_OP_ACOUSTIC_CENTRAL, HGDG_ERR_UNSUPPORTED,
            "tetrahedral meshes run the acoustic operator");
    SimplexMesh& sm = c->sm;
    const int64_t ne = c->n_elem;
    std::vector<double> cinv(ne);
    for (int64_t d = 0; d < ne; ++d) cinv[d] = op->c_inv[sm.mesh_of[d]];
    HGDG_HIP(hipMemcpyAsync(sm.d_geo.ptr + 9 * ne, cinv.data(), size_t(ne) * sizeof(double), hipMemcpyHostToDevice,
                            c->stream));
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

int simplex_threads(int order, int variant) { return simplex_tpe_of(order, variant); }

// Block schedule: the mesh is cut into slabs of consecutive elements and, slab
// after slab, each order's elements of the slab fill blocks of that order's
// size in use. With each block goes the number of face functions its elements
// meet: those of the highest order among them and their neighbours.
void simplex_schedule(hgdg_ctx* c) {
    SimplexMesh& sm = c->sm;
    const int64_t ne = c->n_elem;
    const int64_t slab = std::max<int64_t>(1024, (ne + 255) / 256);  // in locality ranks
    int epb[4];
    for (int g = 0; g < 4; ++g) {
        int top = g + 1;  // the highest order the order's elements meet
        for (int64_t e = sm.group_start[g]; e < sm.group_start[g + 1] && top < kMaxSimplexOrder; ++e)
            for (int f = 0; f < 4; ++f) top = std::max(top, info_pn(sm.info[size_t(f) * ne + e]));
        epb[g] = simplex_epb(g + 1, sm.tpe_variant[g], simplex_ncol(top));
    }
    std::vector<int32_t> blocks;
    int64_t cursor[4] = {sm.group_start[0], sm.group_start[1], sm.group_start[2], sm.group_start[3]};
    for (int64_t lo = 0; lo < ne; lo += slab) {
        const int64_t hi = std::min(ne, lo + slab);
        for (int g = 0; g < 4; ++g) {
            // device elements of order g+1 with locality rank below hi (rank order inside a group)
            int64_t end = cursor[g];
            while (end < sm.group_start[g + 1] && sm.rank[size_t(sm.mesh_of[end])] < hi) ++end;
            for (int64_t b = cursor[g]; b < end; b += epb[g]) {
                const int64_t last = std::min<int64_t>(b + epb[g], end);
                int top = g + 1;
                for (int64_t e = b; e < last; ++e)
                    for (int f = 0; f < 4; ++f) top = std::max(top, info_pn(sm.info[size_t(f) * ne + e]));
                blocks.push_back(g + 1);
                blocks.push_back(int32_t(b));
                blocks.push_back(int32_t(last - b));
                blocks.push_back(simplex_ncol(top));
            }
            cursor[g] = end;
        }
    }
    sm.n_blocks = int64_t(blocks.size() / 4);
    sm.d_blocks.upload(blocks, c->stream);
    HGDG_HIP(hipStreamSynchronize(c->stream));  // `blocks` goes out of scope
}

namespace {

SimplexParams simplex_params(hgdg_ctx* c, const StageIO& io) {
    SimplexMesh& sm = c->sm;
    const int64_t ne = c->n_elem;
    SimplexParams p{};
    p.io = io;
    p.n_elem = ne;
    for (int g = 0; g < 5; ++g) {
        p.group_start[g] = sm.group_start[g];
        p.group_dof[g] = sm.group_dof[g];
    }
    p.jinv = sm.d_geo.ptr;
    p.cinv = sm.d_geo.ptr + 9 * ne;
    p.frec = reinterpret_cast<const uint2*>(sm.d_frec.ptr);
    p.fcode = sm.d_fcode.ptr;
    p.tab = sm.d_tables.ptr;
    for (int g = 0; g < 4; ++g) {
        p.tab_dr[g] = sm.tab_dr[g];
        p.tab_lift[g] = sm.tab_lift[g];
    }
    p.cols = sm.d_tab_index.ptr + kTixCols;
    p.blocks = reinterpret_cast<const int4*>(sm.d_blocks.ptr);
    return p;
}

using SimplexKernel = void (*)(SimplexParams);

void launch_simplex(hgdg_ctx* c, const SimplexParams& p) {
    static constexpr SimplexKernel kernels[6][2] = {
        {&simplex_acoustic_rhs<STAGE_ANY, false>, &simplex_acoustic_rhs<STAGE_ANY, true>},
        {&simplex_acoustic_rhs<STAGE_ONE, false>, &simplex_acoustic_rhs<STAGE_ONE, true>},
        {&simplex_acoustic_rhs<STAGE_TWO, false>, &simplex_acoustic_rhs<STAGE_TWO, true>},
        {&simplex_acoustic_rhs<STAGE_TWO_MIXED, false>, &simplex_acoustic_rhs<STAGE_TWO_MIXED, true>},
        {&simplex_acoustic_rhs<STAGE_ANY, false>, &simplex_acoustic_rhs<STAGE_ANY, true>},
        {&simplex_acoustic_rhs<STAGE_ANY, false>, &simplex_acoustic_rhs<STAGE_ANY, true>}};
    const int64_t grid = c->sm.n_blocks;
    if (grid > 0)
        hipLaunchKernelGGL(kernels[stage_kind(p.io)][p.io.upd.u != nullptr], dim3(unsigned(grid)), dim3(kBlock), 0,
                           c->stream, p);
    HGDG_HIP(hipGetLastError());
}

}  // namespace

void simplex_rhs(hgdg_ctx* c, const StageIO& io) { launch_simplex(c, simplex_params(c, io)); }

// Threads per element, order by order: both candidates of an order are timed
// on the whole mesh (the other orders at their current choice) as one RK
// stage (u + a k -> k' on zero vectors of the operator's storage types; the
// kernel has no data-dependent branches), and the faster is kept. Orders with
// a fixed choice or without elements are not timed.
void simplex_tune(hgdg_ctx* c) {
    SimplexMesh& sm = c->sm;
    for (int g = 0; g < 4; ++g) {
        sm.tpe_variant[g] = sm.tpe_fixed[g] == simplex_tpe_alt(g + 1) ? 1 : 0;
        sm.tpe_ms[g][0] = sm.tpe_ms[g][1] = 0;
    }
    bool any = false;
    for (int g = 0; g < 4; ++g) any = any || (sm.tpe_fixed[g] == 0 && sm.group_start[g + 1] > sm.group_start[g]);
    if (!any) {
        simplex_schedule(c);
        return;
    }
    const bool mixed = c->op.precision == HGDG_PREC_MIXED_FP32;
    const size_t n = size_t(c->n_dof());
    DevBuf<double> u, k, out;
    u.alloc(n);
    k.alloc(n);
    out.alloc(n);
    HGDG_HIP(hipMemsetAsync(u.ptr, 0, n * sizeof(double), c->stream));
    HGDG_HIP(hipMemsetAsync(k.ptr, 0, n * sizeof(double), c->stream));
    StageIO io{};
    io.n_in = 2;
    io.in[0] = u.ptr;
    io.coef[0] = 1.0;
    io.in[1] = k.ptr;
    io.coef[1] = 0.5;
    io.in_f32 = mixed ? 2u : 0u;
    io.out = out.ptr;
    io.out_f32 = mixed ? 1 : 0;
    EventPair ev;
    constexpr int kReps = 10;
    for (int g = 0; g < 4; ++g) {
        if (sm.tpe_fixed[g] != 0 || sm.group_start[g + 1] == sm.group_start[g]) continue;
        for (int pass = 0; pass < 2; ++pass)
            for (int v = 0; v < 2; ++v) {
                sm.tpe_variant[g] = v;
                simplex_schedule(c);
                const SimplexParams p = simplex_params(c, io);
                for (int r = 0; r < 2; ++r) launch_simplex(c, p);
                HGDG_HIP(hipEventRecord(ev.e[0], c->stream));
                for (int r = 0; r < kReps; ++r) launch_simplex(c, p);
                HGDG_HIP(hipEventRecord(ev.e[1], c->stream));
                HGDG_HIP(hipEventSynchronize(ev.e[1]));
                float ms = 0;
                HGDG_HIP(hipEventElapsedTime(&ms, ev.e[0], ev.e[1]));
                const double t = double(ms) / kReps;
                if (pass == 0 || t < sm.tpe_ms[g][v]) sm.tpe_ms[g][v] = t;
            }
        sm.tpe_variant[g] = sm.tpe_ms[g][1] < sm.tpe_ms[g][0] ? 1 : 0;
    }
    simplex_schedule(c);
}

void simplex_state_diff(hgdg_ctx* c, const Vec& vx, const Vec& vy, double* l2, double* max_abs) {
    SimplexMesh& sm = c->sm;
    SimplexDiffParams p{};
    p.n_elem = c->n_elem;
    for (int g = 0; g < 5; ++g) {
        p.group_start[g] = sm.group_start[g];
        p.group_dof[g] = sm.group_dof[g];
    }
    group_blocks(sm, p.group_block);
    p.x = vx.ptr();
    p.y = vy.ptr();
    p.x_f32 = vx.is_f32;
    p.y_f32 = vy.is_f32;
    p.absdet = sm.d_absdet.ptr;
    p.tab = sm.d_tables.ptr;
    p.tix = sm.d_tab_index.ptr;
    const int grid = p.group_block[4];
    if (c->d_partial.n < size_t(2 * grid)) c->d_partial.alloc(size_t(2 * grid));
    p.partial = c->d_partial.ptr;
    hipLaunchKernelGGL(simplex_diff_norm, dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, p);
    HGDG_HIP(hipGetLastError());
    std::vector<double> h(size_t(2 * grid));
    HGDG_HIP(hipMemcpyAsync(h.data(), c->d_partial.ptr, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HGDG_HIP(hipStreamSynchronize(c->stream));
    double s = 0, mx = 0;
    for (int b = 0; b < grid; ++b) {
        s += h[2 * b];
        mx = std::max(mx, h[2 * b + 1]);
    }
    *l2 = std::sqrt(std::max(s, 0.0));
    *max_abs = mx;
}

void simplex_mass_apply(hgdg_ctx* c, Vec& v, bool inverse) {
    require(!v.is_f32, HGDG_ERR_UNSUPPORTED, "mass apply/solve needs a vector stored in FP64");
    require(c->n_fields == 4, HGDG_ERR_STATE, "the tetrahedral mass matrix belongs to the acoustic operator");
    SimplexMesh& sm = c->sm;
    SimplexMassParams p{};
    int32_t at = 0;
    for (int k = 0; k < 2; ++k)
        for (int q = 1; q <= kMaxSimplexOrder; ++q) {
            p.tab_off[k][q - 1] = at;
            at += tet_nb(q) * tet_nb(q);
        }
    require(sm.d_mass.n == size_t(at), HGDG_ERR_STATE, "set the operator before the mass matrix is used");
    p.elem_off = sm.d_elem_off.ptr;
    p.order = sm.d_order.ptr;
    p.tab = sm.d_mass.ptr;
    p.inverse = inverse ? 1 : 0;
    p.v = v.f64->ptr;
    p.absdet = sm.d_absdet.ptr;
    p.cinv = sm.d_geo.ptr + size_t(9) * c->n_elem;
    if (c->n_elem == 0) return;
    hipLaunchKernelGGL(simplex_mass, dim3(unsigned(c->n_elem)), dim3(64), 0, c->stream, p);
    HGDG_HIP(hipGetLastError());
}

namespace {

// hpGEM's rule for a requested order (AllGaussQuadratureRules::getRule).
void ref_tet_rule(int requested, std::vector<long double>& pts, std::vector<long double>& w) {
    require(requested >= 0 && requested <= kRefTetRuleMaxOrder, HGDG_ERR_UNSUPPORTED,
            "no tetrahedral rule of order " + std::to_string(requested));
    const RefTetRule& r = kRefTetRules[requested];
    pts.assign(r.pts, r.pts + 3 * r.n);
    w.assign(r.w, r.w + r.n);
}

// L2 projector of order p on the reference tetrahedron with hpGEM's element
// rule of order 2p+1 (as setInitialSolution integrates): R[i][q] = sum_j
// (M_ref^{-1})_{ij} w_q phi_j(xi_q), so that the coefficients of the
// projection of f on an affine element are sum_q R[i][q] f(x(xi_q)).
struct TetProjector {
    int nb = 0, nq = 0;
    std::vector<double> pts;  // [nq][3]
    std::vector<double> R;    // [nb][nq]
};

TetProjector tet_projector(int p) {
    TetProjector t;
    t.nb = tet_nb(p);
    std::vector<long double> pts, w;
    ref_tet_rule(2 * p + 1, pts, w);
    t.nq = int(w.size());
    const int nb = t.nb, nq = t.nq;
    std::vector<long double> phi(size_t(nq) * nb), grad(size_t(nb) * 3), M(size_t(nb) * nb, 0.0L);
    for (int q = 0; q < nq; ++q) {
        tet_basis(p, &pts[size_t(q) * 3], &phi[size_t(q) * nb], grad.data());
        for (int i = 0; i < nb; ++i)
            for (int j = 0; j < nb; ++j) M[size_t(i) * nb + j] += w[q] * phi[size_t(q) * nb + i] * phi[size_t(q) * nb + j];
    }
    // Gauss-Jordan inverse of the SPD reference mass matrix (long double)
    std::vector<long double> inv(size_t(nb) * nb, 0.0L);
    for (int i = 0; i < nb; ++i) inv[size_t(i) * nb + i] = 1.0L;
    for (int c = 0; c < nb; ++c) {
        int piv = c;
        for (int r = c + 1; r < nb; ++r)
            if (fabsl(M[size_t(r) * nb + c]) > fabsl(M[size_t(piv) * nb + c])) piv = r;
        for (int k = 0; k < nb; ++k) {
            std::swap(M[size_t(c) * nb + k], M[size_t(piv) * nb + k]);
            std::swap(inv[size_t(c) * nb + k], inv[size_t(piv) * nb + k]);
        }
        const long double d = M[size_t(c) * nb + c];
        for (int k = 0; k < nb; ++k) {
            M[size_t(c) * nb + k] /= d;
            inv[size_t(c) * nb + k] /= d;
        }
        for (int r = 0; r < nb; ++r) {
            if (r == c) continue;
            const long double f = M[size_t(r) * nb + c];
            if (f == 0.0L) continue;
            for (int k = 0; k < nb; ++k) {
                M[size_t(r) * nb + k] -= f * M[size_t(c) * nb + k];
                inv[size_t(r) * nb + k] -= f * inv[size_t(c) * nb + k];
            }
        }
    }
    t.pts.assign(pts.begin(), pts.end());
    t.R.assign(size_t(nb) * nq, 0.0);
    for (int i = 0; i < nb; ++i)
        for (int q = 0; q < nq; ++q) {
            long double s = 0;
            for (int j = 0; j < nb; ++j) s += inv[size_t(i) * nb + j] * w[q] * phi[size_t(q) * nb + j];
            t.R[size_t(i) * nq + q] = double(s);
        }
    return t;
}

}  // namespace

// L2 projection of sine modes or a Gaussian pulse (see tensor_project_device)
// into one field or all fields of a tetrahedral vector, computed on the host
// element by element and uploaded; the other fields keep their values.
namespace {

// The quadrature tables of the on-device projection and error norms, and the
// elements' affine maps, uploaded on first use.
SimplexQuadTab simplex_quad_tables(hgdg_ctx* c) {
    SimplexMesh& sm = c->sm;
    SimplexQuadTab t{};
    if (sm.qtab_index.empty()) {
        std::vector<double> tab;
        std::vector<int32_t> ix(40, 0);
        for (int p = 1; p <= kMaxSimplexOrder; ++p) {
            const int g = p - 1, nb = tet_nb(p);
            const TetProjector P = tet_projector(p);
            ix[g] = nb;
            ix[4 + g] = P.nq;
            ix[12 + g] = int32_t(tab.size());
            tab.insert(tab.end(), P.pts.begin(), P.pts.end());
            ix[16 + g] = int32_t(tab.size());
            tab.insert(tab.end(), P.R.begin(), P.R.end());
            std::vector<long double> phi(static_cast<size_t>(nb)), grad(static_cast<size_t>(nb) * 3);
            ix[20 + g] = int32_t(tab.size());
            for (int q = 0; q < P.nq; ++q) {
                const long double xi[3] = {P.pts[3 * q], P.pts[3 * q + 1], P.pts[3 * q + 2]};
                tet_basis(p, xi, phi.data(), grad.data());
                for (int i = 0; i < nb; ++i) tab.push_back(double(phi[i]));
            }
            std::vector<long double> pts, w;
            ref_tet_rule(2 * p + 2, pts, w);
            const int nq = int(w.size());
            ix[8 + g] = nq;
            ix[24 + g] = int32_t(tab.size());
            tab.insert(tab.end(), pts.begin(), pts.end());
            ix[28 + g] = int32_t(tab.size());
            tab.insert(tab.end(), w.begin(), w.end());
            ix[32 + g] = int32_t(tab.size());
            for (int q = 0; q < nq; ++q) {
                tet_basis(p, &pts[size_t(q) * 3], phi.data(), grad.data());
                for (int i = 0; i < nb; ++i) tab.push_back(double(phi[i]));
            }
            require(P.nq <= 64, HGDG_ERR_UNSUPPORTED, "projection rule with more than 64 points");
        }
        std::vector<double> xj(size_t(c->n_elem) * 12);
        for (int64_t d = 0; d < c->n_elem; ++d) {
            for (int r = 0; r < 3; ++r) xj[size_t(d) * 12 + r] = sm.x0[size_t(d) * 3 + r];
            for (int r = 0; r < 9; ++r) xj[size_t(d) * 12 + 3 + r] = sm.jac[size_t(d) * 9 + r];
        }
        sm.d_qtab.upload(tab, c->stream);
        sm.d_xj.upload(xj, c->stream);
        HGDG_HIP(hipStreamSynchronize(c->stream));  // the host vectors go out of scope
        sm.qtab_index = ix;
    }
    const std::vector<int32_t>& ix = sm.qtab_index;
    for (int g = 0; g < 4; ++g) {
        t.nb[g] = ix[g];
        t.nq_p[g] = ix[4 + g];
        t.nq_e[g] = ix[8 + g];
        t.pts_p[g] = ix[12 + g];
        t.R[g] = ix[16 + g];
        t.phi_p[g] = ix[20 + g];
        t.pts_e[g] = ix[24 + g];
        t.w_e[g] = ix[28 + g];
        t.phi_e[g] = ix[32 + g];
    }
    return t;
}

SimplexFnParams simplex_fn_params(hgdg_ctx* c, const Vec& v, int field, int n_modes, const double* amp,
                                  const double* k, const double* gauss, DevBuf<double>& d_modes) {
    SimplexMesh& sm = c->sm;
    SimplexFnParams p{};
    p.t = simplex_quad_tables(c);
    p.tab = sm.d_qtab.ptr;
    p.xj = sm.d_xj.ptr;
    p.elem_off = sm.d_elem_off.ptr;
    p.order = sm.d_order.ptr;
    p.n_fields = c->n_fields;
    p.field = field;
    p.u = v.ptr();
    p.u_f32 = v.is_f32;
    p.absdet = sm.d_absdet.ptr;
    if (gauss) {
        p.gaussian = 1;
        for (int q = 0; q < 5; ++q) p.g[q] = gauss[q];
    } else if (n_modes > 0) {
        std::vector<double> md(size_t(4) * n_modes);
        for (int m = 0; m < n_modes; ++m) {
            md[4 * m] = amp[m];
            for (int d = 0; d < 3; ++d) md[4 * m + 1 + d] = k[3 * m + d];
        }
        d_modes.upload(md, c->stream);
        HGDG_HIP(hipStreamSynchronize(c->stream));
        p.n_modes = n_modes;
        p.modes = d_modes.ptr;
    }
    return p;
}

}  // namespace

// L2 projection of sine modes or a Gaussian pulse, on the device.
void simplex_project(hgdg_ctx* c, Vec& v, int field, int n_modes, const double* amp, const double* k,
                     const double* gauss) {
    require(c->sm.d_order.n == size_t(c->n_elem), HGDG_ERR_STATE, "set the operator before projecting");
    DevBuf<double> d_modes;
    const SimplexFnParams p = simplex_fn_params(c, v, field, n_modes, amp, k, gauss, d_modes);
    if (c->n_elem > 0) hipLaunchKernelGGL(simplex_project, dim3(unsigned(c->n_elem)), dim3(64), 0, c->stream, p);
    HGDG_HIP(hipGetLastError());
    HGDG_HIP(hipStreamSynchronize(c->stream));  // before the modes table goes
}

// Error against f(x - shift) for sine modes f, as tensor_error_modes: L2 with
// hpGEM's tetrahedral rule of order 2p+2, maximum over the points of the
// element rule (order 2p+1), on the device; the per-element sums are added
// on the host in element order.
void simplex_error_modes(hgdg_ctx* c, const Vec& v, int field, int n_modes, const double* amp, const double* k,
                         const double* shift, double* l2, double* max_abs) {
    require(c->sm.d_order.n == size_t(c->n_elem), HGDG_ERR_STATE, "set the operator before computing errors");
    DevBuf<double> d_modes;
    SimplexFnParams p = simplex_fn_params(c, v, field, n_modes, amp, k, nullptr, d_modes);
    for (int d = 0; d < 3; ++d) p.shift[d] = shift[d];
    const int64_t ne = c->n_elem;
    if (c->d_partial.n < size_t(2 * ne)) c->d_partial.alloc(size_t(2 * ne));
    p.partial = c->d_partial.ptr;
    if (ne > 0) hipLaunchKernelGGL(simplex_error, dim3(unsigned(ne)), dim3(64), 0, c->stream, p);
    HGDG_HIP(hipGetLastError());
    std::vector<double> h(size_t(2 * ne));
    HGDG_HIP(hipMemcpyAsync(h.data(), c->d_partial.ptr, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HGDG_HIP(hipStreamSynchronize(c->stream));
    double sum = 0, mx = 0;
    for (int64_t d = 0; d < ne; ++d) {
        sum += h[2 * d];
        mx = std::max(mx, h[2 * d + 1]);
    }
    *l2 = std::sqrt(sum);
    *max_abs = mx;
}

}  // namespace hgdg
