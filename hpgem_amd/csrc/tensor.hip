// hgdg: MI355X (gfx950) explicit DG operator behind a C ABI.
//
// Tensor elements (squares, cubes). On an affine element with constant
// advection velocity a, hpGEM's stiffness, face and mass integrals
// (kernel/Base/HpgemAPILinear_Impl.h:131-139,250-288 with the integrands of
// tests/self/Basic/080AdvectionLinear_SelfTest.cpp:108-170) factor into 1D
// operators: with the basis psi_a(x) psi_b(y) psi_c(z), M = |J| M1 x M1 x M1,
// and after the block-diagonal inverse mass apply the weak form
//
//   k = sum_d ahat_d (D along d) w - sum_{faces (d,s)} (2s-1) ahat_d Mi(:,s) (x) T_{d,s}
//
// (ahat = J^{-1} a, D = M1^{-1} G1, Mi = M1^{-1}, T_{d,s} the upwind trace
// coefficients on face x_d = 2s-1) is evaluated in its integrated-by-parts
// ("lifting") form, which is the same number up to rounding:
//
//   k = -sum_d ahat_d (Dr along d) w - sum_{faces} (2s-1) ahat_d Mi(:,s) (x) (T_{d,s} - own_{d,s})
//
// with Dr = M1^{-1} K the exact 1D derivative matrix (K(a,b) = int psi_a psi_b')
// and own_{d,s} the element's own trace. Outflow faces drop out, and the face
// terms only carry jumps: no large terms cancel. The arithmetic is FP64 in both
// precisions, which differ in the storage of the stage derivatives. The 1D operators are built once on the host in long double by exact Gauss
// quadrature; each element needs its stage input, `dim` numbers of geometry
// and the traces of its inflow neighbours. One thread owns one x-pencil; an
// element's stage input sits in LDS for the other 1D contractions.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <limits>
#include <numeric>
#include <string>
#include <unordered_map>

#include "context.hpp"

namespace hgdg {

// Per-face upwind modes, 3 bits per tensor face f = 2d + s.
enum : uint32_t { MODE_NONE = 0, MODE_OWN = 1, MODE_NBR = 2, MODE_AVG = 3, MODE_HALF_OWN = 4 };

// A face's flux (2s-1) (c_n other - c_o own): the upper halves of the two
// coefficients' upper words (0, 1/2 and 1 need no more bits).
inline uint32_t face_coef(uint32_t mode, int s) {
    const uint32_t sign = s ? 0u : 0x8000u;
    const uint32_t one = 0x3ff0u, half = 0x3fe0u;
    const uint32_t cn = mode == MODE_NBR ? one : mode == MODE_AVG ? half : 0u;
    const uint32_t co = mode == MODE_NBR || mode == MODE_NONE ? one : mode == MODE_OWN ? 0u : half;
    return (cn ? (cn | sign) << 16 : 0u) | (co ? co | sign : 0u);
}

struct RhsParams {
    int64_t n_elem;
    StageIO io;
    const double* ahat;    // [dim][n_elem]
    const int32_t* nbr;    // [2 dim][n_elem]
    const uint32_t* mode;  // [n_elem]
    const uint2* face;     // [n_elem][2 dim]: the neighbour (the element itself where none is met) and face_coef()
    const double* Dr;      // [n1][n1] exact derivative matrix
    const double* Mi;      // [n1][n1] inverse 1D mass
};

template <int DIM, int N1>
struct Tensor {
    static constexpr int NB = N1 * N1 * (DIM == 3 ? N1 : 1);
    static constexpr int L = NB <= 4 ? 4 : NB <= 8 ? 8 : NB <= 16 ? 16 : NB <= 32 ? 32 : NB <= 64 ? 64 : NB <= 128 ? 128 : 256;
    static constexpr int EPB = kBlock / L;
};

// One thread owns one x-pencil of an element (the N1 coefficients with fixed
// y/z indices): the x-contraction and the x-face terms stay in registers, the
// y/z contractions read the other pencils of the element from LDS, and the
// y/z traces arrive as whole pencils of the neighbour.
template <int DIM, int N1>
struct Pencil {
    static constexpr int NP = DIM == 3 ? N1 * N1 : N1;  // pencils per element
    static constexpr int NB = NP * N1;                   // coefficients per element
    static constexpr int EPB = kBlock / NP;              // elements per block
};

// Pencils of one input vector as loaded (load_raw_n's form).
template <int NR, int N1>
__device__ __forceinline__ void load_raw(const void* v, bool f32, int64_t base, int64_t stride, double (&x)[NR][N1]) {
    if (f32) {
        const float* f = static_cast<const float*>(v) + base;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            float t[N1];
            if constexpr (N1 % 4 == 0) {
#pragma unroll
                for (int a = 0; a < N1; a += 4) {
                    const float4 q = *reinterpret_cast<const float4*>(f + r * stride + a);
                    t[a] = q.x; t[a + 1] = q.y; t[a + 2] = q.z; t[a + 3] = q.w;
                }
            } else if constexpr (N1 % 2 == 0) {
#pragma unroll
                for (int a = 0; a < N1; a += 2) {
                    const float2 q = *reinterpret_cast<const float2*>(f + r * stride + a);
                    t[a] = q.x; t[a + 1] = q.y;
                }
            } else {
#pragma unroll
                for (int a = 0; a < N1; ++a) t[a] = f[r * stride + a];
            }
#pragma unroll
            for (int a = 0; a < N1; ++a) x[r][a] = __hiloint2double(0, __float_as_int(t[a]));
        }
    } else {
        const double* d = static_cast<const double*>(v) + base;
#pragma unroll
        for (int r = 0; r < NR; ++r) load_run<N1>(d + r * stride, x[r]);
    }
}

// y += c x for NR pencils as load_raw left them
template <int NR, int N1>
__device__ __forceinline__ void add_raw(double c, const double (&x)[NR][N1], bool f32, double (&y)[NR][N1]) {
    if (f32) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int a = 0; a < N1; ++a) y[r][a] = fma(c, raw_value(x[r][a], true), y[r][a]);
    } else {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int a = 0; a < N1; ++a) y[r][a] = fma(c, x[r][a], y[r][a]);
    }
}

// Stage input of NR pencils at [base + r stride, + N1), in two halves:
// load_pencils issues the first two input vectors' loads (u, x), mix_pencils
// forms combine()'s sums from them in u and adds further inputs one by one.
template <int NR, int N1, int KIND = STAGE_ANY>
__device__ __forceinline__ void load_pencils(const StageIO& p, int64_t base, int64_t stride, double (&u)[NR][N1],
                                             double (&x)[NR][N1]) {
    load_raw<NR, N1>(p.in[0], KIND == STAGE_ANY && (p.in_f32 & 1u), base, stride, u);
    if (stage_two<KIND>(p)) load_raw<NR, N1>(p.in[1], stage_f32<KIND>(p, 1), base, stride, x);
}

template <int NR, int N1, int KIND = STAGE_ANY>
__device__ __forceinline__ void mix_two_pencils(const StageIO& p, double (&u)[NR][N1], const double (&x)[NR][N1]) {
    const bool u32 = KIND == STAGE_ANY && (p.in_f32 & 1u);
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int a = 0; a < N1; ++a) u[r][a] = p.coef[0] * raw_value(u[r][a], u32);
    if (stage_two<KIND>(p)) add_raw<NR, N1>(p.coef[1], x, stage_f32<KIND>(p, 1), u);
}

template <int NR, int N1, int KIND = STAGE_ANY>
__device__ __forceinline__ void mix_pencils(const StageIO& p, int64_t base, int64_t stride, double (&u)[NR][N1],
                                            double (&x)[NR][N1]) {
    mix_two_pencils<NR, N1, KIND>(p, u, x);
    if constexpr (stage_more<KIND>()) {
#pragma unroll 1
        for (int i = 2; i < p.n_in; ++i) {
            load_raw<NR, N1>(p.in[i], stage_f32<KIND>(p, i), base, stride, x);
            add_raw<NR, N1>(p.coef[i], x, stage_f32<KIND>(p, i), u);
        }
    }
}

// The fused RK update of NR pencils but for this kernel's own term, which is
// the last of its sum (RkUpdate::self): y = u + sum_{j != self} c_j x_j in
// rk_update_run's order. u and x are the stage input's first two vectors as
// load_raw left them (not yet mixed): the update reads those two again, so
// they are taken from registers; the first two other terms are loaded
// together, further ones one by one.
template <int NR, int N1>
__device__ __forceinline__ void update_partial(const StageIO& p, int64_t base, int64_t stride,
                                               const double (&u)[NR][N1], const double (&x)[NR][N1],
                                               double (&y)[NR][N1]) {
    const RkUpdate& q = p.upd;
    double t[2][NR][N1];
    auto from_x = [&](int j) { return p.n_in > 1 && q.x[j] == p.in[1]; };
    auto fetch = [&](int j, double (&d)[NR][N1]) {
        if (j < q.n_x && j != q.self && !from_x(j)) load_raw<NR, N1>(q.x[j], (q.x_f32 >> j) & 1u, base, stride, d);
    };
    auto add = [&](int j, const double (&d)[NR][N1]) {
        if (j >= q.n_x || j == q.self) return;
        if (from_x(j)) add_raw<NR, N1>(q.c[j], x, p.in_f32 & 2u, y);
        else add_raw<NR, N1>(q.c[j], d, (q.x_f32 >> j) & 1u, y);
    };
    fetch(0, t[0]);
    fetch(1, t[1]);
    if (q.u == p.in[0]) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int a = 0; a < N1; ++a) y[r][a] = u[r][a];
    } else {
        load_raw<NR, N1>(q.u, false, base, stride, y);
    }
    add(0, t[0]);
    add(1, t[1]);
#pragma unroll
    for (int j = 2; j < kMaxIn; ++j) {
        if (j >= q.n_x) break;
        fetch(j, t[0]);
        add(j, t[0]);
    }
}

// The rest of that update: the own term (k as stored), then y_new.
template <int N1>
__device__ __forceinline__ void update_store(const RkUpdate& q, int64_t o, const double (&k)[N1], double (&y)[N1]) {
    if (q.self >= 0) {
#pragma unroll
        for (int a = 0; a < N1; ++a) y[a] = fma(q.c[q.self], k[a], y[a]);
    }
    if constexpr (N1 % 2 == 0) {
#pragma unroll
        for (int a = 0; a < N1; a += 2) *reinterpret_cast<double2*>(q.y_new + o + a) = make_double2(y[a], y[a + 1]);
    } else {
#pragma unroll
        for (int a = 0; a < N1; ++a) q.y_new[o + a] = y[a];
    }
}

// The output pencil at o, in the output's storage type; v becomes the values
// as stored.
template <int N1>
__device__ __forceinline__ void store_pencil(const StageIO& p, int64_t o, double (&v)[N1]) {
    if (p.out_f32) {
        float* out = static_cast<float*>(p.out) + o;
        float f[N1];
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            f[a] = float(v[a]);
            v[a] = double(f[a]);
        }
        if constexpr (N1 % 4 == 0) {
#pragma unroll
            for (int a = 0; a < N1; a += 4)
                *reinterpret_cast<float4*>(out + a) = make_float4(f[a], f[a + 1], f[a + 2], f[a + 3]);
        } else if constexpr (N1 % 2 == 0) {
#pragma unroll
            for (int a = 0; a < N1; a += 2) *reinterpret_cast<float2*>(out + a) = make_float2(f[a], f[a + 1]);
        } else {
#pragma unroll
            for (int a = 0; a < N1; ++a) out[a] = f[a];
        }
    } else {
        double* out = static_cast<double*>(p.out) + o;
        if constexpr (N1 % 2 == 0) {
#pragma unroll
            for (int a = 0; a < N1; a += 2) *reinterpret_cast<double2*>(out + a) = make_double2(v[a], v[a + 1]);
        } else {
#pragma unroll
            for (int a = 0; a < N1; ++a) out[a] = v[a];
        }
    }
}

// A neighbour is met only where the flux needs it; F = (2s-1) times the jump
// (other - own), halved or without the other side as the mode says, which the
// 1D operator lifts: the terms -(2s-1) ahat_d Mi(idx_d, s) (T_{d,s} - own_{d,s}).
__device__ __forceinline__ bool face_met(uint32_t m) { return m == MODE_NBR || m == MODE_AVG; }
__device__ __forceinline__ double face_flux(uint32_t m, int s, double own, double other) {
    const double h = m == MODE_NONE || m == MODE_NBR ? 1.0 : 0.5;
    return m == MODE_OWN ? 0.0 : (s ? h : -h) * (other - own);
}

__device__ __forceinline__ void face_coef_values(uint32_t c, double& cn, double& co) {
    cn = __hiloint2double(int(c & 0xffff0000u), 0);
    co = __hiloint2double(int(c << 16), 0);
}

// The arithmetic of one pencil, shared by every kernel variant so that they
// agree bit for bit: per direction the one-dimensional operator, its volume
// part here (x with its faces' fluxes fx), y and z faces by advection_face;
// then minus ahat_d times each, summed. Row i of s_row: Dr(i, :), Mi(i, 0..1).
template <int N1>
__device__ __forceinline__ void advection_rows(const RhsParams& p, double* s_row) {
    static_assert(N1 * (N1 + 2) <= 64, "a wavefront's threads");
    const int i = threadIdx.x / (N1 + 2), j = threadIdx.x % (N1 + 2);
    if (i < N1) s_row[threadIdx.x] = j < N1 ? p.Dr[i * N1 + j] : p.Mi[i * N1 + j - N1];
}

template <int DIM, int N1>
__device__ __forceinline__ void advection_volume(const RhsParams& p, const double (&w)[N1], const double (&fx)[2],
                                                 const double* sw, const double* s_row, int ib, int ic,
                                                 double (&t)[DIM][N1]) {
#pragma unroll
    for (int a = 0; a < N1; ++a) {
        double x = 0.0;
#pragma unroll
        for (int j = 0; j < N1; ++j) x = fma(p.Dr[a * N1 + j], w[j], x);
#pragma unroll
        for (int s = 0; s < 2; ++s) x = fma(p.Mi[a * N1 + s], fx[s], x);
        t[0][a] = x;
    }
#pragma unroll
    for (int d = 1; d < DIM; ++d) {
#pragma unroll
        for (int a = 0; a < N1; ++a) t[d][a] = 0.0;
#pragma unroll
        for (int j = 0; j < N1; ++j) {
            const double dr = s_row[(d == 1 ? ib : ic) * (N1 + 2) + j];
            const double* row = sw + (d == 1 ? j + N1 * ic : ib + N1 * j) * N1;
#pragma unroll
            for (int a = 0; a < N1; ++a) t[d][a] = fma(dr, row[a], t[d][a]);
        }
    }
}

template <int N1>
__device__ __forceinline__ void advection_face(const double* s_row, int my, int s, const double* flux,
                                               double (&t)[N1]) {
    const double mi = s_row[my * (N1 + 2) + N1 + s];
#pragma unroll
    for (int a = 0; a < N1; ++a) t[a] = fma(mi, flux[a], t[a]);
}

template <int DIM, int N1>
__device__ __forceinline__ void advection_result(const double (&ah)[DIM], const double (&t)[DIM][N1],
                                                 double (&k)[N1]) {
#pragma unroll
    for (int a = 0; a < N1; ++a) {
        k[a] = -ah[0] * t[0][a];
#pragma unroll
        for (int d = 1; d < DIM; ++d) k[a] = fma(-ah[d], t[d][a], k[a]);
    }
}

// `tiles` consecutive tiles of EPB elements, from tile t0 * tiles on; one
// thread per x-pencil, and the same threads once more as one per y/z face
// pencil (4 N1 an element in 3D, 2 in 2D), so that a face's trace is loaded and
// its flux formed once and shared through LDS. TILED: the next tile's face
// data and own pencils are loaded while this tile is computed, and a launch
// can be sized to fill the GPU in one round. UPD: with the RK update of a
// step's last stage, all of its sum but the own term formed from the stage
// input's loads. Threads without a pencil or face work on the tile's first and
// store nothing.
//
// Bound by instruction issue and by the two loads in a row (face data, then the
// neighbours' values), which a launch of one or two rounds of workgroups cannot
// hide; hence no decisions per face (an outflow face meets the element itself
// with coefficient 0), FP64 arithmetic for FP32 stage values too (it issues at
// the FP32 rate and needs no compensated sums) and a kernel per StageKind. One
// stage of RK4 (us; before: every pencil of a line loaded and lifted each face
// trace itself): 32^3 p = 3 14.1 -> 12.2 (4.3 TB/s), with FP32 stage values
// 11.6 -> 9.4; 61 x 47 x 53 p = 2 26.6 -> 23.9 and 22.5 -> 20.3; 25 x 27 x 26
// p = 4 17.2 -> 14.5; 301 x 257 p = 3 7.4 -> 6.8. The whole step, its last
// stage with the update: 66.4 -> 55.6, 54.5 -> 46.5, 115.6 -> 103.2, 96.8 ->
// 92.4, 76.4 -> 67.0, 37.3 -> 35.2. Reading and writing in memory order through
// LDS instead of by pencil costs more instructions than it saves (32^3 p = 3
// 13.3, 61 x 47 x 53 p = 2 27.2).
template <int DIM, int N1, int KIND, bool UPD, bool TILED>
__device__ __forceinline__ void advection_tiles(const RhsParams& p, int64_t t0, int tiles) {
    using S = Pencil<DIM, N1>;
    constexpr int NB = S::NB, EPB = S::EPB, NF = 2 * DIM;
    constexpr int NQ = 2 * (DIM - 1) * (DIM == 3 ? N1 : 1);  // y/z face pencils of an element
    constexpr int NI = (EPB * NQ + kBlock - 1) / kBlock;     // of a thread
    __shared__ double s_w[EPB * NB];       // stage input
    __shared__ double s_f[EPB * NQ * N1];  // fluxes
    __shared__ double s_row[N1 * (N1 + 2)];
    const int tid = threadIdx.x;
    const int64_t E = p.n_elem;
    const int64_t first = TILED ? t0 * tiles : t0;
    int64_t end = first + 1;
    if (TILED) {
        const int64_t n_tiles = (E + EPB - 1) / EPB;
        end = first + tiles < n_tiles ? first + tiles : n_tiles;
        if (first >= end) return;
    }
    auto item = [&](int k) { return (k + 1) * kBlock <= EPB * NQ || tid + k * kBlock < EPB * NQ; };

    struct Loads {
        uint2 fx[2], fq[NI];
        double ah[DIM];
        double w[1][N1], x[1][N1];
    };
    auto fetch = [&](int64_t t, Loads& l) {
        const int64_t e0 = t * EPB;
        const int n = E - e0 < EPB ? int(E - e0) : EPB;
        const uint2* face = p.face + e0 * NF;
#pragma unroll
        for (int k = 0; k < NI; ++k)
            if (item(k)) {
                const int q = tid + k * kBlock, el = q / NQ < n ? q / NQ : 0;
                l.fq[k] = face[el * NF + 2 + (DIM == 3 ? q % NQ / N1 : q % NQ)];
            }
        const int own = tid < n * S::NP ? tid : 0, le = own / S::NP;
#pragma unroll
        for (int s = 0; s < 2; ++s) l.fx[s] = face[le * NF + s];
        load_pencils<1, N1, KIND>(p.io, e0 * NB + own * N1, 0, l.w, l.x);
#pragma unroll
        for (int d = 0; d < DIM; ++d) l.ah[d] = p.ahat[d * E + e0 + le];
    };
    Loads l;
    fetch(first, l);
    advection_rows<N1>(p, s_row);

    for (int64_t t = first; t < end; ++t) {
        const int64_t e0 = t * EPB;
        const int n = E - e0 < EPB ? int(E - e0) : EPB;
        const bool active = tid < n * S::NP;
        const int own = active ? tid : 0, le = own / S::NP, pc = own % S::NP;
        const int ib = pc % N1, ic = DIM == 3 ? pc / N1 : 0;
        const int64_t base = e0 * NB + own * N1;
        // ---- the neighbours' face pencils and x traces (of the first two inputs)
        int64_t at[NI], atx[2];
        int lx[2];
        double o[NI][1][N1], o1[NI][1][N1], ox[2], ox1[2], cq[NI][2], cx[2][2];
#pragma unroll
        for (int k = 0; k < NI; ++k)
            if (item(k)) {
                const int q = tid + k * kBlock, fi = DIM == 3 ? q % NQ / N1 : q % NQ, j = DIM == 3 ? q % N1 : 0;
                at[k] = int64_t(l.fq[k].x) * NB + (fi / 2 ? j + N1 * (1 - fi % 2) : (1 - fi % 2) + N1 * j) * N1;
                load_pencils<1, N1, KIND>(p.io, at[k], 0, o[k], o1[k]);
                face_coef_values(l.fq[k].y, cq[k][0], cq[k][1]);
            }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int64_t ln = int64_t(l.fx[s].x) - e0;
            lx[s] = ln >= 0 && ln < n ? int(ln) * NB + pc * N1 + (1 - s) : -1;  // in this block's LDS
            atx[s] = int64_t(l.fx[s].x) * NB + pc * N1 + (1 - s);
            if (lx[s] < 0) {
                const int64_t a1[1] = {atx[s]};
                double v[1], v1[1];
                load_two<KIND>(p.io, a1, v, v1);
                ox[s] = v[0];
                ox1[s] = v1[0];
            }
            face_coef_values(l.fx[s].y, cx[s][0], cx[s][1]);
        }
        double y[1][N1];
        if constexpr (UPD) update_partial<1, N1>(p.io, base, 0, l.w, l.x, y);
        // ---- the sums; further inputs two at a time
        mix_two_pencils<1, N1, KIND>(p.io, l.w, l.x);
#pragma unroll
        for (int k = 0; k < NI; ++k)
            if (item(k)) mix_two_pencils<1, N1, KIND>(p.io, o[k], o1[k]);
#pragma unroll
        for (int s = 0; s < 2; ++s)
            if (lx[s] < 0) {
                double v[1][1] = {{ox[s]}}, v1[1][1] = {{ox1[s]}};
                mix_two_pencils<1, 1, KIND>(p.io, v, v1);
                ox[s] = v[0][0];
            }
        constexpr int kStep = 2;
        if constexpr (stage_more<KIND>()) {
#pragma unroll 1
            for (int i = 2; i < p.io.n_in; i += kStep) {
                double a[kStep][1][N1], b[kStep][NI][1][N1], g[kStep][2][1][1];
#pragma unroll
                for (int h = 0; h < kStep; ++h) {
                    if (h > 0 && i + h >= p.io.n_in) break;
                    const void* in = p.io.in[i + h];
                    const bool f = stage_f32<KIND>(p.io, i + h);
                    load_raw<1, N1>(in, f, base, 0, a[h]);
#pragma unroll
                    for (int k = 0; k < NI; ++k)
                        if (item(k)) load_raw<1, N1>(in, f, at[k], 0, b[h][k]);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (lx[s] < 0) load_raw<1, 1>(in, f, atx[s], 0, g[h][s]);
                }
#pragma unroll
                for (int h = 0; h < kStep; ++h) {
                    if (h > 0 && i + h >= p.io.n_in) break;
                    const double c = p.io.coef[i + h];
                    const bool f = stage_f32<KIND>(p.io, i + h);
                    add_raw<1, N1>(c, a[h], f, l.w);
#pragma unroll
                    for (int k = 0; k < NI; ++k)
                        if (item(k)) add_raw<1, N1>(c, b[h][k], f, o[k]);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        if (lx[s] < 0) {
                            double v[1][1] = {{ox[s]}};
                            add_raw<1, 1>(c, g[h][s], f, v);
                            ox[s] = v[0][0];
                        }
                }
            }
        }
        double w[N1], ah[DIM];
#pragma unroll
        for (int a = 0; a < N1; ++a) w[a] = l.w[0][a];
#pragma unroll
        for (int d = 0; d < DIM; ++d) ah[d] = l.ah[d];
        if (TILED && t != first) __syncthreads();  // the previous tile's readers are done
        if (EPB * S::NP == kBlock || tid < EPB * S::NP) {
#pragma unroll
            for (int a = 0; a < N1; ++a) s_w[tid * N1 + a] = w[a];
        }
        __syncthreads();
        if (TILED && t + 1 < end) fetch(t + 1, l);

        // ---- each face pencil's flux, and the volume terms
#pragma unroll
        for (int k = 0; k < NI; ++k)
            if (item(k)) {
                const int q = tid + k * kBlock, fi = DIM == 3 ? q % NQ / N1 : q % NQ, j = DIM == 3 ? q % N1 : 0;
                const double* oq = s_w + q / NQ * NB + (fi / 2 ? j + N1 * (fi % 2) : fi % 2 + N1 * j) * N1;
#pragma unroll
                for (int a = 0; a < N1; ++a) s_f[q * N1 + a] = fma(cq[k][0], o[k][0][a], -(cq[k][1] * oq[a]));
            }
        double tt[DIM][N1], fx[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (lx[s] >= 0) ox[s] = s_w[lx[s]];
            fx[s] = fma(cx[s][0], ox[s], -(cx[s][1] * w[s]));
        }
        advection_volume<DIM, N1>(p, w, fx, s_w + le * NB, s_row, ib, ic, tt);
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
            for (int a = 0; a < N1; ++a) form_here(tt[d][a]);
        __syncthreads();
#pragma unroll
        for (int f = 2; f < NF; ++f) {
            const int q = le * NQ + (DIM == 3 ? (f - 2) * N1 + (f / 2 == 1 ? ic : ib) : f - 2);
            advection_face<N1>(s_row, f / 2 == 1 ? ib : ic, f % 2, s_f + q * N1, tt[f / 2]);
        }
        double k[N1];
        advection_result<DIM, N1>(ah, tt, k);
        if (active) {
            store_pencil<N1>(p.io, base, k);
            if constexpr (UPD) update_store<N1>(p.io.upd, base, k, y[0]);
        }
    }
}

// Whole RK steps of a small advection mesh in one workgroup: the solution,
// the stage input, every stage derivative and the per-element face data stay
// in LDS for all n_steps steps, with workgroup barriers between the phases,
// so one launch replaces 5 n_steps launches (meshes this small are bound by
// launch latency, not by HBM). The arithmetic is the graph path's, operation
// for operation: the stage input as combine() forms it, the RHS by the same
// sums with the neighbour traces read from LDS, the update as
// multi_axpy forms it; results are bitwise the same (tested).
// The one workgroup: 16 wavefronts where the kernel fits in 128 registers,
// else 8 (256 registers).
template <int DIM, int N1>
constexpr int rk_tiny_block() {
    return (DIM == 2 ? N1 <= 4 : N1 <= 3) ? 1024 : 512;
}

struct RkTinyParams {
    RhsParams rhs;          // geometry, tables; io unused
    double* u;              // [n_dof] solution (read, then written after the last step)
    void* k[kMaxIn];        // stage vectors (written with the last step's derivatives)
    int32_t stages;
    int32_t n_steps;
    double ca[kMaxIn * kMaxIn];  // dt a_ij, row i
    double cb[kMaxIn];           // dt b_j
    uint32_t amask[kMaxIn];      // bit j of row i: a_ij != 0 (the graph path skips zero entries)
    uint32_t bmask;              // bit j: b_j != 0
};

// T: the stage derivatives' storage.
template <int DIM, int N1, typename T>
__global__ __launch_bounds__((rk_tiny_block<DIM, N1>())) void tensor_advection_rk_tiny(const RkTinyParams p) {
    constexpr int kTinyBlock = rk_tiny_block<DIM, N1>();
    using S = Pencil<DIM, N1>;
    extern __shared__ __align__(16) double dyn[];
    __shared__ double s_row[N1 * (N1 + 2)];
    const int64_t E = p.rhs.n_elem, n = E * S::NB;
    const int st = p.stages;
    double* su = dyn;                                  // [n] solution
    double* sw = su + n;                               // [n] stage input
    uint32_t* smd = reinterpret_cast<uint32_t*>(sw + n);  // [E] upwind modes
    int32_t* snb = reinterpret_cast<int32_t*>(smd + E);   // [2 DIM][E] neighbours
    double* sah = reinterpret_cast<double*>(snb + 2 * DIM * E + ((E * (1 + 2 * DIM)) & 1));  // [DIM][E]
    T* sk = reinterpret_cast<T*>(sah + DIM * E);       // [stages][n] stage derivatives
    advection_rows<N1>(p.rhs, s_row);
    for (int64_t i = threadIdx.x; i < n; i += kTinyBlock) su[i] = p.u[i];
    for (int64_t e = threadIdx.x; e < E; e += kTinyBlock) {
        smd[e] = p.rhs.mode[e];
#pragma unroll
        for (int d = 0; d < DIM; ++d) sah[d * E + e] = p.rhs.ahat[d * E + e];
#pragma unroll
        for (int f = 0; f < 2 * DIM; ++f) snb[f * E + e] = p.rhs.nbr[f * E + e];
    }
    __syncthreads();
    for (int step = 0; step < p.n_steps; ++step) {
        for (int i = 0; i < st; ++i) {
            // stage input: 1 * u, then + (dt a_ij) k_j in order of j
            for (int64_t q = threadIdx.x; q < n; q += kTinyBlock) {
                double v = 1.0 * su[q];
                for (int j = 0; j < i; ++j)
                    if ((p.amask[i] >> j) & 1u) v = fma(p.ca[i * kMaxIn + j], double(sk[int64_t(j) * n + q]), v);
                sw[q] = v;
            }
            __syncthreads();
            for (int64_t q = threadIdx.x; q < E * S::NP; q += kTinyBlock) {
                const int64_t e = q / S::NP;
                const int pc = int(q % S::NP);
                double w[N1];
#pragma unroll
                for (int a = 0; a < N1; ++a) w[a] = sw[e * S::NB + pc * N1 + a];
                double ah[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) ah[d] = sah[d * E + e];
                const uint32_t md = smd[e];
                const double* we = sw + e * S::NB;
                const int ib = pc % N1, ic = DIM == 3 ? pc / N1 : 0;
                double fx[2], t[DIM][N1];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint32_t m = (md >> (3 * s)) & 7u;
                    const double o = face_met(m) ? sw[int64_t(snb[s * E + e]) * S::NB + pc * N1 + (1 - s)] : 0.0;
                    fx[s] = face_flux(m, s, w[s], o);
                }
                advection_volume<DIM, N1>(p.rhs, w, fx, we, s_row, ib, ic, t);
#pragma unroll
                for (int f = 2; f < 2 * DIM; ++f) {
                    const uint32_t m = (md >> (3 * f)) & 7u;
                    const int s = f % 2, k = f / 2 == 1 ? ic : ib;
                    const int own = f / 2 == 1 ? s + N1 * k : k + N1 * s, nbr = f / 2 == 1 ? (1 - s) + N1 * k : k + N1 * (1 - s);
                    double flux[N1];
                    if (face_met(m)) {
                        const double* o = sw + int64_t(snb[f * E + e]) * S::NB + nbr * N1;
#pragma unroll
                        for (int a = 0; a < N1; ++a) flux[a] = face_flux(m, s, we[own * N1 + a], o[a]);
                    } else {
#pragma unroll
                        for (int a = 0; a < N1; ++a) flux[a] = face_flux(m, s, we[own * N1 + a], 0.0);
                    }
                    advection_face<N1>(s_row, f / 2 == 1 ? ib : ic, s, flux, t[f / 2]);
                }
                double kv[N1];
                advection_result<DIM, N1>(ah, t, kv);
#pragma unroll
                for (int a = 0; a < N1; ++a) sk[int64_t(i) * n + e * S::NB + pc * N1 + a] = T(kv[a]);
            }
            __syncthreads();
        }
        // update: u + (dt b_j) k_j in order of j
        for (int64_t q = threadIdx.x; q < n; q += kTinyBlock) {
            double y = su[q];
            for (int j = 0; j < st; ++j)
                if ((p.bmask >> j) & 1u) y = fma(p.cb[j], double(sk[int64_t(j) * n + q]), y);
            su[q] = y;
        }
        __syncthreads();
    }
    for (int64_t q = threadIdx.x; q < n; q += kTinyBlock) {
        p.u[q] = su[q];
        for (int j = 0; j < st; ++j) static_cast<T*>(p.k[j])[q] = sk[int64_t(j) * n + q];
    }
}

// The same for meshes with at most one x-pencil a thread: the thread keeps its
// pencil of the solution, the update's running sum and what it needs of the
// faces and operators in registers for all steps, and the stage input goes
// through two LDS buffers in turn, so that a stage has one barrier (a buffer is
// written again only after the barrier of the other one, which every reader
// passes later). The last stage derivative is a register too; older ones, where
// the tableau uses them, are the thread's own values in LDS.
// Bound by latency (16^2 p = 2: 12 wavefronts' LDS reads and multiply-adds
// between barriers on one CU). A step of RK4, us, by the kernel above and here:
// 16^2 p = 2 7.2 and 4.6, 20^2 p = 1 6.0 and 3.1, 10^2 p = 4 10.9 and 6.9, 3^3
// cells of p = 3 10.3 and 6.1, 3^3 of p = 1 4.5 and 2.2 (a wavefront without work costs
// as much as one with: only as many are launched as there are pencils). Reading
// the next stage's tableau entries ahead gained nothing (5.3 against 5.1).
// Threads: as many as leave every value a register; none for 3D p = 4 and up,
// where 512 threads spill (3 x 3 x 2 cells of p = 4: 14.5 us a step, no gain).
template <int DIM, int N1>
constexpr int rk_pencil_block() {
    return DIM == 2 ? (N1 <= 3 ? 1024 : 512) : (N1 <= 2 ? 1024 : N1 <= 4 ? 512 : 0);
}

template <int DIM, int N1, typename T>
__global__ __launch_bounds__((rk_pencil_block<DIM, N1>())) void tensor_advection_rk_pencil(const RkTinyParams p) {
    using S = Pencil<DIM, N1>;
    constexpr int NF = 2 * DIM;
    extern __shared__ __align__(16) double dyn[];
    const int n = int(p.rhs.n_elem) * S::NB, st = p.stages;
    T* sk = reinterpret_cast<T*>(dyn + 2 * n);  // [stages][n]
    const bool active = threadIdx.x < unsigned(p.rhs.n_elem) * S::NP;
    const int q = active ? int(threadIdx.x) : 0, e = q / S::NP, pc = q % S::NP;
    const int ib = pc % N1, ic = DIM == 3 ? pc / N1 : 0;
    // face f: where its neighbour's values start (x: the one value), and the flux's coefficients
    int at[NF];
    uint32_t coef[NF];
    double ah[DIM];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const uint2 rec = p.rhs.face[e * NF + f];
        const int s = f % 2;
        const int pen = f < 2 ? pc : f < 4 ? (1 - s) + N1 * ic : ib + N1 * (1 - s);
        at[f] = int(rec.x) * S::NB + pen * N1 + (f < 2 ? 1 - s : 0);
        coef[f] = rec.y;
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) ah[d] = p.rhs.ahat[d * p.rhs.n_elem + e];
    // the rows of the operators of this pencil's y and z index: registers where
    // they leave no value to spill (2D up to p = 2), else LDS
    constexpr bool kRows = DIM == 2 && N1 <= 3;
    __shared__ double s_row[N1 * (N1 + 2)];
    advection_rows<N1>(p.rhs, s_row);
    double regs[kRows ? N1 + 2 : 1];
    if constexpr (kRows) {
#pragma unroll
        for (int j = 0; j < N1 + 2; ++j) regs[j] = j < N1 ? p.rhs.Dr[ib * N1 + j] : p.rhs.Mi[ib * N1 + j - N1];
    }
    auto row_of = [&](int d, int j) {
        if constexpr (kRows) return regs[j];
        else return s_row[(d == 1 ? ib : ic) * (N1 + 2) + j];
    };
    double u[N1], kl[N1];
#pragma unroll
    for (int a = 0; a < N1; ++a) {
        u[a] = p.u[q * N1 + a];
        kl[a] = 0.0;
    }
    int buf = 0;
    for (int step = 0; step < p.n_steps; ++step) {
        double y[N1];
#pragma unroll
        for (int a = 0; a < N1; ++a) y[a] = u[a];
        for (int i = 0; i < st; ++i) {
            double w[N1];
#pragma unroll
            for (int a = 0; a < N1; ++a) w[a] = 1.0 * u[a];
            for (uint32_t m = p.amask[i]; m != 0; m &= m - 1) {
                const int j = __builtin_ctz(m);
                const double c = p.ca[i * kMaxIn + j];
                if (j == i - 1) {
#pragma unroll
                    for (int a = 0; a < N1; ++a) w[a] = fma(c, kl[a], w[a]);
                } else {
#pragma unroll
                    for (int a = 0; a < N1; ++a) w[a] = fma(c, double(sk[j * n + q * N1 + a]), w[a]);
                }
            }
            double* sw = dyn + buf * n;
            buf ^= 1;
            if (active) {
#pragma unroll
                for (int a = 0; a < N1; ++a) sw[q * N1 + a] = w[a];
            }
            __syncthreads();
            double fx[2], t[DIM][N1], cn, co;
            auto face = [&](int f) {
                if constexpr (!kRows) asm volatile("" : "+v"(coef[f]));  // not unpacked for all stages at once
                face_coef_values(coef[f], cn, co);
            };
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                face(s);
                fx[s] = fma(cn, sw[at[s]], -(co * w[s]));
            }
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                double x = 0.0;
#pragma unroll
                for (int j = 0; j < N1; ++j) x = fma(p.rhs.Dr[a * N1 + j], w[j], x);
#pragma unroll
                for (int s = 0; s < 2; ++s) x = fma(p.rhs.Mi[a * N1 + s], fx[s], x);
                t[0][a] = x;
            }
#pragma unroll
            for (int d = 1; d < DIM; ++d) {
                double own[2][N1];  // the element's own traces: rows 0 and 1 of the line
#pragma unroll
                for (int a = 0; a < N1; ++a) t[d][a] = 0.0;
#pragma unroll
                for (int j = 0; j < N1; ++j) {
                    const double* row = sw + e * S::NB + (d == 1 ? j + N1 * ic : ib + N1 * j) * N1;
#pragma unroll
                    for (int a = 0; a < N1; ++a) {
                        const double v = row[a];
                        if (j < 2) own[j][a] = v;
                        t[d][a] = fma(row_of(d, j), v, t[d][a]);
                    }
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    face(2 * d + s);
#pragma unroll
                    for (int a = 0; a < N1; ++a) {
                        const double flux = fma(cn, sw[at[2 * d + s] + a], -(co * own[s][a]));
                        t[d][a] = fma(row_of(d, N1 + s), flux, t[d][a]);
                    }
                }
            }
            advection_result<DIM, N1>(ah, t, kl);
            const bool used = (p.bmask >> i) & 1u;
            const double cb = p.cb[i];
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                const T v = T(kl[a]);
                if (active) sk[i * n + q * N1 + a] = v;
                kl[a] = double(v);
                if (used) y[a] = fma(cb, kl[a], y[a]);
            }
        }
#pragma unroll
        for (int a = 0; a < N1; ++a) u[a] = y[a];
    }
    if (active) {
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            p.u[q * N1 + a] = u[a];
            for (int j = 0; j < st; ++j) static_cast<T*>(p.k[j])[q * N1 + a] = sk[j * n + q * N1 + a];
        }
    }
}

// UPD: the RK update fused into this (last) stage, StageIO::upd.
template <int DIM, int N1, int KIND, bool UPD>
__global__ __launch_bounds__(kBlock) void tensor_advection_rhs(const RhsParams p) {
    advection_tiles<DIM, N1, KIND, UPD, false>(p, xcd_block(blockIdx.x, gridDim.x), 1);
}

template <int DIM, int N1, int KIND>
__global__ __launch_bounds__(kBlock) void tensor_advection_rhs_tiled(const RhsParams p, int tiles) {
    advection_tiles<DIM, N1, KIND, false, true>(p, xcd_block(blockIdx.x, gridDim.x), tiles);
}

// Block b of a batched launch belongs to problem s with off[s] <= b < off[s+1].
__device__ __forceinline__ int find_problem(const int64_t* off, int n, int64_t b) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (off[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Many independent problems of one kind in one launch: every block runs the
// exact code of the single-problem kernel on its own problem's data (UPD:
// with each problem's fused RK update, StageIO::upd).
template <int DIM, int N1, bool UPD = false>
__global__ __launch_bounds__(kBlock) void tensor_advection_rhs_batched(const RhsParams* __restrict__ ps,
                                                                       const int64_t* __restrict__ off, int n) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);
    const int s = __builtin_amdgcn_readfirstlane(find_problem(off, n, b));
    advection_tiles<DIM, N1, STAGE_ANY, UPD, false>(ps[s], b - off[s], 1);
}

// Acoustic wave system on tensor elements (AcousticWaveLinear_Impl.h:102-283):
// fields v, s_1..s_dim stored field-major per element. With g_r = sum_d
// (J^{-1})_{r,d} s_d, the element's own J throughout, and per face (r, s)
//   F_v = -1/2 (2s-1) (g_r,own - sum_d (J^{-1})_{r,d} s_d,nbr),
//   F_s = -1/2 (2s-1) (v_own - v_nbr)
// on internal faces, F_v = -(2s-1) g_r,own and F_s = 0 on reflecting walls,
//   k_v   =             sum_r [ (Dr along r) g_r + sum_s Mi(:,s) (x) F_v(r,s) ]
//   k_s_d = (1/c_inv) sum_r (J^{-1})_{r,d} [ (Dr along r) v + sum_s Mi(:,s) (x) F_s(r,s) ].
// Both brackets are the same one-dimensional operator, applied to g_r and to
// v; the s fields are only combined from the second at the end. The
// arithmetic is FP64 in both precisions (an FP64 multiply-add issues at the
// FP32 rate here); the mixed path differs in the storage of its stage
// derivatives.
struct AcousticParams {
    int64_t n_elem;
    StageIO io;
    const double* jinv;   // [dim*dim][n_elem]: (J^{-1})_{r,d} at [(r dim + d) n_elem + e]
    const double* cinv;   // [n_elem]
    const int32_t* nbr;   // [2 dim][n_elem], -1 on walls
    const double* Dr;
    const double* Mi;
    const double* absdet;  // [n_elem] and
    const double* M1;      // the 1D mass: MASS only
    const int32_t* order;  // the workgroup of each place in the launch, or NULL: in turn (acoustic_order)
};

// One thread owns one x-pencil of an element with all its fields; v, g_y and
// g_z go to LDS for the y and z contractions, and each y or z face pencil's
// fluxes are formed once, by one of the element's threads (NQ face pencils),
// and shared through LDS. Nothing but an element's own threads meets at a
// barrier, so a workgroup is the smallest of 64, 128 and 256 threads that
// leaves at most one lane in sixteen idle: one wavefront where it can.
// Sums are explicit multiply-adds: every instance (with and without the
// update, batched) rounds alike.
// Bound by memory: 32^3 p = 3 in FP64 takes 44 us for 208 MB of vectors and
// geometry, 4.7 TB/s; with the z neighbours that come from memory again it is
// 254 MB at 5.8 TB/s (a copy of that size reaches 5.4 - 6.9). One lane per field
// and pencil, which applies the derivative of v once per s field and forms every
// face pencil's flux N1 times, took 104 us FP64 / 80 mixed there against 44 / 33
// (47 / 36 with the workgroups in plain order, see acoustic_order: so are the next
// figures); 30^3 p = 2 42 against 23, 23x19x21 p = 4 66 against 37 (FP64).
// kAhead: the first face pencil's neighbour values are loaded together with
// the own ones, one memory round trip less (32^3 p = 3 53 -> 47 us, 256^2
// p = 3 20.1 -> 17.7); at orders 4 and 5 in 3D, and with the update's terms
// held too, its registers cost as much as that gains (20^3 p = 5 60 -> 64 us).
// kTogether: of stages of three and more inputs, each is read at once for all
// that is loaded here, and for the x faces: one memory round trip for it, where
// pencils and faces summing their inputs each for itself take up to five. us
// with 3, 5 and 7 inputs by STAGE_ANY and so: 6x7x5 p = 1 6.1, 8.4 and 10.6,
// 6.0, 6.2 and 6.7; p = 2 6.9, 9.4 and 11.9, 6.1, 6.8 and 8.0; 40x30 p = 4 6.4,
// 8.3 and 10.3, 6.0, 6.2 and 6.6; 24^3 p = 3 34.8, 59.5 and 84.9, 33.8, 47.9 and
// 63.8. (At order 5 in 3D a SIMD has one wavefront in any case: kAhead there too.)
// kEarly: all of the update's sum but the own term is formed before the
// volume terms, from u and k as they are loaded anyway (RK4 step of 30^3 p = 2
// 107 -> 103 us, 256^2 p = 1 34.8 -> 32.3); at orders 4 and 5 the 4 N1 sums do
// not fit beside the rest (20^3 p = 5 276 -> 288 us), so there it comes last.
template <int DIM, int N1>
struct AcousticShape {
    static constexpr int NF = DIM + 1;
    static constexpr int NP = Pencil<DIM, N1>::NP;
    static constexpr int NB = Pencil<DIM, N1>::NB;
    static constexpr int NQ = 2 * (DIM - 1) * (DIM == 3 ? N1 : 1);
    static constexpr int THREADS = (64 % NP) * 16 <= 64 ? 64 : (128 % NP) * 16 <= 128 ? 128 : 256;
    static constexpr int EPB = THREADS / NP;
    // LDS strides (doubles) of a plane and an element: even orders' planes
    // are a multiple of the 64 banks' period apart without the padding
    static constexpr int PS = N1 * N1 + (N1 % 2 == 0 ? 2 : 0);
    static constexpr int ES = (DIM == 3 ? N1 : 1) * PS;
};

template <int DIM, int N1, int KIND, bool UPD, bool MASS = false>
__device__ __forceinline__ void acoustic_block(const AcousticParams& p, int64_t blk) {
    using S = AcousticShape<DIM, N1>;
    constexpr int NF = S::NF, NB = S::NB, NP = S::NP, NQ = S::NQ;
    __shared__ double s_v[S::EPB * S::ES];                  // v
    __shared__ double s_g[(DIM - 1) * S::EPB * S::ES];      // g_y, g_z
    __shared__ double s_f[S::EPB * NQ * 2 * N1];            // per y/z face pencil: F_v, F_s
    const int tid = threadIdx.x;
    const int le = tid / NP, pc = tid % NP;
    const int64_t e = blk * S::EPB + le;
    const bool active = (le < S::EPB) && (e < p.n_elem);
    const int ib = pc % N1;
    const int ic = DIM == 3 ? pc / N1 : 0;
    auto row = [](int b, int c) { return c * S::PS + b * N1; };
    const int64_t base = e * NF * NB;
    // face pencil q: face (r, s) with (r - 1) * 2 + s = q / N1 (2D: q), pencil
    // q % N1 of it; where its values start in neighbour nb
    auto face_pencil = [](int q, int32_t nb) {
        const int fi = DIM == 3 ? q / N1 : q, k = DIM == 3 ? q % N1 : 0, s = fi % 2;
        return int64_t(nb) * NF * NB + (fi / 2 ? k + N1 * (1 - s) : (1 - s) + N1 * k) * N1;
    };

    // ---- own pencil of every field; g_r
    // (kAhead: and the neighbour's pencils of the first face pencil: all loads of
    // both are in flight before any is used)
    constexpr bool kTogether = KIND == STAGE_MANY || KIND == STAGE_MANY_MIXED;
    constexpr bool kAhead = (!UPD && (DIM == 2 || N1 <= 4)) || (kTogether && DIM == 3 && N1 == 6);
    double w[NF][N1], J[DIM][DIM], wq[NF][N1];
    constexpr bool kEarly = UPD && N1 <= 4;
    double y[NF][N1];  // kEarly: the update's sum but for this stage's own term
    int32_t nbx[2] = {-1, -1}, nbq = -1;
    // x faces: a neighbour whose pencil lies in this wavefront (lane srcx) hands
    // its values over by a lane shuffle, another one's are loaded from atx on
    auto x_face = [&](int s, int& src, int64_t (&at)[NF]) {
        const int64_t ln = int64_t(nbx[s]) - blk * S::EPB;
        const bool here = ln >= 0 && ln < S::EPB && (int(ln) * NP + pc) / 64 == tid / 64;
        src = here ? (int(ln) * NP + pc) % 64 : tid % 64;
#pragma unroll
        for (int f = 0; f < NF; ++f) at[f] = (int64_t(nbx[s]) * NF + f) * NB + pc * N1 + (1 - s);
        return active && nbx[s] >= 0 && !here;
    };
    double ox[2][NF];
    if (active) {
        if (pc < NQ) nbq = p.nbr[(2 + (DIM == 3 ? pc / N1 : pc)) * p.n_elem + e];
#pragma unroll
        for (int s = 0; s < 2; ++s) nbx[s] = p.nbr[s * p.n_elem + e];
#pragma unroll
        for (int r = 0; r < DIM; ++r)
#pragma unroll
            for (int d = 0; d < DIM; ++d) J[r][d] = p.jinv[(r * DIM + d) * p.n_elem + e];
        double x[NF][N1];
        load_pencils<NF, N1, KIND>(p.io, base + pc * N1, NB, w, x);
        if constexpr (kEarly) update_partial<NF, N1>(p.io, base + pc * N1, NB, w, x, y);
        if constexpr (kTogether) {
            double xq[NF][N1], x1[2][NF];
            const int64_t bq = face_pencil(pc, nbq);
            const bool ahead = kAhead && nbq >= 0;
            bool far[2];
            int src[2];
            int64_t at[2][NF];
            if (ahead) load_pencils<NF, N1, KIND>(p.io, bq, NB, wq, xq);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                far[s] = x_face(s, src[s], at[s]);
                if (far[s]) load_two<KIND>(p.io, at[s], ox[s], x1[s]);
            }
            mix_two_pencils<NF, N1, KIND>(p.io, w, x);
            if (ahead) mix_two_pencils<NF, N1, KIND>(p.io, wq, xq);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                if (far[s]) mix_first<KIND>(p.io, ox[s], x1[s]);
#pragma unroll 1
            for (int i = 2; i < p.io.n_in; ++i) {
                const bool f32 = stage_f32<KIND>(p.io, i);
                const double c = p.io.coef[i];
                load_raw<NF, N1>(p.io.in[i], f32, base + pc * N1, NB, x);
                if (ahead) load_raw<NF, N1>(p.io.in[i], f32, bq, NB, xq);
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (far[s]) load_raw_n(p.io.in[i], f32, at[s], x1[s]);
                add_raw<NF, N1>(c, x, f32, w);
                if (ahead) add_raw<NF, N1>(c, xq, f32, wq);
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    if (far[s]) add_raw_n(c, x1[s], f32, ox[s]);
            }
        } else if constexpr (kAhead) {
            double xq[NF][N1];
            const int64_t bq = face_pencil(pc, nbq);
            if (nbq >= 0) load_pencils<NF, N1, KIND>(p.io, bq, NB, wq, xq);
            mix_pencils<NF, N1, KIND>(p.io, base + pc * N1, NB, w, x);
            if (nbq >= 0) mix_pencils<NF, N1, KIND>(p.io, bq, NB, wq, xq);
        } else {
            mix_pencils<NF, N1, KIND>(p.io, base + pc * N1, NB, w, x);
        }
    } else {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int a = 0; a < N1; ++a) w[f][a] = 0.0;
#pragma unroll
        for (int r = 0; r < DIM; ++r)
#pragma unroll
            for (int d = 0; d < DIM; ++d) J[r][d] = 0.0;
    }
    double gx[N1];
    if (active) {
#pragma unroll
        for (int r = 0; r < DIM; ++r) {
            double g[N1];
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                g[a] = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) g[a] = fma(J[r][d], w[1 + d][a], g[a]);
            }
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                if (r == 0) gx[a] = g[a];
                else s_g[((r - 1) * S::EPB + le) * S::ES + row(ib, ic) + a] = g[a];
            }
        }
#pragma unroll
        for (int a = 0; a < N1; ++a) s_v[le * S::ES + row(ib, ic) + a] = w[0][a];
    }

    // ---- x faces: one trace value per pencil
    double fvx[2], fsx[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        int src;
        int64_t at[NF];
        const bool far = x_face(s, src, at);
        double o[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) o[f] = __shfl(w[f][1 - s], src, 64);
        fvx[s] = fsx[s] = 0.0;
        if (active && nbx[s] >= 0) {
            if constexpr (kTogether) {
#pragma unroll
                for (int f = 0; f < NF; ++f) o[f] = far ? ox[s][f] : o[f];
            } else if (far) {
                double x[NF];
                load_two<KIND>(p.io, at, o, x);
                mix_two<KIND>(p.io, at, o, x);
            }
            double gn = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) gn = fma(J[0][d], o[1 + d], gn);
            fvx[s] = (s ? -0.5 : 0.5) * (gx[s] - gn);
            fsx[s] = (s ? -0.5 : 0.5) * (w[0][s] - o[0]);
        } else if (active) {
            fvx[s] = (s ? -1.0 : 1.0) * gx[s];
        }
    }
    double v[N1];
#pragma unroll
    for (int a = 0; a < N1; ++a) v[a] = w[0][a];
    __syncthreads();

    // ---- y and z faces: each face pencil's fluxes once, into LDS
#pragma unroll
    for (int q0 = 0; q0 < NQ; q0 += NP) {
        const int q = q0 + pc;
        if (!active || q >= NQ) continue;
        const int fi = DIM == 3 ? q / N1 : q;     // (r - 1) * 2 + s
        const int k = DIM == 3 ? q % N1 : 0;
        const int s = fi % 2, z = fi / 2;          // z: 0 a y face, 1 a z face
        const int32_t nb = q0 == 0 ? nbq : p.nbr[(2 + fi) * p.n_elem + e];
        double Jr[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) Jr[d] = z ? J[DIM - 1][d] : J[1][d];
        const double* vo = s_v + le * S::ES + (z ? row(k, s) : row(s, k));
        const double* go = s_g + (z * S::EPB + le) * S::ES + (z ? row(k, s) : row(s, k));
        double* out = s_f + (le * NQ + q) * 2 * N1;
        if (nb >= 0) {
            double o[NF][N1];
            if (kAhead && q0 == 0) {
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int a = 0; a < N1; ++a) o[f][a] = wq[f][a];
            } else {
                double x[NF][N1];
                load_pencils<NF, N1, KIND>(p.io, face_pencil(q, nb), NB, o, x);
                mix_pencils<NF, N1, KIND>(p.io, face_pencil(q, nb), NB, o, x);
            }
            const double h = s ? -0.5 : 0.5;
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                double gn = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) gn = fma(Jr[d], o[1 + d][a], gn);
                out[a] = h * (go[a] - gn);
                out[N1 + a] = h * (vo[a] - o[0][a]);
            }
        } else {
            const double h = s ? -1.0 : 1.0;
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                out[a] = h * go[a];
                out[N1 + a] = 0.0;
            }
        }
    }
    __syncthreads();
    if constexpr (!MASS) {  // (the mass below meets at barriers: threads without a pencil stay, on the first element)
        if (!active) return;
    }
    const int lr = MASS && le >= S::EPB ? 0 : le;

    // ---- per direction: the one-dimensional operator on g_r and on v
    double kv[N1], ks[DIM][N1];
#pragma unroll
    for (int a = 0; a < N1; ++a) {
        double x = 0.0, t = 0.0;
#pragma unroll
        for (int j = 0; j < N1; ++j) {
            x = fma(p.Dr[a * N1 + j], gx[j], x);
            t = fma(p.Dr[a * N1 + j], v[j], t);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            x = fma(p.Mi[a * N1 + s], fvx[s], x);
            t = fma(p.Mi[a * N1 + s], fsx[s], t);
        }
        kv[a] = x;
#pragma unroll
        for (int d = 0; d < DIM; ++d) ks[d][a] = J[0][d] * t;
    }
#pragma unroll
    for (int r = 1; r < DIM; ++r) {
        const int my = r == 1 ? ib : ic;
        const double* sv = s_v + lr * S::ES;
        const double* sg = s_g + ((r - 1) * S::EPB + lr) * S::ES;
        double t[N1];
#pragma unroll
        for (int a = 0; a < N1; ++a) t[a] = 0.0;
#pragma unroll
        for (int j = 0; j < N1; ++j) {
            const double dr = p.Dr[my * N1 + j];
            const int at = r == 1 ? row(j, ic) : row(ib, j);
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                kv[a] = fma(dr, sg[at + a], kv[a]);
                t[a] = fma(dr, sv[at + a], t[a]);
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const double mi = p.Mi[my * N1 + s];
            const int q = DIM == 3 ? ((r - 1) * 2 + s) * N1 + (r == 1 ? ic : ib) : s;
            const double* f = s_f + (lr * NQ + q) * 2 * N1;
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                kv[a] = fma(mi, f[a], kv[a]);
                t[a] = fma(mi, f[N1 + a], t[a]);
            }
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
            for (int a = 0; a < N1; ++a) ks[d][a] = fma(J[r][d], t[a], ks[d][a]);
    }
    // ---- MASS: the right-hand side itself, M_e times this; c_inv of the s fields'
    // mass cancels theirs here. Field by field, v's place in LDS for the passes
    // along y and z.
    if constexpr (MASS) {
        const double det = active ? p.absdet[e] : 0.0;
        auto mass = [&](double (&k)[N1]) {
            double y[N1];
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                y[a] = 0.0;
#pragma unroll
                for (int j = 0; j < N1; ++j) y[a] = fma(p.M1[a * N1 + j], k[j], y[a]);
            }
#pragma unroll
            for (int r = 1; r < DIM; ++r) {
                __syncthreads();  // the last readers are done
                if (le < S::EPB) {
#pragma unroll
                    for (int a = 0; a < N1; ++a) s_v[le * S::ES + row(ib, ic) + a] = y[a];
                }
                __syncthreads();
#pragma unroll
                for (int a = 0; a < N1; ++a) y[a] = 0.0;
#pragma unroll
                for (int j = 0; j < N1; ++j) {
                    const double m = p.M1[(r == 1 ? ib : ic) * N1 + j];
                    const double* x = s_v + lr * S::ES + (r == 1 ? row(j, ic) : row(ib, j));
#pragma unroll
                    for (int a = 0; a < N1; ++a) y[a] = fma(m, x[a], y[a]);
                }
            }
#pragma unroll
            for (int a = 0; a < N1; ++a) k[a] = y[a] * det;
        };
        mass(kv);
#pragma unroll
        for (int d = 0; d < DIM; ++d) mass(ks[d]);
        if (active) {
            store_pencil<N1>(p.io, base + pc * N1, kv);
#pragma unroll
            for (int d = 0; d < DIM; ++d) store_pencil<N1>(p.io, base + pc * N1 + (1 + d) * NB, ks[d]);
        }
        return;
    }
    const double ci = 1.0 / p.cinv[e];
    const int64_t o = base + pc * N1;
    store_pencil<N1>(p.io, o, kv);
    if constexpr (kEarly) update_store<N1>(p.io.upd, o, kv, y[0]);
    else if constexpr (UPD) rk_update_run<N1>(p.io.upd, o, kv);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
#pragma unroll
        for (int a = 0; a < N1; ++a) ks[d][a] *= ci;
        store_pencil<N1>(p.io, o + (1 + d) * NB, ks[d]);
        if constexpr (kEarly) update_store<N1>(p.io.upd, o + (1 + d) * NB, ks[d], y[1 + d]);
        else if constexpr (UPD) rk_update_run<N1>(p.io.upd, o + (1 + d) * NB, ks[d]);
    }
}

// UPD: the RK update fused into this (last) stage, StageIO::upd.
template <int DIM, int N1, int KIND, bool UPD>
__global__ __launch_bounds__((AcousticShape<DIM, N1>::THREADS)) void tensor_acoustic_rhs(const AcousticParams p) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);
    acoustic_block<DIM, N1, KIND, UPD>(p, p.order ? p.order[b] : b);
}

// hgdg_right_hand_side: the result times the mass, in one launch instead of this
// kernel's and tensor_mass's; small meshes are bound by the launches, large ones
// by the result going through memory twice more. us a call: 48 x 40 p = 2 9.6 ->
// 6.6, 256^2 p = 3 29 -> 15, 30^3 p = 1 15 -> 7.9, p = 2 34 -> 21, 32^3 p = 3 68 ->
// 53 (one wavefront a SIMD there), 16^3 p = 5 50 -> 43.
template <int DIM, int N1>
__global__ __launch_bounds__((AcousticShape<DIM, N1>::THREADS)) void tensor_acoustic_weak(const AcousticParams p) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);
    acoustic_block<DIM, N1, STAGE_ANY, false, true>(p, p.order ? p.order[b] : b);
}

template <int DIM, int N1, bool UPD = false>
__global__ __launch_bounds__((AcousticShape<DIM, N1>::THREADS)) void tensor_acoustic_rhs_batched(
    const AcousticParams* __restrict__ ps, const int64_t* __restrict__ off, int n) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);
    const int s = __builtin_amdgcn_readfirstlane(find_problem(off, n, b));
    const int32_t* order = ps[s].order;
    acoustic_block<DIM, N1, STAGE_ANY, UPD>(ps[s], order ? order[b - off[s]] : b - off[s]);
}

// L2 projection of f(x) = sum_m amp_m sin(2 pi k_m . x) on affine tensor
// elements (HpgemAPISimplified::setInitialSolution with the element rule of
// order 2p+1): the coefficients are (Mi B^T W) applied along each direction
// to f at the n1^dim Gauss points, P(a, q) = sum_b Mi(a, b) psi_b(x_q) w_q.
// One thread per x-line of quadrature points; the y/z passes go through LDS.
struct ProjParams {
    int64_t n_elem;
    int32_t nf, field;          // fields per element; target field (-1: all)
    void* out;
    int32_t out_f32;
    int32_t n_modes;
    const double* modes;        // [n_modes][4]: amp, k_x, k_y, k_z
    int32_t gaussian;           // 1: f = amplitude exp(-|x - centre|^2 / width^2) instead of modes
    double g[5];                // centre x, y, z, width, amplitude
    const double* X0;           // [dim][n_elem] (generic meshes)
    const double* E;            // [dim*dim][n_elem] (generic meshes)
    int32_t structured;
    int32_t cells[3];
    const double* P;            // [n1][n1]
    const double* xq;           // [n1]
};

template <int DIM, int N1>
__global__ __launch_bounds__(kBlock) void tensor_project(const ProjParams p) {
    using S = Pencil<DIM, N1>;
    __shared__ double s_a[S::EPB * S::NB];
    __shared__ double s_b[S::EPB * S::NB];
    const int tid = threadIdx.x;
    const int le = tid / S::NP;
    const int pc = tid % S::NP;
    const int64_t e = int64_t(blockIdx.x) * S::EPB + le;
    const bool active = (le < S::EPB) && (e < p.n_elem);
    const int i1 = pc % N1;
    const int i2 = DIM == 3 ? pc / N1 : 0;
    double X0[3] = {0, 0, 0}, E[3][3] = {{0}};
    if (active) {
        if (p.structured) {
            int64_t idx[3] = {e % p.cells[0], (e / p.cells[0]) % p.cells[1],
                              DIM == 3 ? e / (int64_t(p.cells[0]) * p.cells[1]) : 0};
            for (int d = 0; d < DIM; ++d) {
                X0[d] = 0.0 + double(idx[d]) * (1.0 - 0.0) / p.cells[d];
                E[d][d] = (0.0 + double(idx[d] + 1) * (1.0 - 0.0) / p.cells[d]) - X0[d];
            }
        } else {
            for (int d = 0; d < DIM; ++d) {
                X0[d] = p.X0[d * p.n_elem + e];
                for (int k = 0; k < DIM; ++k) E[d][k] = p.E[(d * DIM + k) * p.n_elem + e];
            }
        }
    }
    double* A = s_a + le * S::NB;
    double* B = s_b + le * S::NB;
    if (active) {
        double f[N1];
#pragma unroll
        for (int q = 0; q < N1; ++q) {
            const int qi[3] = {q, i1, i2};
            double x[3] = {X0[0], X0[1], X0[2]};
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const double t = (p.xq[qi[d]] + 1) / 2;
#pragma unroll
                for (int k = 0; k < DIM; ++k) x[k] += t * E[d][k];
            }
            double v = 0;
            if (p.gaussian) {
                double r2 = 0;
#pragma unroll
                for (int d = 0; d < DIM; ++d) r2 += (x[d] - p.g[d]) * (x[d] - p.g[d]);
                v = p.g[4] * exp(-r2 / (p.g[3] * p.g[3]));
            } else {
                for (int m = 0; m < p.n_modes; ++m) {
                    double arg = 0;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) arg += p.modes[4 * m + 1 + d] * x[d];
                    v += p.modes[4 * m] * sin(2 * M_PI * arg);
                }
            }
            f[q] = v;
        }
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            double t = 0;
#pragma unroll
            for (int q = 0; q < N1; ++q) t += p.P[a * N1 + q] * f[q];
            A[pc * N1 + a] = t;  // (a, q_y, q_z)
        }
    }
    __syncthreads();
    if (active) {  // y pass: this thread makes (., b = i1, q_z = i2)
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            double t = 0;
#pragma unroll
            for (int q = 0; q < N1; ++q) t += p.P[i1 * N1 + q] * A[(q + N1 * i2) * N1 + a];
            B[pc * N1 + a] = t;
        }
    }
    __syncthreads();
    if (!active) return;
    double coef[N1];
    if (DIM == 3) {  // z pass: (., b, c) from (., b, q_z)
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            double t = 0;
#pragma unroll
            for (int q = 0; q < N1; ++q) t += p.P[i2 * N1 + q] * B[(i1 + N1 * q) * N1 + a];
            coef[a] = t;
        }
    } else {
#pragma unroll
        for (int a = 0; a < N1; ++a) coef[a] = B[pc * N1 + a];
    }
    for (int f = 0; f < p.nf; ++f) {
        if (p.field >= 0 && f != p.field) continue;
        const int64_t o = (e * p.nf + f) * S::NB + pc * N1;
        if (p.out_f32) {
#pragma unroll
            for (int a = 0; a < N1; ++a) static_cast<float*>(p.out)[o + a] = float(coef[a]);
        } else {
#pragma unroll
            for (int a = 0; a < N1; ++a) static_cast<double*>(p.out)[o + a] = coef[a];
        }
    }
}

// Per-element mass-norm of x - y: |J| dx^T (M1 x M1 x M1) dx, and max |dx|;
// one partial per block.
struct DiffParams {
    int64_t n_elem;
    const void* x;
    const void* y;
    int32_t x_f32, y_f32;
    const double* absdet;  // [n_elem / fields]
    int32_t fields;        // consecutive blocks of one element
    const double* M1;      // [n1][n1]
    double* partial;       // [grid][2]
};

template <int DIM, int N1>
__global__ __launch_bounds__(kBlock) void tensor_diff_norm(const DiffParams p) {
    using S = Tensor<DIM, N1>;
    __shared__ double s_a[S::EPB * S::NB];
    __shared__ double s_b[S::EPB * S::NB];
    __shared__ double s_M[N1 * N1];
    __shared__ double s_red[2][kBlock];
    const int tid = threadIdx.x;
    if (tid < N1 * N1) s_M[tid] = p.M1[tid];
    const int le = tid / S::L;
    const int dof = tid % S::L;
    const int64_t e = int64_t(blockIdx.x) * S::EPB + le;
    const bool active = (e < p.n_elem) && (dof < S::NB);
    double dx = 0;
    if (active) {
        const int64_t i = e * S::NB + dof;
        const double xv = p.x_f32 ? double(static_cast<const float*>(p.x)[i]) : static_cast<const double*>(p.x)[i];
        const double yv = p.y_f32 ? double(static_cast<const float*>(p.y)[i]) : static_cast<const double*>(p.y)[i];
        dx = xv - yv;
        s_a[le * S::NB + dof] = dx;
    }
    __syncthreads();
    const int idx[3] = {dof % N1, (dof / N1) % N1, DIM == 3 ? dof / (N1 * N1) : 0};
    constexpr int stride[3] = {1, N1, N1 * N1};
    double* src = s_a;
    double* dst = s_b;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        if (active) {
            const int row = dof - idx[d] * stride[d];
            double s = 0;
            for (int j = 0; j < N1; ++j) s += s_M[idx[d] * N1 + j] * src[le * S::NB + row + j * stride[d]];
            dst[le * S::NB + dof] = s;
        }
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
    }
    double v = 0, m = 0;
    if (active) {
        v = dx * src[le * S::NB + dof] * p.absdet[e / p.fields];
        m = fabs(dx);
    }
    s_red[0][tid] = v;
    s_red[1][tid] = m;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (tid < w) {
            s_red[0][tid] += s_red[0][tid + w];
            s_red[1][tid] = fmax(s_red[1][tid], s_red[1][tid + w]);
        }
        __syncthreads();
    }
    if (tid == 0) {
        p.partial[2 * blockIdx.x] = s_red[0][0];
        p.partial[2 * blockIdx.x + 1] = s_red[1][0];
    }
}

// The block-diagonal mass matrix (HpgemAPILinear::createMassMatrices, with
// the acoustic weighting of AcousticWaveLinear_Impl.h:102-129) applied to a
// vector, or solved against it, in place: per element and field the 1D factor
// A1 = M1 (apply) or Mi = M1^{-1} (solve) along every direction, then times
// |det J| w_f (apply) or divided by it (solve); w_f = c_inv on the s fields of
// the acoustic system, else 1.
struct MassParams {
    int64_t n_blocks;      // elements x fields, field-major inside an element
    int32_t fields;
    int32_t inverse;
    double* v;
    const double* absdet;  // [n_elem]
    const double* cinv;    // [n_elem], or NULL
    const double* A1;      // [n1][n1]
};

template <int DIM, int N1>
__global__ __launch_bounds__(kBlock) void tensor_mass(const MassParams p) {
    using S = Tensor<DIM, N1>;
    __shared__ double s_a[S::EPB * S::NB];
    __shared__ double s_b[S::EPB * S::NB];
    __shared__ double s_M[N1 * N1];
    const int tid = threadIdx.x;
    if (tid < N1 * N1) s_M[tid] = p.A1[tid];
    const int le = tid / S::L;
    const int dof = tid % S::L;
    const int64_t b = int64_t(blockIdx.x) * S::EPB + le;
    const bool active = (b < p.n_blocks) && (dof < S::NB);
    if (active) s_a[le * S::NB + dof] = p.v[b * S::NB + dof];
    __syncthreads();
    const int idx[3] = {dof % N1, (dof / N1) % N1, DIM == 3 ? dof / (N1 * N1) : 0};
    constexpr int stride[3] = {1, N1, N1 * N1};
    double* src = s_a;
    double* dst = s_b;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        if (active) {
            const int row = dof - idx[d] * stride[d];
            double s = 0;
            for (int j = 0; j < N1; ++j) s += s_M[idx[d] * N1 + j] * src[le * S::NB + row + j * stride[d]];
            dst[le * S::NB + dof] = s;
        }
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
    }
    if (active) {
        const int64_t e = b / p.fields;
        double w = p.absdet[e];
        if (p.cinv != nullptr && b % p.fields > 0) w *= p.cinv[e];
        const double x = src[le * S::NB + dof];
        p.v[b * S::NB + dof] = p.inverse ? x / w : x * w;
    }
}

template <typename F>
void dispatch_tensor(int dim, int n1, F&& f) {
#define HGDG_CASE(D, N) \
    if (dim == D && n1 == N) return f(std::integral_constant<int, D>{}, std::integral_constant<int, N>{});
    HGDG_CASE(2, 2) HGDG_CASE(2, 3) HGDG_CASE(2, 4) HGDG_CASE(2, 5) HGDG_CASE(2, 6)
    HGDG_CASE(3, 2) HGDG_CASE(3, 3) HGDG_CASE(3, 4) HGDG_CASE(3, 5) HGDG_CASE(3, 6)
#undef HGDG_CASE
    throw Failure(HGDG_ERR_UNSUPPORTED, "no tensor kernel for this dimension and order");
}

// Error of one field (or every field) against f(x - shift), f = sum_m amp_m
// sin(2 pi k_m . x) (HpgemAPISimplified::computeTotalError and computeMaxError,
// kernel/Base/HpgemAPISimplified_Impl.h:293-530): the squared L2 error with
// the (p+2)-point Gauss rule per direction (order 2p+2) and the largest
// pointwise error at the element rule's (p+1)^dim points (order 2p+1). One
// thread per element; per-block partial sums and maxima.
struct ErrParams {
    int64_t n_elem;
    int32_t nf, field;
    const void* u;
    int32_t u_f32;
    int32_t n_modes;
    const double* modes;   // [n_modes][4]: amp, k
    double shift[3];
    const double* X0;      // [dim][n_elem]
    const double* E;       // [dim*dim][n_elem]
    const double* absdet;  // [n_elem]
    const double* tab;     // psi at the L2 points [N1][N1+1], their weights and points [N1+1] each,
                           // psi at the element rule points [N1][N1], those points [N1]
    double* partial;       // [blocks][2]
};

template <int DIM, int N1>
__global__ __launch_bounds__(kBlock) void tensor_error(const ErrParams p) {
    constexpr int NB = N1 * N1 * (DIM == 3 ? N1 : 1);
    __shared__ double s_red[2][kBlock];
    const int64_t e = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    double sum = 0, mx = 0;
    if (e < p.n_elem) {
        double X0[3] = {0, 0, 0}, E[3][3] = {{0}};
        for (int d = 0; d < DIM; ++d) {
            X0[d] = p.X0[d * p.n_elem + e];
            for (int k = 0; k < DIM; ++k) E[d][k] = p.E[(d * DIM + k) * p.n_elem + e];
        }
        const double det = p.absdet[e];
        for (int fld = 0; fld < p.nf; ++fld) {
            if (p.field >= 0 && fld != p.field) continue;
            const int64_t base = (e * p.nf + fld) * NB;
            for (int pass = 0; pass < 2; ++pass) {
                const int NQ = pass == 0 ? N1 + 1 : N1;
                const double* psi = pass == 0 ? p.tab : p.tab + N1 * (N1 + 1) + 2 * (N1 + 1);
                const double* wq = p.tab + N1 * (N1 + 1);
                const double* xq = pass == 0 ? wq + (N1 + 1) : psi + N1 * N1;
                const int nz = DIM == 3 ? NQ : 1;
                for (int qz = 0; qz < nz; ++qz)
                    for (int qy = 0; qy < NQ; ++qy)
                        for (int qx = 0; qx < NQ; ++qx) {
                            double val = 0;
                            for (int c = 0; c < (DIM == 3 ? N1 : 1); ++c) {
                                double vy = 0;
                                for (int b = 0; b < N1; ++b) {
                                    double vx = 0;
                                    for (int a = 0; a < N1; ++a) {
                                        const int64_t i = base + a + N1 * (b + N1 * c);
                                        const double cf = p.u_f32 ? double(static_cast<const float*>(p.u)[i])
                                                                  : static_cast<const double*>(p.u)[i];
                                        vx += cf * psi[a * NQ + qx];
                                    }
                                    vy += vx * psi[b * NQ + qy];
                                }
                                val += DIM == 3 ? vy * psi[c * NQ + qz] : vy;
                            }
                            const int q[3] = {qx, qy, qz};
                            double x[3] = {X0[0], X0[1], X0[2]};
                            for (int d = 0; d < DIM; ++d) {
                                const double t = (xq[q[d]] + 1) / 2;
                                for (int k = 0; k < DIM; ++k) x[k] += t * E[d][k];
                            }
                            double ex = 0;
                            for (int m = 0; m < p.n_modes; ++m) {
                                double arg = 0;
                                for (int d = 0; d < DIM; ++d) arg += p.modes[4 * m + 1 + d] * (x[d] - p.shift[d]);
                                ex += p.modes[4 * m] * sin(2 * M_PI * arg);
                            }
                            const double err = ex - val;
                            if (pass == 0) {
                                double w = det;
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

// ---------------------------------------------------------------- host side
namespace {
const double* Dr_ptr(hgdg_ctx* c) { return c->tm.d_ops.ptr; }
const double* Mi_ptr(hgdg_ctx* c) { return c->tm.d_ops.ptr + c->tm.n1 * c->tm.n1; }
const double* M1_ptr(hgdg_ctx* c) { return c->tm.d_ops.ptr + 2 * c->tm.n1 * c->tm.n1; }
}  // namespace

// J (column d = E_d / 2), |det J| and J^{-1} of affine element e from its edge
// vectors E[d] = X_{2^d} - X_0; shared by the generic and the structured setup
// so both produce the same numbers.
void affine_geometry(hgdg_ctx* c, int64_t e, const double (&E)[3][3]) {
    const int dim = c->dim;
    double J[3][3] = {{0}};  // J[r][c] = d x_r / d xi_c
    for (int r = 0; r < dim; ++r)
        for (int col = 0; col < dim; ++col) J[r][col] = E[col][r] / 2;
    double det, inv[3][3];
    if (dim == 2) {
        det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
        inv[0][0] = J[1][1] / det;
        inv[0][1] = -J[0][1] / det;
        inv[1][0] = -J[1][0] / det;
        inv[1][1] = J[0][0] / det;
    } else {
        det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
              J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
        for (int r = 0; r < 3; ++r)
            for (int col = 0; col < 3; ++col) {
                const int r1 = (col + 1) % 3, r2 = (col + 2) % 3, c1 = (r + 1) % 3, c2 = (r + 2) % 3;
                inv[r][col] = (J[r1][c1] * J[r2][c2] - J[r1][c2] * J[r2][c1]) / det;
            }
    }
    require(det != 0.0 && std::isfinite(det), HGDG_ERR_ARG, "degenerate element " + std::to_string(e));
    c->tm.absdet[e] = std::fabs(det);
    for (int r = 0; r < dim; ++r)
        for (int col = 0; col < dim; ++col) c->tm.Jinv[(size_t(e) * dim + r) * dim + col] = inv[r][col];
}

void finish_tensor_upload(hgdg_ctx* c) {
    c->n_fields = 1;
    c->dof = c->n_elem * c->tm.nb;
    c->tm.ops = tensor_ops(c->tm.p);
    std::vector<double> opsv;
    opsv.insert(opsv.end(), c->tm.ops.Dr.begin(), c->tm.ops.Dr.end());
    opsv.insert(opsv.end(), c->tm.ops.Mi.begin(), c->tm.ops.Mi.end());
    opsv.insert(opsv.end(), c->tm.ops.M1.begin(), c->tm.ops.M1.end());
    c->tm.d_ops.upload(opsv, c->stream);
    c->tm.d_nbr.upload(c->tm.nbr, c->stream);
    c->tm.d_absdet.upload(c->tm.absdet, c->stream);
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

// The periodic box [0,1]^dim with n[d] cells, as structured_mesh builds it
// (x fastest, vertex order x fastest, coordinates lo + i (hi - lo) / n), set
// up without the generic face search: neighbours are known from the indices.
void tensor_structured_upload(hgdg_ctx* c, int dim, const int32_t* n, int p) {
    require(dim == 2 || dim == 3, HGDG_ERR_ARG, "dim must be 2 or 3");
    require(p >= 1 && p <= 5, HGDG_ERR_UNSUPPORTED, "polynomial order must be in 1..5");
    int64_t ne = 1;
    for (int d = 0; d < dim; ++d) {
        require(n[d] >= 3, HGDG_ERR_ARG, "periodic boxes need at least 3 cells per direction");
        ne *= n[d];
    }
    c->shape = dim == 3 ? SHAPE_CUBE : SHAPE_SQUARE;
    c->dim = dim;
    c->n_elem = ne;
    c->tm.p = p;
    c->tm.n1 = p + 1;
    c->tm.nb = dim == 3 ? c->tm.n1 * c->tm.n1 * c->tm.n1 : c->tm.n1 * c->tm.n1;
    c->tm.perm = tensor_permutation(dim, p);
    c->tm.structured = true;
    for (int d = 0; d < 3; ++d) c->tm.cells[d] = d < dim ? n[d] : 1;
    c->tm.Jinv.assign(size_t(ne) * dim * dim, 0.0);
    c->tm.absdet.assign(ne, 0.0);
    c->tm.nbr.assign(size_t(2 * dim) * ne, -1);
    int64_t stride[3] = {1, n[0], dim == 3 ? int64_t(n[0]) * n[1] : 0};
    for (int64_t e = 0; e < ne; ++e) {
        int64_t idx[3] = {e % n[0], (e / n[0]) % n[1], dim == 3 ? e / (int64_t(n[0]) * n[1]) : 0};
        double E[3][3] = {{0}};
        for (int d = 0; d < dim; ++d)
            E[d][d] = (0.0 + double(idx[d] + 1) * (1.0 - 0.0) / n[d]) - (0.0 + double(idx[d]) * (1.0 - 0.0) / n[d]);
        affine_geometry(c, e, E);
        for (int d = 0; d < dim; ++d) {
            const int64_t lo_n = idx[d] == 0 ? e + (n[d] - 1) * stride[d] : e - stride[d];
            const int64_t hi_n = idx[d] == n[d] - 1 ? e - (n[d] - 1) * stride[d] : e + stride[d];
            c->tm.nbr[size_t(2 * d) * ne + e] = int32_t(lo_n);
            c->tm.nbr[size_t(2 * d + 1) * ne + e] = int32_t(hi_n);
        }
    }
    c->n_faces = int64_t(dim) * ne;
    c->n_internal = c->n_faces;
    finish_tensor_upload(c);
}

void tensor_mesh_upload(hgdg_ctx* c, const hgdg_mesh_desc* m) {
    const int dim = shape_dim(m->shape);
    const int64_t ne = m->n_elements;
    int p = m->order ? m->order[0] : m->uniform_order;
    if (m->order)
        for (int64_t e = 0; e < ne; ++e)
            require(m->order[e] == p, HGDG_ERR_UNSUPPORTED,
                    "tensor elements need one polynomial order per mesh");
    require(p >= 1 && p <= 5, HGDG_ERR_UNSUPPORTED, "polynomial order must be in 1..5");
    const int nv = shape_vertices(m->shape);

    c->tm.p = p;
    c->tm.n1 = p + 1;
    c->tm.nb = dim == 3 ? c->tm.n1 * c->tm.n1 * c->tm.n1 : c->tm.n1 * c->tm.n1;
    c->tm.perm = tensor_permutation(dim, p);
    if (c->tensor_general_forced) {
        tensor_general_upload(c, m);
        return;
    }

    // geometry: affine hypercubes here (J column d = (X_{2^d} - X_0) / 2);
    // any other element sends the mesh to the Gauss-point path
    c->tm.Jinv.assign(size_t(ne) * dim * dim, 0.0);
    c->tm.absdet.assign(ne, 0.0);
    c->tm.X0.assign(size_t(ne) * dim, 0.0);
    c->tm.E.assign(size_t(ne) * dim * dim, 0.0);
    for (int64_t e = 0; e < ne; ++e) {
        const double* X = m->coords + size_t(e) * nv * dim;
        double E[3][3] = {{0}};
        double scale = 0;
        for (int d = 0; d < dim; ++d)
            for (int r = 0; r < dim; ++r) {
                E[d][r] = X[(1 << d) * dim + r] - X[r];
                scale = std::max(scale, std::fabs(E[d][r]));
            }
        for (int d = 0; d < dim; ++d) {
            c->tm.X0[size_t(e) * dim + d] = X[d];
            for (int r = 0; r < dim; ++r) c->tm.E[(size_t(e) * dim + d) * dim + r] = E[d][r];
        }
        for (int v = 0; v < nv; ++v)
            for (int r = 0; r < dim; ++r) {
                double pred = X[r];
                for (int d = 0; d < dim; ++d)
                    if ((v >> d) & 1) pred += E[d][r];
                if (!(std::fabs(pred - X[v * dim + r]) <= 1e-12 * scale)) {
                    tensor_general_upload(c, m);
                    return;
                }
            }
        affine_geometry(c, e, E);
    }

    // faces: match sorted node tuples; the lower element index is hpGEM's
    // left element (faces are created while elements are visited in order).
    const int nfaces = 2 * dim;
    const int fverts = 1 << (dim - 1);
    c->tm.nbr.assign(size_t(nfaces) * ne, -1);
    std::unordered_map<std::string, std::pair<int64_t, int>> open;
    open.reserve(size_t(ne) * nfaces);
    int64_t n_internal = 0, n_total = 0;
    auto face_vertex = [&](int f, int q) {
        // local vertex of tensor face f = 2d + s: bit d = s, the other bits from q in order
        const int d = f / 2, s = f % 2;
        int v = 0, bit = 0;
        for (int k = 0; k < dim; ++k) {
            if (k == d) {
                v |= s << k;
            } else {
                v |= ((q >> bit) & 1) << k;
                ++bit;
            }
        }
        return v;
    };
    for (int64_t e = 0; e < ne; ++e) {
        const int64_t* nid = m->node_ids + size_t(e) * nv;
        for (int f = 0; f < nfaces; ++f) {
            std::array<int64_t, 4> key{};
            for (int q = 0; q < fverts; ++q) key[q] = nid[face_vertex(f, q)];
            std::sort(key.begin(), key.begin() + fverts);
            std::string k(reinterpret_cast<const char*>(key.data()), sizeof(int64_t) * fverts);
            auto it = open.find(k);
            if (it == open.end()) {
                open.emplace(std::move(k), std::make_pair(e, f));
                continue;
            }
            const int64_t o = it->second.first;
            const int fo = it->second.second;
            require(o != e, HGDG_ERR_UNSUPPORTED, "element " + std::to_string(e) + " meets itself across a face");
            require(c->tm.nbr[size_t(fo) * ne + o] < 0, HGDG_ERR_ARG, "a face is bounded by more than two elements");
            // the sum-factorised kernels need the neighbour's opposite face in
            // the same orientation: my face (d, s) against its (d, 1-s), vertex
            // by vertex; any other neighbour sends the mesh to the Gauss-point path
            bool aligned = fo / 2 == f / 2 && fo % 2 != f % 2;
            const int64_t* onid = m->node_ids + size_t(o) * nv;
            for (int q = 0; q < fverts && aligned; ++q) aligned = onid[face_vertex(fo, q)] == nid[face_vertex(f, q)];
            if (!aligned) {
                tensor_general_upload(c, m);
                return;
            }
            c->tm.nbr[size_t(f) * ne + e] = int32_t(o);
            c->tm.nbr[size_t(fo) * ne + o] = int32_t(e);
            open.erase(it);
            ++n_internal;
            ++n_total;
        }
    }
    n_total += int64_t(open.size());
    c->n_faces = n_total;
    c->n_internal = n_internal;
    finish_tensor_upload(c);
}

// The order in which the acoustic kernel's workgroups take the elements of a
// box too large to go plane by plane: an XCD's share of the launch is a range
// of planes, a z neighbour is a plane away, and three vectors' planes (two
// inputs, one output) beyond the 4 MB L2 are read again from farther off. The
// rows are then taken in columns of as many as fit 1.5 MB, through all planes.
// Rows and planes are guessed from the numbering (the distances to an
// element's upper y and z neighbours); a wrong guess changes the order only.
// RK4 step of 32^3 p = 3 (6.3 MB a plane) 234 -> 220 us, 48^3 p = 2 (6 MB) 437 ->
// 399; of boxes around the line (23 x 19 planes of p = 4, 5.2 MB) the same.
static std::vector<int32_t> acoustic_order(const hgdg_ctx* c) {
    if (c->dim != 3) return {};
    const int64_t ne = c->n_elem, bytes = 3 * int64_t(sizeof(double)) * c->tm.nb * c->n_fields;
    int64_t sy = 0, sz = 0;
    for (int64_t e = ne / 2; e < ne && (sy <= 0 || sz <= sy); ++e) {
        sy = c->tm.nbr[size_t(3) * ne + e] - e;
        sz = c->tm.nbr[size_t(5) * ne + e] - e;
    }
    if (sy <= 0 || sz <= sy || sz * bytes <= (int64_t(4) << 20)) return {};
    int64_t epb = 1;
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        epb = AcousticShape<decltype(D)::value, decltype(N)::value>::EPB;
    });
    const int64_t n = (ne + epb - 1) / epb, rows = std::max<int64_t>(1, (int64_t(3) << 19) / (sy * bytes));
    if (n > std::numeric_limits<int32_t>::max()) return {};
    std::vector<int32_t> order(static_cast<size_t>(n));
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        auto column = [&](int32_t i) { return i * epb % sz / sy / rows; };
        return column(a) < column(b);
    });
    return order;
}

void tensor_operator_set(hgdg_ctx* c, const hgdg_op_desc* op) {
    if (c->tm.general) {
        tensor_general_operator_set(c, op);
        return;
    }
    const int dim = c->dim;
    const int64_t ne = c->n_elem;
    if (op->kind == HGDG_OP_ACOUSTIC_CENTRAL) {
        std::vector<double> geo(size_t(dim) * dim * ne + ne);
        for (int64_t e = 0; e < ne; ++e) {
            for (int r = 0; r < dim; ++r)
                for (int d = 0; d < dim; ++d)
                    geo[(size_t(r) * dim + d) * ne + e] = c->tm.Jinv[(size_t(e) * dim + r) * dim + d];
            geo[size_t(dim) * dim * ne + e] = c->cinv[e];
        }
        c->tm.d_geo.upload(geo, c->stream);
        c->n_fields = dim + 1;
        c->dof = ne * c->tm.nb * c->n_fields;
        const std::vector<int32_t> order = acoustic_order(c);
        c->tm.d_order.reset();
        if (!order.empty()) c->tm.d_order.upload(order, c->stream);
        HGDG_HIP(hipStreamSynchronize(c->stream));
        return;
    }
    c->n_fields = 1;
    c->dof = ne * c->tm.nb;
    std::vector<double> ahat(size_t(dim) * ne);
    std::vector<double> rownorm(size_t(dim) * ne);
    for (int64_t e = 0; e < ne; ++e)
        for (int d = 0; d < dim; ++d) {
            double s = 0, n2 = 0;
            for (int k = 0; k < dim; ++k) {
                const double v = c->tm.Jinv[(size_t(e) * dim + d) * dim + k];
                s += v * op->velocity[k];
                n2 += v * v;
            }
            ahat[size_t(d) * ne + e] = s;
            rownorm[size_t(d) * ne + e] = std::sqrt(n2);
        }
    // a . n_unit on face (d, s) of element e: outward normal (2s-1) J^{-T} e_d
    auto a_dot_n = [&](int64_t e, int f) {
        const int d = f / 2, s = f % 2;
        return (2 * s - 1) * ahat[size_t(d) * ne + e] / rownorm[size_t(d) * ne + e];
    };
    std::vector<uint32_t> mode(ne, 0);
    std::vector<uint2> face(size_t(2) * dim * ne);
    for (int64_t e = 0; e < ne; ++e) {
        uint32_t word = 0;
        for (int f = 0; f < 2 * dim; ++f) {
            const int32_t o = c->tm.nbr[size_t(f) * ne + e];
            uint32_t m;
            if (o < 0) {
                // boundary: only the left (own) trial functions exist
                const double A = a_dot_n(e, f);
                m = A > 1e-12 ? MODE_OWN : (A < -1e-12 ? MODE_NONE : MODE_HALF_OWN);
            } else {
                // the left element's normal decides the upwind side
                const bool left = e < o;
                const double A = left ? a_dot_n(e, f) : a_dot_n(o, f ^ 1);
                if (A > 1e-12) m = left ? MODE_OWN : MODE_NBR;
                else if (A < -1e-12) m = left ? MODE_NBR : MODE_OWN;
                else m = MODE_AVG;
            }
            word |= m << (3 * f);
        }
        mode[e] = word;
        for (int f = 0; f < 2 * dim; ++f) {
            const uint32_t m = (word >> (3 * f)) & 7u;
            face[size_t(e) * 2 * dim + f] = 
                make_uint2(uint32_t(m == MODE_NBR || m == MODE_AVG ? c->tm.nbr[size_t(f) * ne + e] : e), face_coef(m, f % 2));
        }
    }
    c->tm.d_geo.upload(ahat, c->stream);
    c->tm.d_mode.upload(mode, c->stream);
    c->tm.d_face.upload(face, c->stream);
    HGDG_HIP(hipStreamSynchronize(c->stream));
}

static RhsParams advection_params(hgdg_ctx* c, const StageIO& io) {
    RhsParams p{};
    p.n_elem = c->n_elem;
    p.io = io;
    p.ahat = c->tm.d_geo.ptr;
    p.nbr = c->tm.d_nbr.ptr;
    p.mode = c->tm.d_mode.ptr;
    p.face = c->tm.d_face.ptr;
    p.Dr = Dr_ptr(c);
    p.Mi = Mi_ptr(c);
    return p;
}

// MANY: with kernels of their own for three and more inputs, as the stages of
// Dormand-Prince have. By STAGE_ANY each of an input's loads asks for its type
// and an FP32 value waits in two registers, which costs half the wavefronts:
// 301 x 257 p = 3 with FP32 stages, 3, 5 and 7 inputs, 10.2, 15.0 and 19.8 us so
// against 7.3, 9.4 and 11.6 (FP64 11.1, 14.9, 17.8 and 9.0, 12.8, 16.2); 600 x
// 500 p = 5 82, 119 and 151 against 60, 85 and 107.
template <bool MANY, typename F>
static void with_stage_kind(const StageIO& io, F&& f) {
    switch (stage_kind(io)) {
        case STAGE_ONE: f(std::integral_constant<int, STAGE_ONE>{}); break;
        case STAGE_TWO: f(std::integral_constant<int, STAGE_TWO>{}); break;
        case STAGE_TWO_MIXED: f(std::integral_constant<int, STAGE_TWO_MIXED>{}); break;
        case STAGE_MANY: f(std::integral_constant<int, MANY ? int(STAGE_MANY) : int(STAGE_ANY)>{}); break;
        case STAGE_MANY_MIXED: f(std::integral_constant<int, MANY ? int(STAGE_MANY_MIXED) : int(STAGE_ANY)>{}); break;
        default: f(std::integral_constant<int, STAGE_ANY>{}); break;
    }
}

static void launch_advection(hgdg_ctx* c, const RhsParams& p, int tiles) {
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = Pencil<DIMc, N1c>;
        const int64_t n_tiles = (c->n_elem + S::EPB - 1) / S::EPB;
        const bool upd = p.io.upd.u != nullptr;  // the fused RK update runs in the one-tile kernel
        with_stage_kind<true>(p.io, [&](auto K) {
            constexpr int KIND = decltype(K)::value;
            if (upd)
                hipLaunchKernelGGL((tensor_advection_rhs<DIMc, N1c, KIND, true>), dim3(unsigned(n_tiles)),
                                   dim3(kBlock), 0, c->stream, p);
            else if (tiles > 1)
                hipLaunchKernelGGL((tensor_advection_rhs_tiled<DIMc, N1c, KIND>),
                                   dim3(unsigned((n_tiles + tiles - 1) / tiles)), dim3(kBlock), 0, c->stream, p,
                                   tiles);
            else
                hipLaunchKernelGGL((tensor_advection_rhs<DIMc, N1c, KIND, false>), dim3(unsigned(n_tiles)),
                                   dim3(kBlock), 0, c->stream, p);
        });
    });
    HGDG_HIP(hipGetLastError());
}

void tensor_tune(hgdg_ctx* c) {
    for (double& t : c->adv_tile_ms) t = 0;
    if (c->op.kind != HGDG_OP_ADVECTION_UPWIND || c->tm.general) return;
    if (c->adv_tiles_fixed > 0) {
        c->adv_tiles = c->adv_tiles_fixed;
        return;
    }
    // One RK stage's shape: u + a k -> k', with the stage vectors in the
    // storage type of the operator's precision. Values do not change the
    // timing (no data-dependent branches), so the inputs are zero.
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
    const RhsParams p = advection_params(c, io);
    EventPair events;
    hipEvent_t* ev = events.e;
    constexpr int kCand[4] = {1, 2, 4, 8};
    constexpr int kReps = 20;
    constexpr int n_cand = 4;
    double best = 0;
    int best_tiles = 1;
    for (int pass = 0; pass < 2; ++pass)
        for (int i = 0; i < n_cand; ++i) {
            for (int r = 0; r < 3; ++r) launch_advection(c, p, kCand[i]);
            HGDG_HIP(hipEventRecord(ev[0], c->stream));
            for (int r = 0; r < kReps; ++r) launch_advection(c, p, kCand[i]);
            HGDG_HIP(hipEventRecord(ev[1], c->stream));
            HGDG_HIP(hipEventSynchronize(ev[1]));
            float ms = 0;
            HGDG_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
            const double t = double(ms) / kReps;
            if (pass == 0 || t < c->adv_tile_ms[i]) c->adv_tile_ms[i] = t;
        }
    // Several tiles have to win clearly: over the sizes and orders of the figures
    // at advection_tiles one tile a workgroup is the fastest (32^3 p = 3: RK4 step
    // 60 against 67, 75 and 90 us with 2, 4 and 8), and a choice by noise costs more.
    for (int i = 0; i < n_cand; ++i)
        if (i == 0 || c->adv_tile_ms[i] < 0.9 * best) {
            best = c->adv_tile_ms[i];
            best_tiles = kCand[i];
        }
    HGDG_HIP(hipStreamSynchronize(c->stream));
    c->adv_tiles = best_tiles;
}

// Largest dynamic LDS the fused RK kernel asks for (MI355X: 160 KB per
// workgroup; the kernel's tables take a few hundred bytes of static LDS).
constexpr size_t kRkTinyMaxLds = 150 * 1024;
constexpr int kRkTinyChunk = 500;  // steps per launch

bool tensor_rk_tiny(hgdg_ctx* c, int solution, const int* aux, int stages, const double* a, const double* b,
                    double dt, int n_steps) {
    if (c->rk_fused == 0 || c->simplex() || c->tm.general || c->op.kind != HGDG_OP_ADVECTION_UPWIND || n_steps < 1)
        return false;
    const bool mixed = c->op.precision == HGDG_PREC_MIXED_FP32;
    const int64_t E = c->n_elem, n = c->n_dof();
    const size_t tb = mixed ? 4 : 8;
    const size_t bytes = size_t(16 * n) + size_t(4 * E * (1 + 2 * c->dim) + 4) + size_t(8 * c->dim * E) +
                         size_t(stages) * size_t(n) * tb;
    if (bytes > kRkTinyMaxLds) return false;
    RkTinyParams p{};
    StageIO io{};
    p.rhs = advection_params(c, io);
    Vec& u = vec_at(c, solution);
    p.u = u.f64->ptr;
    for (int j = 0; j < stages; ++j) {
        Vec& k = vec_at(c, aux[j]);
        require(k.is_f32 == mixed, HGDG_ERR_ARG, "stage vector storage does not match the operator's precision");
        p.k[j] = k.ptr();
    }
    p.stages = stages;
    p.n_steps = n_steps;
    for (int i = 0; i < stages; ++i)
        for (int j = 0; j < i; ++j) {
            p.ca[i * kMaxIn + j] = dt * a[i * stages + j];
            if (a[i * stages + j] != 0.0) p.amask[i] |= 1u << j;
        }
    for (int j = 0; j < stages; ++j) {
        p.cb[j] = dt * b[j];
        if (b[j] != 0.0) p.bmask |= 1u << j;
    }
    bool launched = false;
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        auto go = [&](auto kernel, int threads, size_t lds) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds)) != hipSuccess) {
                (void)hipGetLastError();  // this device cannot give the LDS: the graph path runs instead
                return false;
            }
            // at most kRkTinyChunk steps per launch, so that no launch runs for
            // long; the solution goes through HBM between launches exactly (FP64)
            for (int done = 0; done < n_steps; done += kRkTinyChunk) {
                RkTinyParams q = p;
                q.n_steps = std::min(kRkTinyChunk, n_steps - done);
                hipLaunchKernelGGL(kernel, dim3(1), dim3(unsigned(threads)), lds, c->stream, q);
                HGDG_HIP(hipGetLastError());
                ++c->rk_fused_launches;
            }
            return true;
        };
        // one x-pencil a thread where the workgroup has that many threads
        // (2D p = 2 with RK4: every mesh whose state fits)
        constexpr int kPencil = rk_pencil_block<DIMc, N1c>(), kTiny = rk_tiny_block<DIMc, N1c>();
        const size_t lds = size_t(16 * n) + size_t(stages) * size_t(n) * tb;
        if constexpr (kPencil > 0) {
            if (E * Pencil<DIMc, N1c>::NP <= kPencil) {
                const int threads = int((E * Pencil<DIMc, N1c>::NP + 63) / 64 * 64);  // no wavefront without work
                launched = mixed ? go(tensor_advection_rk_pencil<DIMc, N1c, float>, threads, lds)
                                 : go(tensor_advection_rk_pencil<DIMc, N1c, double>, threads, lds);
                return;
            }
        }
        launched = mixed ? go(tensor_advection_rk_tiny<DIMc, N1c, float>, kTiny, bytes)
                         : go(tensor_advection_rk_tiny<DIMc, N1c, double>, kTiny, bytes);
    });
    return launched;
}

static AcousticParams acoustic_params(hgdg_ctx* c, const StageIO& io) {
    AcousticParams a{};
    a.n_elem = c->n_elem;
    a.io = io;
    a.jinv = c->tm.d_geo.ptr;
    a.cinv = c->tm.d_geo.ptr + size_t(c->dim) * c->dim * c->n_elem;
    a.nbr = c->tm.d_nbr.ptr;
    a.Dr = Dr_ptr(c);
    a.Mi = Mi_ptr(c);
    a.order = c->tm.d_order.ptr;
    a.absdet = c->tm.d_absdet.ptr;
    a.M1 = M1_ptr(c);
    return a;
}

// hgdg_right_hand_side in one launch, where there is a kernel for it.
bool tensor_weak_rhs(hgdg_ctx* c, const StageIO& io) {
    if (c->tm.general || c->op.kind != HGDG_OP_ACOUSTIC_CENTRAL) return false;
    // few cubes of order 5: the passes of the mass, one after another in a few
    // workgroups, take longer than another launch (6x7x5 14.9 us against 11.4,
    // 12^3 19.5 against 19.8)
    if (c->dim == 3 && c->tm.p == 5 && c->n_elem < 1024) return false;
    const AcousticParams a = acoustic_params(c, io);
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = AcousticShape<DIMc, N1c>;
        hipLaunchKernelGGL((tensor_acoustic_weak<DIMc, N1c>), dim3(unsigned((c->n_elem + S::EPB - 1) / S::EPB)),
                           dim3(S::THREADS), 0, c->stream, a);
    });
    HGDG_HIP(hipGetLastError());
    return true;
}

void tensor_rhs(hgdg_ctx* c, const StageIO& io) {
    if (c->tm.general) {
        tensor_general_rhs(c, io);
        return;
    }
    if (c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL) {
        const AcousticParams a = acoustic_params(c, io);
        dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
            constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
            using S = AcousticShape<DIMc, N1c>;
            const int64_t grid = (c->n_elem + S::EPB - 1) / S::EPB;
            // kTogether's registers at 3D p = 2 (177 against 164) leave two
            // wavefronts a SIMD instead of three, which costs large boxes more
            // than one further input gains (40^3 76 against 70 us; 24^3 the same)
            const bool many = !(DIMc == 3 && N1c == 3 && io.n_in == 3 && c->n_elem > 30 * 30 * 30);
            auto launch = [&](auto K) {
                constexpr int KIND = decltype(K)::value;
                // the update at 3D p = 3 is the one form that needs more registers
                // by its kind (280 against 225: one wavefront a SIMD instead of two);
                // kTogether beside it only where there is one in any case
                constexpr bool kAny = (DIMc == 3 && N1c == 4) ||
                                      ((KIND == STAGE_MANY || KIND == STAGE_MANY_MIXED) && !(DIMc == 3 && N1c == 6));
                constexpr int KU = kAny ? int(STAGE_ANY) : KIND;
                if (io.upd.u != nullptr)  // the fused RK update of a step's last stage
                    hipLaunchKernelGGL((tensor_acoustic_rhs<DIMc, N1c, KU, true>), dim3(unsigned(grid)),
                                       dim3(S::THREADS), 0, c->stream, a);
                else
                    hipLaunchKernelGGL((tensor_acoustic_rhs<DIMc, N1c, KIND, false>), dim3(unsigned(grid)),
                                       dim3(S::THREADS), 0, c->stream, a);
            };
            if (many) with_stage_kind<true>(io, launch);
            else with_stage_kind<false>(io, launch);
        });
        HGDG_HIP(hipGetLastError());
        return;
    }
    launch_advection(c, advection_params(c, io), c->adv_tiles);
}

void tensor_state_diff(hgdg_ctx* c, const Vec& vx, const Vec& vy, double* l2, double* max_abs) {
    if (c->tm.general) {
        tensor_general_state_diff(c, vx, vy, l2, max_abs);
        return;
    }
    DiffParams p{};
    p.n_elem = c->n_elem * c->n_fields;
    p.fields = c->n_fields;
    p.x = vx.ptr();
    p.y = vy.ptr();
    p.x_f32 = vx.is_f32;
    p.y_f32 = vy.is_f32;
    p.absdet = c->tm.d_absdet.ptr;
    p.M1 = M1_ptr(c);
    int64_t grid = 0;
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = Tensor<DIMc, N1c>;
        grid = (p.n_elem + S::EPB - 1) / S::EPB;
        if (c->d_partial.n < size_t(2 * grid)) c->d_partial.alloc(size_t(2 * grid));
        p.partial = c->d_partial.ptr;
        hipLaunchKernelGGL((tensor_diff_norm<DIMc, N1c>), dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, p);
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

void tensor_mass_apply(hgdg_ctx* c, Vec& v, bool inverse) {
    if (c->tm.general) {
        tensor_general_mass_apply(c, v, inverse);
        return;
    }
    require(!v.is_f32, HGDG_ERR_UNSUPPORTED, "mass apply/solve needs a vector stored in FP64");
    MassParams p{};
    p.n_blocks = c->n_elem * c->n_fields;
    p.fields = c->n_fields;
    p.inverse = inverse ? 1 : 0;
    p.v = v.f64->ptr;
    p.absdet = c->tm.d_absdet.ptr;
    p.cinv = c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL ? c->tm.d_geo.ptr + size_t(c->dim) * c->dim * c->n_elem : nullptr;
    p.A1 = inverse ? Mi_ptr(c) : M1_ptr(c);
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = Tensor<DIMc, N1c>;
        const int64_t grid = (p.n_blocks + S::EPB - 1) / S::EPB;
        hipLaunchKernelGGL((tensor_mass<DIMc, N1c>), dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, p);
    });
    HGDG_HIP(hipGetLastError());
}

void tensor_error_modes(hgdg_ctx* c, const Vec& v, int field, int n_modes, const double* amp, const double* k,
                        const double* shift, double* l2, double* max_abs) {
    if (c->tm.general) {
        tensor_general_error_modes(c, v, field, n_modes, amp, k, shift, l2, max_abs);
        return;
    }
    const int n1 = c->tm.n1, dim = c->dim;
    const int64_t ne = c->n_elem;
    std::vector<double> x2, w2, x1, w1;
    gauss_legendre(n1 + 1, x2, w2);
    gauss_legendre(n1, x1, w1);
    std::vector<double> tab;
    for (int a = 0; a < n1; ++a)
        for (int q = 0; q <= n1; ++q) tab.push_back(psi(a, x2[q]));
    tab.insert(tab.end(), w2.begin(), w2.end());
    tab.insert(tab.end(), x2.begin(), x2.end());
    for (int a = 0; a < n1; ++a)
        for (int q = 0; q < n1; ++q) tab.push_back(psi(a, x1[q]));
    tab.insert(tab.end(), x1.begin(), x1.end());
    for (int m = 0; m < n_modes; ++m) {
        tab.push_back(amp[m]);
        for (int d = 0; d < 3; ++d) tab.push_back(k[3 * m + d]);
    }
    // element origins and edge vectors, SoA
    std::vector<double> x0(size_t(dim) * ne), ed(size_t(dim) * dim * ne);
    for (int64_t e = 0; e < ne; ++e) {
        if (c->tm.structured) {
            const int64_t idx[3] = {e % c->tm.cells[0], (e / c->tm.cells[0]) % c->tm.cells[1],
                                    dim == 3 ? e / (int64_t(c->tm.cells[0]) * c->tm.cells[1]) : 0};
            for (int d = 0; d < dim; ++d) {
                x0[size_t(d) * ne + e] = double(idx[d]) / c->tm.cells[d];
                for (int r = 0; r < dim; ++r)
                    ed[(size_t(d) * dim + r) * ne + e] = r == d ? double(idx[d] + 1) / c->tm.cells[d] - double(idx[d]) / c->tm.cells[d] : 0.0;
            }
        } else {
            for (int d = 0; d < dim; ++d) {
                x0[size_t(d) * ne + e] = c->tm.X0[size_t(e) * dim + d];
                for (int r = 0; r < dim; ++r) ed[(size_t(d) * dim + r) * ne + e] = c->tm.E[(size_t(e) * dim + d) * dim + r];
            }
        }
    }
    DevBuf<double> d_tab, d_x0, d_e;
    d_tab.upload(tab, c->stream);
    d_x0.upload(x0, c->stream);
    d_e.upload(ed, c->stream);
    ErrParams p{};
    p.n_elem = ne;
    p.nf = c->n_fields;
    p.field = field;
    p.u = v.ptr();
    p.u_f32 = v.is_f32;
    p.n_modes = n_modes;
    p.modes = d_tab.ptr + (tab.size() - size_t(4) * n_modes);
    for (int d = 0; d < 3; ++d) p.shift[d] = shift ? shift[d] : 0.0;
    p.X0 = d_x0.ptr;
    p.E = d_e.ptr;
    p.absdet = c->tm.d_absdet.ptr;
    p.tab = d_tab.ptr;
    const int64_t grid = (ne + kBlock - 1) / kBlock;
    if (c->d_partial.n < size_t(2 * grid)) c->d_partial.alloc(size_t(2 * grid));
    p.partial = c->d_partial.ptr;
    dispatch_tensor(dim, n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        hipLaunchKernelGGL((tensor_error<DIMc, N1c>), dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, p);
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

// ---------------------------------------------------------------- batched launches
// Problems of one family (kind, dim, order) advance together: their per-problem
// parameter blocks go into `params` (device, written by the caller beforehand
// through `host_staging`), and one launch covers all their elements.
size_t tensor_batch_param_bytes(const hgdg_ctx* c) {
    return c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL ? sizeof(AcousticParams) : sizeof(RhsParams);
}

int64_t tensor_batch_blocks(const hgdg_ctx* c) {
    int64_t blocks = 0;
    dispatch_tensor(c->dim, c->tm.n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        const int64_t epb = c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL ? AcousticShape<DIMc, N1c>::EPB
                                                                   : Pencil<DIMc, N1c>::EPB;
        blocks = (c->n_elem + epb - 1) / epb;
    });
    return blocks;
}

void tensor_batch_param(hgdg_ctx* c, const StageIO& io, void* out) {
    if (c->op.kind == HGDG_OP_ACOUSTIC_CENTRAL) {
        const AcousticParams a = acoustic_params(c, io);
        std::memcpy(out, &a, sizeof(a));
    } else {
        RhsParams r{};
        r.n_elem = c->n_elem;
        r.io = io;
        r.ahat = c->tm.d_geo.ptr;
        r.nbr = c->tm.d_nbr.ptr;
        r.mode = c->tm.d_mode.ptr;
        r.face = c->tm.d_face.ptr;
        r.Dr = Dr_ptr(c);
        r.Mi = Mi_ptr(c);
        std::memcpy(out, &r, sizeof(r));
    }
}

void tensor_batch_launch(hipStream_t stream, int kind, int dim, int n1, bool mixed, bool upd, const void* params,
                         const int64_t* off, int n, int64_t blocks) {
    if (n == 0 || blocks == 0) return;
    dispatch_tensor(dim, n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        const dim3 grid{unsigned(blocks), 1, 1}, block{unsigned(kBlock), 1, 1};
        const dim3 acoustic_block{unsigned(AcousticShape<DIMc, N1c>::THREADS), 1, 1};
        auto go = [&](auto U) {
            constexpr bool Uc = decltype(U)::value;
            if (kind == HGDG_OP_ACOUSTIC_CENTRAL)
                hipLaunchKernelGGL((tensor_acoustic_rhs_batched<DIMc, N1c, Uc>), grid, acoustic_block, 0, stream,
                                   static_cast<const AcousticParams*>(params), off, n);
            else
                hipLaunchKernelGGL((tensor_advection_rhs_batched<DIMc, N1c, Uc>), grid, block, 0, stream,
                                   static_cast<const RhsParams*>(params), off, n);
        };
        if (upd) go(std::true_type{});
        else go(std::false_type{});
    });
    HGDG_HIP(hipGetLastError());
}

void tensor_project_device(hgdg_ctx* c, Vec& v, int field, int n_modes, const double* amp, const double* k,
                           const double* gauss) {
    if (c->tm.general) {
        tensor_general_project(c, v, field, n_modes, amp, k, gauss);
        return;
    }
    const int n1 = c->tm.n1, dim = c->dim;
    std::vector<double> xq, wq;
    gauss_legendre(n1, xq, wq);
    std::vector<double> P(size_t(n1) * n1, 0.0);
    for (int a = 0; a < n1; ++a)
        for (int q = 0; q < n1; ++q) {
            double s = 0;
            for (int b = 0; b < n1; ++b) s += c->tm.ops.Mi[a * n1 + b] * psi(b, xq[q]);
            P[a * n1 + q] = s * wq[q];
        }
    std::vector<double> tab(P);
    tab.insert(tab.end(), xq.begin(), xq.end());
    for (int m = 0; m < n_modes; ++m) {
        tab.push_back(amp[m]);
        for (int d = 0; d < 3; ++d) tab.push_back(k[3 * m + d]);
    }
    DevBuf<double> d_tab;
    d_tab.upload(tab, c->stream);
    DevBuf<double> d_x0, d_e;
    ProjParams pp{};
    pp.n_elem = c->n_elem;
    pp.nf = c->n_fields;
    pp.field = field;
    pp.out = v.ptr();
    pp.out_f32 = v.is_f32;
    pp.n_modes = n_modes;
    if (gauss) {
        pp.gaussian = 1;
        for (int q = 0; q < 5; ++q) pp.g[q] = gauss[q];
    }
    pp.P = d_tab.ptr;
    pp.xq = d_tab.ptr + size_t(n1) * n1;
    pp.modes = d_tab.ptr + size_t(n1) * n1 + n1;
    pp.structured = c->tm.structured;
    for (int d = 0; d < 3; ++d) pp.cells[d] = c->tm.cells[d];
    if (!c->tm.structured) {
        const int64_t ne = c->n_elem;
        std::vector<double> x0(size_t(dim) * ne), ed(size_t(dim) * dim * ne);
        for (int64_t e = 0; e < ne; ++e)
            for (int d = 0; d < dim; ++d) {
                x0[size_t(d) * ne + e] = c->tm.X0[size_t(e) * dim + d];
                for (int r = 0; r < dim; ++r) ed[(size_t(d) * dim + r) * ne + e] = c->tm.E[(size_t(e) * dim + d) * dim + r];
            }
        d_x0.upload(x0, c->stream);
        d_e.upload(ed, c->stream);
        pp.X0 = d_x0.ptr;
        pp.E = d_e.ptr;
    }
    dispatch_tensor(dim, n1, [&](auto D, auto N) {
        constexpr int DIMc = decltype(D)::value, N1c = decltype(N)::value;
        using S = Pencil<DIMc, N1c>;
        const int64_t grid = (c->n_elem + S::EPB - 1) / S::EPB;
        hipLaunchKernelGGL((tensor_project<DIMc, N1c>), dim3(unsigned(grid)), dim3(kBlock), 0, c->stream, pp);
    });
    HGDG_HIP(hipGetLastError());
    HGDG_HIP(hipStreamSynchronize(c->stream));  // before the temporary tables go
}

}  // namespace hgdg
