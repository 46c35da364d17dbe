// HIP kernels of the tri_hp_cns residual/relaxation path (gfx950): compressible
// Navier-Stokes in the primitive variables (p, u, v, RT), steady, straight-sided
// elements, diagonal preconditioner with the per-vertex 4x4 block preconditioner of
// the primitive-variable projection.
//
// Element residual: the matrix-core layout of tri_kernels.hip (16 elements per wave, every
// transform a contraction on v_mfma_f64_16x16x4f64 or v_mfma_f32_16x16x4f32), with the
// pointwise physics -- the stabilisation solve at every Gauss point above all -- in the
// lane that holds the point; project_new_variables' interior sweep likewise.
#include <hip/hip_runtime.h>
#include "tri_kernels.h"

namespace hpg {

constexpr int NVC = 4;

struct CnsPhys {
    double mu, kcond, Rgas, gamma, adis;
};

// per-level operator pack for the cns kernels (doubles): proj operators transposed
// to [mode][32 points], derivative operators to [point'][32 points], integration
// operators to [point][16 modes]; padded entries are zero
template <int P>
struct CDims {
    static constexpr int TM = Dims<P>::TM, SM = Dims<P>::SM, IM = Dims<P>::IM, BM = Dims<P>::BM, G = Dims<P>::G;
    static constexpr int OP_P = 0, OP_PR = TM * 32, OP_PS = 2 * TM * 32, OP_DR = 3 * TM * 32;
    static constexpr int OP_DS = OP_DR + G * 32, OP_IR = OP_DS + G * 32, OP_IS = OP_IR + G * 16;
    static constexpr int SIZE = OP_IS + G * 16;
};

// ---------------------------------------------------------------------------------
// 4x4 helpers
template <typename T>
__device__ __forceinline__ void mm4(const T A[4][4], const T B[4][4], T C[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            T t = T(0.0);
#pragma unroll
            for (int k = 0; k < 4; ++k) t += A[i][k] * B[k][j];
            C[i][j] = t;
        }
}

// Solves A X = B for the four columns of B (overwritten by X); Gaussian elimination
// with partial pivoting (first row of largest |pivot|), A is destroyed.  Row swaps
// are unrolled selects so that everything stays in registers.
template <typename T>
__device__ __forceinline__ void solve4(T a[4][4], T b[4][4]) {
    int piv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        int p = k;
        T best = fabs(a[k][k]);
#pragma unroll
        for (int r = k + 1; r < 4; ++r) {
            const T v = fabs(a[r][k]);
            if (v > best) { best = v; p = r; }
        }
        piv[k] = p;
#pragma unroll
        for (int r = k + 1; r < 4; ++r)
            if (p == r) {
#pragma unroll
                for (int c = 0; c < 4; ++c) { const T tmp = a[k][c]; a[k][c] = a[r][c]; a[r][c] = tmp; }
            }
        const T inv = T(1.0) / a[k][k];
#pragma unroll
        for (int r = k + 1; r < 4; ++r) {
            a[r][k] *= inv;
            const T f = a[r][k];
            if (f != T(0.0)) {
#pragma unroll
                for (int c = k + 1; c < 4; ++c) a[r][c] -= f * a[k][c];
            }
        }
    }
#pragma unroll
    for (int col = 0; col < 4; ++col) {
        T x[4] = {b[0][col], b[1][col], b[2][col], b[3][col]};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int r = k + 1; r < 4; ++r)
                if (piv[k] == r) { const T tmp = x[k]; x[k] = x[r]; x[r] = tmp; }
#pragma unroll
        for (int r = 1; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < r; ++c) x[r] -= a[r][c] * x[c];
#pragma unroll
        for (int r = 3; r >= 0; --r) {
#pragma unroll
            for (int c = r + 1; c < 4; ++c) x[r] -= a[r][c] * x[c];
            x[r] /= a[r][r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r][col] = x[r];
    }
}

// utilities/matrix.cpp:16-37: 20 power iterations from x = 1 and the Rayleigh quotient
template <typename T>
__device__ __forceinline__ T spectral_radius4(const T A[4][4]) {
    T x[4] = {T(1.0), T(1.0), T(1.0), T(1.0)}, t[4] = {T(0.0), T(0.0), T(0.0), T(0.0)};
    for (int it = 0; it < 20; ++it) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            T s = T(0.0);
#pragma unroll
            for (int j = 0; j < 4; ++j) s += A[i][j] * x[j];
            t[i] = s;
        }
        T s = T(0.0);
#pragma unroll
        for (int i = 0; i < 4; ++i) s += t[i] * t[i];
        const T nrm = sqrt(s);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = t[i] / nrm;
    }
    T num = T(0.0), den = T(0.0);
#pragma unroll
    for (int i = 0; i < 4; ++i) num += x[i] * t[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) den += x[i] * x[i];
    return fabs(num / den);
}

// tri_hp_cns::calculate_tau (tri_hp/cns/setup_preconditioner.cpp:241-515), steady
// (hdt = 0) and with alph = 0 as the reference forces it: Pinv (the inverse of the
// low-Mach preconditioner), Tau = Tinv^-1 P with Tinv = 2(|A| + |B| + h S)/h, and,
// when requested, timestep = 1/spectral_radius(Tinv).
template <typename T>
__device__ __forceinline__ void cns_tau(const CnsPhys& ph, T pr, T u, T v, T rt, T h,
                                        T Pinv[4][4], T Tau[4][4], T* timestep) {
    const T gam = T(ph.gamma), gm1 = gam - T(1.0), gogm1 = gam / gm1;
    const T rho = pr / rt, ke = T(0.5) * (u * u + v * v), c2 = gam * rt, c = sqrt(c2);
    const T nu = T(ph.mu) / rho, cp = gogm1 * T(ph.Rgas), alpha = T(ph.kcond) / (rho * cp);
    const T umag = sqrt(u * u + v * v);
    const T M = (umag / c > T(1.0e-5)) ? umag / c : T(1.0e-5);
    const T nuh = T(4.0) * nu / (h * c);
    const T alh = T(2.0) * alpha / (h * c);
    T b2 = T(1.0);
    if (M < T(0.8)) {
        const T s = M * M / (T(1.0) - M * M) + T(0.0) * T(0.0) + nuh * nuh + alh * alh;
        b2 = (s < T(1.0)) ? s : T(1.0);
    }
    // alph = 0: P and Pinv have b2 on (0,0) and the (3,0) coupling only
    T P[4][4] = {{b2, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 1, 0}, {(b2 - T(1.0)) / (gogm1 * rho), 0, 0, 1}};
    const T Pi[4][4] = {{T(1.0) / b2, 0, 0, 0}, {0, 1, 0, 0}, {0, 0, 1, 0}, {-(b2 - T(1.0)) / (gogm1 * rho * b2), 0, 0, 1}};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) Pinv[i][j] = Pi[i][j];
    const T dpdc[4][4] = {{ke * gm1, -u * gm1, -v * gm1, gm1},
                               {-u / rho, T(1.0) / rho, 0, 0},
                               {-v / rho, 0, T(1.0) / rho, 0},
                               {(gm1 * ke - rt) / rho, -u * gm1 / rho, -v * gm1 / rho, gm1 / rho}};
    {
        T t[4][4];
        mm4(P, dpdc, t);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) P[i][j] = t[i][j];
    }
    T Tinv[4][4];
    {
        const T temp1 = sqrt(u * u * (T(1.0) - T(2.0) * b2 + b2 * b2) + T(4.0) * b2 * c2);
        const T V[4][4] = {{T(0.5) * (u * (b2 - T(1.0)) + temp1) * rho, T(0.5) * (u * (b2 - T(1.0)) - temp1) * rho, 0, 0},
                                {1, 1, 0, 0},
                                {0, 0, 1, 0},
                                {T(0.5) * (u * (b2 - T(1.0)) * gm1 + gm1 * temp1) / gam, T(0.5) * (u * (b2 - T(1.0)) * gm1 - gm1 * temp1) / gam, 0, 1}};
        const T e[4] = {fabs(T(0.5) * (u + u * b2 + temp1)), fabs(T(0.5) * (u + u * b2 - temp1)), fabs(u), fabs(u)};
        T W[4][4] = {{T(1.0) / (temp1 * rho), -T(0.5) * (u * (b2 - T(1.0)) - temp1) / temp1, 0, 0},
                          {-T(1.0) / (temp1 * rho), T(0.5) * (u * (b2 - T(1.0)) + temp1) / temp1, 0, 0},
                          {0, 0, 1, 0},
                          {-gm1 / (gam * rho), 0, 0, 1}};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) W[i][j] = e[i] * W[i][j];
        mm4(V, W, Tinv);  // |A|
    }
    {
        const T temp2 = sqrt(v * v * (T(1.0) - T(2.0) * b2 + b2 * b2) + T(4.0) * b2 * c2);
        const T V[4][4] = {{0, 0, T(0.5) * (v * (b2 - T(1.0)) + temp2) * rho, T(0.5) * (v * (b2 - T(1.0)) - temp2) * rho},
                                {0, 1, 0, 0},
                                {0, 0, 1, 1},
                                {1, 0, T(0.5) * (gm1 * v * (b2 - T(1.0)) + gm1 * temp2) / gam, T(0.5) * (gm1 * v * (b2 - T(1.0)) - gm1 * temp2) / gam}};
        const T e[4] = {fabs(v), fabs(v), fabs(T(0.5) * (v + v * b2 + temp2)), fabs(T(0.5) * (v + v * b2 - temp2))};
        T W[4][4] = {{-gm1 / (gam * rho), 0, 0, 1},
                          {0, 1, 0, 0},
                          {T(1.0) / (temp2 * rho), 0, T(0.5) * (-v * (b2 - T(1.0)) + temp2) / temp2, 0},
                          {-T(1.0) / (rho * temp2), 0, T(0.5) * (v * (b2 - T(1.0)) + temp2) / temp2, 0}};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) W[i][j] = e[i] * W[i][j];
        T B[4][4];
        mm4(V, W, B);
        const T Sd[4][4] = {{0, 0, 0, 0}, {0, nu / (h * h), 0, 0}, {0, 0, nu / (h * h), 0}, {0, 0, 0, alpha / (h * h)}};
        T S[4][4];
        mm4(P, Sd, S);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) Tinv[i][j] = T(2.0) * (Tinv[i][j] + B[i][j] + h * S[i][j]) / h;
    }
    if (timestep) *timestep = T(1.0) / spectral_radius4(Tinv);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) Tau[i][j] = P[i][j];
    solve4(Tinv, Tau);
}

// conservative -> primitive change at state (p, u, v, RT) (tri_hp/cns/update.cpp:247-271);
// written with one division (the matrix form has ten, and the projections are bound by
// their pointwise FP64 work)
__device__ __forceinline__ void switch_vars(const double w[4], double a[4], double gm1) {
    const double u = w[1], v = w[2], rt = w[3], irho = rt / w[0];
    const double z = gm1 * (0.5 * (u * u + v * v) * a[0] - u * a[1] - v * a[2] + a[3]);
    a[1] = irho * (a[1] - u * a[0]);
    a[2] = irho * (a[2] - v * a[0]);
    a[3] = irho * (z - rt * a[0]);
    a[0] = z;
}

// forward substitution with the lower triangle (diagonal included) of a row-major 4x4
__device__ __forceinline__ void lower4(const double L[16], double r[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        double l0 = r[j];
#pragma unroll
        for (int k = 0; k < j; ++k) l0 -= L[j * 4 + k] * r[k];
        r[j] = l0 / L[j * 4 + j];
    }
}

// ---------------------------------------------------------------------------------
// T: arithmetic type of the element kernel (double, or float in the FP32 inner solve of
// the defect correction); the state and residual arrays are FP64 in both
template <typename T>
struct CnsElemArgsT {
    const double* pnts;
    const int* tri_pnt;
    const int* tri_seg;
    const int* tri_sgn;
    const int* order;  // null: mesh order
    int begin, end;
    const double* ugv;
    const double* ugs;
    const double* ugi;
    double* resi;
    double* rri;
    double* eres;  // element-major vertex and side modes, (element, 3p, im | re, 4); stages
                   // without the real part (element, 3p, 4)
    const T* ops;  // double: the operator pack of the ins element kernel; float: CDims pack
    int sm0, im0;
    CnsPhys ph;
    double beta, keep;
    // FP32 kernel: constant source sfac[0] * srci of the interior modes (the scaled FP64
    // residual of the defect correction); null otherwise
    const double* srci;
    const double* sfac;
    // FP32 kernel: each element's colour and the first colour at each vertex and side
    const unsigned char* tcol;
    const unsigned char* fcv;
    const unsigned char* fcs;
    int colour;
    // element Jacobians: as ElemArgsT
    int jcols;
    double jeps_r, jeps_a;
    double* jbase;
    double* jK;
};
typedef CnsElemArgsT<double> CnsElemArgs;
typedef CnsElemArgsT<float> CnsElemArgs32;

// octet loop of the persistent element kernels: XCD x of the 8 walks the contiguous
// octet range [x*per, (x+1)*per) with the gridDim/8 blocks it is given
// LDS exchange among the lanes of one wave.  Every LDS buffer written inside the
// octet loops is private to a half-wave, so ordering the wave's own LDS accesses is
// enough: a wave's LDS instructions complete in issue order, and the fences and
// wave barrier keep the compiler from moving memory operations across this point.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

#define HPG_OCTET_LOOP_OF(noct, oc, blk, nblk)                                            \
    const int nbx_ = (nblk) >> 3, xcd_ = (blk) & 7, jb_ = (blk) >> 3;                      \
    const int per_ = ((noct) + 7) / 8;                                                     \
    const int oend_ = min((xcd_ + 1) * per_, (noct));                                      \
    for (int oc = xcd_ * per_ + jb_; oc < oend_; oc += nbx_)
#define HPG_OCTET_LOOP(noct, oc) HPG_OCTET_LOOP_OF(noct, oc, (int)blockIdx.x, (int)gridDim.x)

// Stabilised residual Tau res at one Gauss point, Tau = Tinv^-1 P dpdc with
// Tinv = 2 (|A| + |B| + h S) / h (tri_hp/cns/setup_preconditioner.cpp:241-515, alph = 0,
// hdt = 0; the full matrices are cns_tau).  Only one right-hand side is needed here, and
// the closed forms leave few entries: with |A| = V |L| W written out, Tinv couples u and v
// to p alone, so rows 1 and 2 are eliminated by their own positive pivots and a 2 x 2
// system in (p, RT) remains.  About 200 operations against about 700 for the general
// products and a four-column solve.
struct CnsStab {
    double gam, gm1, gogm1, kg, mu, acp, h, ih, hh;
};

__device__ __forceinline__ void cns_stab(const CnsStab& k, double pr, double u, double v, double rt, const double* res, double* x) {
    const double irho = rt / pr, rho = pr / rt;
    const double qq = u * u + v * v, ke = 0.5 * qq, c2 = k.gam * rt;
    const double ic = 1.0 / sqrt(c2);  // NaN for RT < 0, as every quantity below
    const double nu = k.mu * irho, al = k.acp * irho;
    const double m2u = qq * ic * ic;
    const double m2 = m2u > 1e-10 ? m2u : 1e-10;
    double b2 = 1.0;
    if (m2 < 0.64) {
        const double hc = k.ih * ic, a = 4.0 * nu * hc, b = 2.0 * al * hc;
        const double s = m2 / (1.0 - m2) + a * a + b * b;
        b2 = s < 1.0 ? s : 1.0;
    }
    const double bm = b2 - 1.0, c3 = bm * irho / k.gogm1;
    const double f4 = 4.0 * b2 * c2, bb = 1.0 - 2.0 * b2 + b2 * b2;
    // |A|: eigenvalues e0, e1, |u| with p, m the roots of the acoustic pair
    const double t1 = sqrt(u * u * bb + f4), it1 = 1.0 / t1;
    const double p1 = 0.5 * (u * bm + t1), m1 = 0.5 * (u * bm - t1);
    const double e0 = fabs(0.5 * (u + u * b2 + t1)) * it1, e1 = fabs(0.5 * (u + u * b2 - t1)) * it1;
    const double au = fabs(u), av = fabs(v);
    const double A00 = p1 * e0 - m1 * e1, A01 = p1 * m1 * (e1 - e0), A10 = irho * (e0 - e1), A11 = p1 * e1 - m1 * e0;
    const double t2 = sqrt(v * v * bb + f4), it2 = 1.0 / t2;
    const double p2 = 0.5 * (v * bm + t2), n2 = 0.5 * (v * bm - t2);
    const double g0 = fabs(0.5 * (v + v * b2 + t2)) * it2, g1 = fabs(0.5 * (v + v * b2 - t2)) * it2;
    const double B00 = p2 * g0 - n2 * g1, B02 = p2 * n2 * (g1 - g0), B20 = irho * (g0 - g1), B22 = p2 * g1 - n2 * g0;
    // h S = h (P dpdc) diag(0, nu, nu, alpha) / h^2
    const double Dn = nu * k.ih, Da = al * k.ih, w = k.gm1 * (irho + c3), kr = k.kg * irho;
    const double M00 = A00 + B00, M01 = rho * A01 - b2 * k.gm1 * u * Dn, M02 = rho * B02 - b2 * k.gm1 * v * Dn;
    const double M03 = b2 * k.gm1 * Da;
    const double M11 = A11 + av + irho * Dn, M22 = au + B22 + irho * Dn;
    const double M30 = kr * (A00 - au) + kr * (B00 - av), M31 = k.kg * A01 - w * u * Dn, M32 = k.kg * B02 - w * v * Dn;
    const double M33 = au + av + w * Da;
    // P dpdc res
    const double z = k.gm1 * (ke * res[0] - u * res[1] - v * res[2] + res[3]);
    const double r0 = b2 * z, r1 = irho * (res[1] - u * res[0]), r2 = irho * (res[2] - v * res[0]);
    const double r3 = irho * (z - rt * res[0]) + c3 * z;
    const double i1 = 1.0 / M11, i2 = 1.0 / M22;
    const double a1 = A10 * i1, a2 = B20 * i2, y1 = r1 * i1, y2 = r2 * i2;
    const double d00 = M00 - M01 * a1 - M02 * a2, d30 = M30 - M31 * a1 - M32 * a2;
    const double s0 = r0 - M01 * y1 - M02 * y2, s3 = r3 - M31 * y1 - M32 * y2;
    const double q = d30 / d00;
    const double x3 = (s3 - q * s0) / (M33 - q * M03);
    const double x0 = (s0 - M03 * x3) / d00;
    x[0] = k.hh * x0;
    x[1] = k.hh * (y1 - a1 * x0);
    x[2] = k.hh * (y2 - a2 * x0);
    x[3] = k.hh * x3;
}

// tri_hp_cns::element_rsdl, straight branch (tri_hp/cns/rsdl.cpp:312-530), steady, source
// "zero", CALC_TAU2 (tau at every Gauss point), 16 elements per wave in the layout of
// elem_ins_body: operators of the ins pack, accumulators fed back as operands, element-major
// output.  Fluxes are formed right before the matrix instructions that consume them; the
// values (U), the viscous fluxes (F) and the strong residual (R) of the element's points
// stay in registers.  JAC: entries are (element, column) pairs as in elem_ins_body.
template <int P, bool FULL, bool JAC = false>
__device__ __forceinline__ void elem_cns_body(const CnsElemArgs& a, int eblk = 0) {
    using D = Dims<P>;
    using T = double;
    using V4 = d4;
    constexpr int GT = D::GT, KT = D::KT;
    __shared__ T sops[D::PACK];
    for (int k = threadIdx.x; k < D::PACK; k += blockDim.x) sops[k] = a.ops[k];
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int e = lane & 15, q = lane >> 4;
    const int WX = (((int)gridDim.x - eblk) >> 3) * 4;
    const int rank = (((int)blockIdx.x - eblk) >> 3) * 4 + wv;
    const int xcd = blockIdx.x & 7;
    const int ng = (a.end - a.begin + 15) >> 4;
    const int gpx = (ng + 7) >> 3;
    const int g0 = xcd * gpx + rank;
    const int gend = min(ng, (xcd + 1) * gpx);
    if (g0 >= gend) return;

    CnsStab ks;
    ks.gam = T(a.ph.gamma);
    ks.gm1 = ks.gam - T(1);
    ks.gogm1 = ks.gam / ks.gm1;
    ks.kg = ks.gm1 / ks.gam;
    ks.mu = T(a.ph.mu);
    ks.acp = T(a.ph.kcond) / (ks.gogm1 * T(a.ph.Rgas));
    const T igm1 = T(1) / ks.gm1;
    // a K-step (tile kt, register i; points 16 kt + 4 i + q) of padding points adds nothing
    auto dead = [](int kt, int i) { return 16 * kt + 4 * i >= D::G; };

    ElemSlots<P> S = elem_slots<P, NVC>(a, elem_conn(a, elem_of_group<JAC>(a, g0, gend, e)), q);
    ElemConn cnext = elem_conn(a, elem_of_group<JAC>(a, g0 + WX, gend, e));
    int tnext2 = elem_of_group<JAC>(a, g0 + 2 * WX, gend, e);
    for (int g = g0; g < gend; g += WX) {
        const ElemSlots<P> Sn = elem_slots<P, NVC>(a, cnext, q);
        const ElemConn cn2 = elem_conn(a, tnext2);
        const int tn3 = elem_of_group<JAC>(a, g + 3 * WX, gend, e);

        // modal coefficients: K-step s of lane l is mode 4s + l/16; padding elements carry
        // p = RT = 1 in their vertex modes
        T b[NVC][KT];
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = 4 * s + q, kind = mode_kind<P>(k);
            const bool live = S.t >= 0 && k < D::TM;
            const int off = S.off[s] < 0 ? ~S.off[s] : S.off[s];
            const T sg = S.off[s] < 0 ? T(-1) : T(1);
            const double* src = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
#pragma unroll
            for (int n = 0; n < NVC; ++n)
                b[n][s] = live ? sg * T(src[off + n]) : ((k < 3 && (n == 0 || n == 3)) ? T(1) : T(0));
        }
        int jcol = 0, jel = 0;
        T jdw = T(1);
        if constexpr (JAC) {
            const int idx = a.begin + g * 16 + e;
            jel = idx / a.jcols;
            jcol = idx - jel * a.jcols;
            if (a.jK) {
                const int jm = jcol / NVC, jn = jcol - jm * NVC;
#pragma unroll
                for (int n = 0; n < NVC; ++n) {
                    T v = T(0);
#pragma unroll
                    for (int k = 0; k < 3; ++k) v = v + fabs(__shfl(b[n][0], 16 * k + e, 64));
                    const T dw = v * T(a.jeps_r) + T(a.jeps_a);
                    if (n != jn) continue;
                    jdw = dw;
#pragma unroll
                    for (int s = 0; s < KT; ++s)
                        if (4 * s + q == jm && S.t >= 0) b[n][s] += dw;
                }
            }
        }
        const double x0 = S.x[0], y0 = S.y[0], x1 = S.x[1], y1 = S.y[1], x2 = S.x[2], y2 = S.y[2];
        // ldcrd(n,0) = dx_n/dr, ldcrd(n,1) = dx_n/ds (rsdl.cpp:56-59)
        const T l00 = T(0.5 * (x2 - x1)), l01 = T(0.5 * (x0 - x1));
        const T l10 = T(0.5 * (y2 - y1)), l11 = T(0.5 * (y0 - y1));

        const V4 zz = {T(0), T(0), T(0), T(0)};
        V4 U[NVC][GT];
#pragma unroll
        for (int mt = 0; mt < GT; ++mt) {
            V4 c[NVC] = {zz, zz, zz, zz};
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const T av = sops[D::OFF_P + (mt * KT + s) * 64 + lane];
#pragma unroll
                for (int n = 0; n < NVC; ++n) c[n] = mfma(av, b[n][s], c[n]);
            }
            // padding rows of the point tiles: p = u = v = RT = 1, where the pointwise work
            // is finite also for mu = 0 (a zero operator column does not cancel a NaN)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (16 * mt + 4 * i + q >= D::G) { c[0][i] = T(1); c[1][i] = T(1); c[2][i] = T(1); c[3][i] = T(1); }
#pragma unroll
            for (int n = 0; n < NVC; ++n) U[n][mt] = c[n];
        }
        // convective fluxes of point (kt, i) (rsdl.cpp:315-351)
        auto conv = [&](int kt, int i, T* cv) {
            const T pr = U[0][kt][i], u = U[1][kt][i], v = U[2][kt][i], rt = U[3][kt][i];
            const T rho = pr / rt, fx = rho * u, fy = rho * v;
            cv[0] = l11 * fx - l01 * fy;
            cv[1] = -l10 * fx + l00 * fy;
            cv[2] = u * cv[0] + l11 * pr;
            cv[3] = u * cv[1] - l10 * pr;
            cv[4] = v * cv[0] - l01 * pr;
            cv[5] = v * cv[1] + l00 * pr;
            const T E = rt * igm1 + T(0.5) * (u * u + v * v);
            const T nx = E * fx + pr * u, ny = E * fy + pr * v;
            cv[6] = l11 * nx - l01 * ny;
            cv[7] = -l10 * nx + l00 * ny;
        };

        V4 LI[NVC] = {zz, zz, zz, zz}, LR[NVC] = {zz, zz, zz, zz};
        if constexpr (!FULL) {
#pragma unroll
            for (int kt = 0; kt < GT; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (dead(kt, i)) continue;
                    T cv[8];
                    conv(kt, i, cv);
                    const T ar = sops[D::OFF_IR + (kt * 4 + i) * 64 + lane];
                    const T as = sops[D::OFF_IS + (kt * 4 + i) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < NVC; ++n) {
                        LI[n] = mfma(ar, cv[2 * n], LI[n]);
                        LI[n] = mfma(as, cv[2 * n + 1], LI[n]);
                    }
                }
        } else {
            // viscous stress and heat flux coefficients (rsdl.cpp:355-380), rhorbd0 = 0
            const T cjcb = l00 * l11 - l10 * l01;
            const T mj = ks.mu / cjcb, kj = T(a.ph.kcond) / cjcb / T(a.ph.Rgas);
            const T f43 = T(4.) / T(3.), f23 = T(2.) / T(3.), f13 = T(1.) / T(3.);
            const T v0000 = -mj * (f43 * l11 * l11 + l01 * l01), v0011 = -mj * (f43 * l10 * l10 + l00 * l00);
            const T v0001 = mj * (f43 * l11 * l10 + l01 * l00);
            const T v1100 = -mj * (l11 * l11 + f43 * l01 * l01), v1111 = -mj * (l10 * l10 + f43 * l00 * l00);
            const T v1101 = mj * (l11 * l10 + f43 * l01 * l00);
            const T v0100 = mj * f13 * l01 * l11, v0111 = mj * f13 * l00 * l10;
            const T v0101 = -mj * (l01 * l10 - f23 * l00 * l11), v0110 = -mj * (l00 * l11 - f23 * l01 * l10);
            const T k00 = -kj * (l11 * l11 + l01 * l01), k11 = -kj * (l10 * l10 + l00 * l00);
            const T k01 = kj * (l11 * l10 + l01 * l00);
            T F[GT][4][6];
            V4 R[NVC][GT];
#pragma unroll
            for (int mt = 0; mt < GT; ++mt)
#pragma unroll
                for (int n = 0; n < NVC; ++n) R[n][mt] = zz;
#pragma unroll
            for (int kt = 0; kt < GT; ++kt) {
                V4 dr[3] = {zz, zz, zz}, ds[3] = {zz, zz, zz};  // of u, v, RT on point tile kt
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    const T ar = sops[D::OFF_PR + (kt * KT + s) * 64 + lane];
                    const T as = sops[D::OFF_PS + (kt * KT + s) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        dr[n] = mfma(ar, b[n + 1][s], dr[n]);
                        ds[n] = mfma(as, b[n + 1][s], ds[n]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (dead(kt, i)) continue;
                    if (GT > 1) __builtin_amdgcn_sched_barrier(0);
                    T cv[8];
                    conv(kt, i, cv);
                    const T ar = sops[D::OFF_IR + (kt * 4 + i) * 64 + lane];
                    const T as = sops[D::OFF_IS + (kt * 4 + i) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < NVC; ++n) {
                        LI[n] = mfma(ar, cv[2 * n], LI[n]);
                        LI[n] = mfma(as, cv[2 * n + 1], LI[n]);
                    }
                    const T ur = dr[0][i], vr = dr[1][i], tr = dr[2][i], us = ds[0][i], vs = ds[1][i], ts = ds[2][i];
                    const T u = U[1][kt][i], v = U[2][kt][i];
                    T* f = F[kt][i];
                    f[0] = v0000 * ur + v0100 * vr + v0001 * us + v0101 * vs;
                    f[1] = v0001 * ur + v0110 * vr + v0011 * us + v0111 * vs;
                    f[2] = v0100 * ur + v1100 * vr + v0110 * us + v1101 * vs;
                    f[3] = v0101 * ur + v1101 * vr + v0111 * us + v1111 * vs;
                    f[4] = k00 * tr + k01 * ts + f[0] * u + f[2] * v;
                    f[5] = k01 * tr + k11 * ts + f[1] * u + f[3] * v;
#pragma unroll
                    for (int j = 0; j < 6; ++j) cv[j + 2] += f[j];
                    // strong residual: derivr/derivs of the total fluxes (rsdl.cpp:425-429)
#pragma unroll
                    for (int mt = 0; mt < GT; ++mt) {
                        const T odr = sops[D::OFF_DR + ((mt * GT + kt) * 4 + i) * 64 + lane];
                        const T ods = sops[D::OFF_DS + ((mt * GT + kt) * 4 + i) * 64 + lane];
#pragma unroll
                        for (int n = 0; n < NVC; ++n) {
                            R[n][mt] = mfma(odr, cv[2 * n], R[n][mt]);
                            R[n][mt] = mfma(ods, cv[2 * n + 1], R[n][mt]);
                        }
                    }
                }
            }
            // CALC_TAU2 (rsdl.cpp:431-452), the stabilisation (:454-488) and
            // lf_re = intgrtrs(viscous - stabilisation fluxes) (:490-497)
            const T dx1 = T(x0 - x2), dy1 = T(y0 - y2), dx2 = T(x1 - x0), dy2 = T(y1 - y0);
            const T ar2 = dx1 * dy2 - dy1 * dx2;
            const T perim = sqrt(dx1 * dx1 + dy1 * dy1) + sqrt(dx2 * dx2 + dy2 * dy2) +
                            sqrt((dx1 + dx2) * (dx1 + dx2) + (dy1 + dy2) * (dy1 + dy2));
            ks.h = T(0.25) * ar2 / ((ar2 / perim) * (T(0.25) * (P + 1) * (P + 1)));
            ks.ih = T(1) / ks.h;
            ks.hh = T(0.5) * ks.h * (T(a.ph.adis) / cjcb);
#pragma unroll
            for (int kt = 0; kt < GT; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (dead(kt, i)) continue;
                    const T pr = U[0][kt][i], u = U[1][kt][i], v = U[2][kt][i], rt = U[3][kt][i];
                    const T res[4] = {R[0][kt][i], R[1][kt][i], R[2][kt][i], R[3][kt][i]};
                    if (GT > 1) __builtin_amdgcn_sched_barrier(0);  // one point's solve at a time (registers)
                    T x[4];
                    cns_stab(ks, pr, u, v, rt, res, x);
                    // the primitive flux Jacobians A, B times x
                    const T rho = pr / rt, H = ks.gogm1 * rt + T(0.5) * (u * u + v * v);
                    const T dr = (x[0] - rho * x[3]) / rt;
                    const T fa0 = u * dr + rho * x[1], fb0 = v * dr + rho * x[2];
                    const T ru = rho * u, rv = rho * v;
                    const T fa1 = u * fa0 + ru * x[1] + x[0], fb2 = v * fb0 + rv * x[2] + x[0];
                    const T fab = u * fb0 + rv * x[1];
                    const T en = u * x[1] + v * x[2] + ks.gogm1 * x[3];
                    const T fa3 = H * fa0 + ru * en, fb3 = H * fb0 + rv * en;
                    const T* f = F[kt][i];
                    const T w[8] = {-(l11 * fa0 - l01 * fb0),        -(l00 * fb0 - l10 * fa0),
                                    f[0] - (l11 * fa1 - l01 * fab), f[1] - (l00 * fab - l10 * fa1),
                                    f[2] - (l11 * fab - l01 * fb2), f[3] - (l00 * fb2 - l10 * fab),
                                    f[4] - (l11 * fa3 - l01 * fb3), f[5] - (l00 * fb3 - l10 * fa3)};
                    const T ar = sops[D::OFF_IR + (kt * 4 + i) * 64 + lane];
                    const T as = sops[D::OFF_IS + (kt * 4 + i) * 64 + lane];
#pragma unroll
                    for (int n = 0; n < NVC; ++n) {
                        LR[n] = mfma(ar, w[2 * n], LR[n]);
                        LR[n] = mfma(as, w[2 * n + 1], LR[n]);
                    }
                }
        }

        const T bt = T(a.beta);
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = 4 * s + q, kind = mode_kind<P>(k);
            if (S.t < 0 || k >= D::TM) continue;
            const T sg = S.off[s] < 0 ? T(-1) : T(1);
            if constexpr (JAC) {
                constexpr int N = D::TM * NVC;
#pragma unroll
                for (int n = 0; n < NVC; ++n) {
                    const T rr = FULL ? LR[n][s] * bt + LI[n][s] : LI[n][s];
                    const size_t r = (size_t)jel * N + (k * NVC + n);
                    if (a.jK) a.jK[r * N + jcol] = (rr - a.jbase[r]) / jdw;
                    else a.jbase[r] = rr;
                }
            } else if (kind < 2) {
                double* o = a.eres + ((size_t)S.t * D::BM + k) * (FULL ? 2 * NVC : NVC);
#pragma unroll
                for (int n = 0; n < NVC; ++n) {
                    o[n] = sg * LI[n][s];
                    if constexpr (FULL) o[NVC + n] = sg * (LR[n][s] * bt);
                }
            } else {
                const int off = S.off[s];
#pragma unroll
                for (int n = 0; n < NVC; ++n) {
                    const double r0 = a.keep == 0.0 ? 0.0 : a.keep * a.rri[off + n];
                    const double lr = FULL ? LR[n][s] * bt : 0.0;
                    if (FULL || a.keep != 1.0) a.rri[off + n] = r0 + lr;
                    a.resi[off + n] = r0 + lr + LI[n][s];
                }
            }
        }
        S = Sn;
        cnext = cn2;
        tnext2 = tn3;
    }
}

// ---------------------------------------------------------------------------------
// edge-boundary flux residual (tri_hp/hp_boundary.cpp:973-1049) with the
// bdry_cns::generic flux (tri_hp/cns/bdry.cpp:192-245); p_bc = boundary pressure
struct CnsEdgeArgs {
    const int* eseg;
    int end;
    const int* seg_pnt;
    const double* pnts;
    const double* ugv;
    const double* ugs;
    double* eout;  // (edge, 2 ends then the side modes, 4), added by the gathers
    const double* g1;
    const double* dg1;
    const double* w1;
    int sm0;
    double gamma, pbc;
};

template <int P>
__device__ __forceinline__ void edge_cns_body(const CnsEdgeArgs& a, int idx) {
    constexpr int SM = Dims<P>::SM, N1 = SM + 2, GPX = P + 1;
    if (idx >= a.end) return;
    const int sind = a.eseg[idx];
    const int v0 = a.seg_pnt[2 * sind], v1 = a.seg_pnt[2 * sind + 1];
    double uh[NVC][N1];
#pragma unroll
    for (int n = 0; n < NVC; ++n) {
        uh[n][0] = a.ugv[v0 * NVC + n];
        uh[n][1] = a.ugv[v1 * NVC + n];
#pragma unroll
        for (int m = 0; m < SM; ++m) uh[n][m + 2] = a.ugs[(sind * a.sm0 + m) * NVC + n];
    }
    const double X0 = a.pnts[2 * v0], Y0 = a.pnts[2 * v0 + 1], X1 = a.pnts[2 * v1], Y1 = a.pnts[2 * v1 + 1];
    const double gm1 = a.gamma - 1.0, pbc = a.pbc;
    double lf[NVC][N1];
#pragma unroll
    for (int n = 0; n < NVC; ++n)
#pragma unroll
        for (int k = 0; k < N1; ++k) lf[n][k] = 0.0;
#pragma unroll
    for (int ip = 0; ip < GPX; ++ip) {
        const double* g = a.g1 + ip * N1;
        const double* dg = a.dg1 + ip * N1;
        const double dxc = X0 * dg[0] + X1 * dg[1];
        const double dyc = Y0 * dg[0] + Y1 * dg[1];
        double u[NVC];
#pragma unroll
        for (int n = 0; n < NVC; ++n) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < N1; ++k) s += uh[n][k] * g[k];
            u[n] = s;
        }
        double nx = dyc, ny = -dxc;
        const double jcb = sqrt(nx * nx + ny * ny);
        nx /= jcb; ny /= jcb;
        const double un = u[1] * nx + u[2] * ny;
        const double f0 = pbc / u[3] * un;
        const double rho = u[0] / u[3];
        const double E = pbc / (rho * gm1) + 0.5 * (u[1] * u[1] + u[2] * u[2]);
        const double fl[NVC] = {f0, f0 * u[1] + pbc * nx, f0 * u[2] + pbc * ny, rho * E * un + pbc * un};
#pragma unroll
        for (int n = 0; n < NVC; ++n) {
            const double r = fl[n] * jcb * a.w1[ip];
#pragma unroll
            for (int k = 0; k < N1; ++k) lf[n][k] += g[k] * r;
        }
    }
#pragma unroll
    for (int n = 0; n < NVC; ++n)
#pragma unroll
        for (int k = 0; k < N1; ++k) a.eout[((long)idx * N1 + k) * NVC + n] = lf[n][k];
}

// The element launch (persistent over every element in mesh order after the first eblk
// blocks, which compute the boundary-edge fluxes).  Bound: the FP64 matrix cores and the
// pointwise solves, one wave per SIMD.  105 800 elements, p = 4: 176 us full and 53 us
// inviscid, against 7 x 114 us and 7 x 35 us for colour launches with an element per 32
// lanes (a general 4 x 4 product and solve per point, 25 of 32 lanes in use).
template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_cns(CnsElemArgs a, CnsEdgeArgs e, int eblk) {
    if ((int)blockIdx.x < eblk) {
        edge_cns_body<P>(e, blockIdx.x * 256 + threadIdx.x);
        return;
    }
    elem_cns_body<P, FULL>(a, eblk);
}

// FP32 arithmetic (the inner solve of the defect correction), FP64 state and residual: one
// element per 32 lanes, one Gauss point per lane; transforms are per-lane dot products
// against operator rows in LDS (point-contiguous), derivative and integration
// contractions exchange point values through LDS.  It keeps the order of every FP32
// operation: the residual of a near-uniform stream is a small difference of FP32 fluxes, and
// another order, as accurate against FP64, moves the mixed iterates.  Measured after 12
// updates with every dot product summed backwards, relative change of the side and interior
// modes: p = 4 3e-3 at 100 x 100 and 8e-3 at 230 x 230, p = 2 9e-4 at 200 x 200 (corrections
// 1e-3), p = 1 1e-4.  (The same iteration from a start changed in its 10th digit, the order
// kept, moves by 2e-4.)
template <int P, bool FULL>
__device__ __forceinline__ void elem_cns_lane_body(const CnsElemArgs32& a, int noct, int blk, int nblk) {
    using D = CDims<P>;
    using T = float;
    constexpr int TM = D::TM, G = D::G, NO = NVC * TM;
    constexpr int SMD = D::SM > 0 ? D::SM : 1;
    __shared__ T sops[D::SIZE];
    // rows padded by one word: the lanes of a half-wave read different variables' rows at
    // one Gauss point, and the two half-waves of a wave read their own buffers, which
    // unpadded sit a multiple of the LDS bank period apart
    __shared__ T suh[8][NVC][17];
    __shared__ T sf[8][8][33];
    for (int k = threadIdx.x; k < D::SIZE; k += blockDim.x) sops[k] = a.ops[k];
    const int hw = threadIdx.x >> 5, g = threadIdx.x & 31;
    const T gm1 = T(a.ph.gamma) - T(1.0), gogm1 = T(a.ph.gamma) / gm1;
    __syncthreads();  // operators staged

    HPG_OCTET_LOOP_OF(noct, oc, blk, nblk) {
        wave_lds_sync();  // previous octet done with this half-wave's LDS buffers
        const int idx = a.begin + oc * 8 + hw;
        const bool valid = idx < a.end;
        const int t = valid ? idx : a.begin;
        int vtx[3], seg[3], sgn[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            vtx[k] = a.tri_pnt[3 * t + k];
            seg[k] = a.tri_seg[3 * t + k];
            sgn[k] = a.tri_sgn[3 * t + k];
        }
        const double x0 = a.pnts[2 * vtx[0]], y0 = a.pnts[2 * vtx[0] + 1];
        const double x1 = a.pnts[2 * vtx[1]], y1 = a.pnts[2 * vtx[1] + 1];
        const double x2 = a.pnts[2 * vtx[2]], y2 = a.pnts[2 * vtx[2] + 1];
        // ldcrd(n,0) = dx_n/dr, ldcrd(n,1) = dx_n/ds (rsdl.cpp:56-59)
        const T l00 = T(T(0.5) * (x2 - x1)), l01 = T(T(0.5) * (x0 - x1));
        const T l10 = T(T(0.5) * (y2 - y1)), l11 = T(T(0.5) * (y0 - y1));

        if (g < TM) {
            int kind;
            double sg;
            const int off = mode_offset<P, NVC>(g, t, vtx, seg, sgn, a.sm0, a.im0, kind, sg);
            const double* src = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
#pragma unroll
            for (int n = 0; n < NVC; ++n)
                suh[hw][n][g] = valid ? T(sg * src[off + n]) : ((g < 3 && (n == 0 || n == 3)) ? T(T(1.0)) : T(T(0.0)));
        }
        wave_lds_sync();

        // values (and derivatives of u, v, RT) at this lane's Gauss point
        T u[NVC], ur[NVC], us[NVC];
#pragma unroll
        for (int n = 0; n < NVC; ++n) { u[n] = T(0.0); ur[n] = T(0.0); us[n] = T(0.0); }
#pragma unroll 3
        for (int k = 0; k < TM; ++k) {
            const T pk = sops[D::OP_P + k * 32 + g];
#pragma unroll
            for (int n = 0; n < NVC; ++n) u[n] += pk * suh[hw][n][k];
            if constexpr (FULL) {
                const T prk = sops[D::OP_PR + k * 32 + g], psk = sops[D::OP_PS + k * 32 + g];
#pragma unroll
                for (int n = 1; n < NVC; ++n) { ur[n] += prk * suh[hw][n][k]; us[n] += psk * suh[hw][n][k]; }
            }
        }
        if (g >= G) { u[0] = T(1.0); u[3] = T(1.0); }  // padding lanes: keep the pointwise work finite

        // convective terms (rsdl.cpp:315-351)
        T cv[NVC][2];
        {
            const T rho = u[0] / u[3];
            const T fluxx = rho * (u[1] - T(0.0)), fluxy = rho * (u[2] - T(0.0));
            cv[0][0] = +l11 * fluxx - l01 * fluxy;
            cv[0][1] = -l10 * fluxx + l00 * fluxy;
            cv[1][0] = u[1] * cv[0][0] + l11 * u[0];
            cv[1][1] = u[1] * cv[0][1] - l10 * u[0];
            cv[2][0] = u[2] * cv[0][0] - l01 * u[0];
            cv[2][1] = u[2] * cv[0][1] + l00 * u[0];
            const T E = u[3] / gm1 + T(0.5) * (u[1] * u[1] + u[2] * u[2]);
            const T nfx = E * fluxx + u[0] * u[1], nfy = E * fluxy + u[0] * u[2];
            cv[3][0] = +l11 * nfx - l01 * nfy;
            cv[3][1] = -l10 * nfx + l00 * nfy;
        }
#pragma unroll
        for (int n = 0; n < NVC; ++n) { sf[hw][2 * n][g] = cv[n][0]; sf[hw][2 * n + 1][g] = cv[n][1]; }
        wave_lds_sync();
        // lf_im = intgrtrs of the convective fluxes; lane g owns outputs g and g + 32
        T li[2] = {T(0.0), T(0.0)};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int o = g + 32 * r;
            if (o < NO) {
                const int n = o / TM, k = o - n * TM;
                T s = T(0.0);
#pragma unroll 5
                for (int q = 0; q < G; ++q)
                    s += sops[D::OP_IR + q * 16 + k] * sf[hw][2 * n][q] + sops[D::OP_IS + q * 16 + k] * sf[hw][2 * n + 1][q];
                li[r] = s;
            }
        }
        T lr[2] = {T(0.0), T(0.0)};
        if constexpr (FULL) {
            // viscous stress and heat flux (rsdl.cpp:355-420), steady: rhorbd0 = 0
            const T cjcb = l00 * l11 - l10 * l01;
            const T mujcbi = T(a.ph.mu) / cjcb;
            const T kcjcbi = T(a.ph.kcond) / cjcb / T(a.ph.Rgas);
            const T v0000 = -mujcbi * (T(4.) / T(3.) * l11 * l11 + l01 * l01);
            const T v0011 = -mujcbi * (T(4.) / T(3.) * l10 * l10 + l00 * l00);
            const T v0001 = mujcbi * (T(4.) / T(3.) * l11 * l10 + l01 * l00);
            const T v1100 = -mujcbi * (l11 * l11 + T(4.) / T(3.) * l01 * l01);
            const T v1111 = -mujcbi * (l10 * l10 + T(4.) / T(3.) * l00 * l00);
            const T v1101 = mujcbi * (l11 * l10 + T(4.) / T(3.) * l01 * l00);
            const T v0100 = mujcbi * T(1.) / T(3.) * l01 * l11;
            const T v0111 = mujcbi * T(1.) / T(3.) * l00 * l10;
            const T v0101 = -mujcbi * (l01 * l10 - T(2.) / T(3.) * l00 * l11);
            const T v0110 = -mujcbi * (l00 * l11 - T(2.) / T(3.) * l01 * l10);
            const T k00 = -kcjcbi * (l11 * l11 + l01 * l01);
            const T k11 = -kcjcbi * (l10 * l10 + l00 * l00);
            const T k01 = kcjcbi * (l11 * l10 + l01 * l00);
            T df[NVC][2];
            df[0][0] = T(0.0); df[0][1] = T(0.0);
            df[1][0] = v0000 * ur[1] + v0100 * ur[2] + v0001 * us[1] + v0101 * us[2];
            df[1][1] = v0001 * ur[1] + v0110 * ur[2] + v0011 * us[1] + v0111 * us[2];
            df[2][0] = v0100 * ur[1] + v1100 * ur[2] + v0110 * us[1] + v1101 * us[2];
            df[2][1] = v0101 * ur[1] + v1101 * ur[2] + v0111 * us[1] + v1111 * us[2];
            df[3][0] = k00 * ur[3] + k01 * us[3];
            df[3][1] = k01 * ur[3] + k11 * us[3];
            df[3][0] += df[1][0] * u[1] + df[2][0] * u[2];
            df[3][1] += df[1][1] * u[1] + df[2][1] * u[2];
            wave_lds_sync();  // the half-wave is done reading the convective fluxes
#pragma unroll
            for (int n = 0; n < NVC; ++n) {
                sf[hw][2 * n][g] = cv[n][0] + df[n][0];
                sf[hw][2 * n + 1][g] = cv[n][1] + df[n][1];
            }
            wave_lds_sync();
            // strong residual: derivr/derivs of the total fluxes (rsdl.cpp:425-429)
            T res[NVC] = {T(0.0), T(0.0), T(0.0), T(0.0)};
#pragma unroll 5
            for (int q = 0; q < G; ++q) {
                const T dr = sops[D::OP_DR + q * 32 + g], ds = sops[D::OP_DS + q * 32 + g];
#pragma unroll
                for (int n = 0; n < NVC; ++n) res[n] += dr * sf[hw][2 * n][q] + ds * sf[hw][2 * n + 1][q];
            }
            // CALC_TAU2 (rsdl.cpp:431-452) and the stabilisation (:454-488)
            const T dx1 = T(x0 - x2), dy1 = T(y0 - y2), dx2 = T(x1 - x0), dy2 = T(y1 - y0);
            const T ar2 = dx1 * dy2 - dy1 * dx2;
            const T perim = sqrt(dx1 * dx1 + dy1 * dy1) + sqrt(dx2 * dx2 + dy2 * dy2) +
                                 sqrt((dx1 + dx2) * (dx1 + dx2) + (dy1 + dy2) * (dy1 + dy2));
            const T hmax = T(0.25) * ar2 / ((ar2 / perim) * (T(0.25) * (P + 1) * (P + 1)));
            {
                const T pr = u[0], uv = u[1], vv = u[2], rt = u[3];
                T Pi[4][4], tau[4][4];
                cns_tau<T>(a.ph, pr, uv, vv, rt, hmax, Pi, tau, nullptr);
                const T tf = T(a.ph.adis) / cjcb;
                T tres[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    T s = T(0.0);
#pragma unroll
                    for (int n = 0; n < 4; ++n) s += (tau[m][n] * tf) * res[n];
                    tres[m] = s;
                }
                const T rho = pr / rt, ke = T(0.5) * (uv * uv + vv * vv);
                const T A[4][4] = {
                    {uv / rt, rho, T(0.0), -rho * uv / rt},
                    {uv * uv / rt + T(1.0), T(2.0) * rho * uv, T(0.0), -rho * uv * uv / rt},
                    {uv * vv / rt, rho * vv, rho * uv, -rho * uv * vv / rt},
                    {uv * (gogm1 * rt + ke) / rt, rho * (gogm1 * rt + ke) + rho * uv * uv, rho * uv * vv,
                     -rho * uv * (gogm1 * rt + ke) / rt + rho * uv * gogm1}};
                const T B[4][4] = {
                    {vv / rt, T(0.0), rho, -rho * vv / rt},
                    {uv * vv / rt, rho * vv, rho * uv, -rho * uv * vv / rt},
                    {vv * vv / rt + T(1.0), T(0.0), T(2.0) * rho * vv, -rho * vv * vv / rt},
                    {vv * (gogm1 * rt + ke) / rt, rho * uv * vv, rho * (gogm1 * rt + ke) + rho * vv * vv,
                     -rho * vv * (gogm1 * rt + ke) / rt + rho * vv * gogm1}};
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        df[m][0] -= (+l11 * A[m][n] - l01 * B[m][n]) * tres[n];
                        df[m][1] -= (-l10 * A[m][n] + l00 * B[m][n]) * tres[n];
                    }
            }
            wave_lds_sync();  // the half-wave is done reading the total fluxes
#pragma unroll
            for (int n = 0; n < NVC; ++n) { sf[hw][2 * n][g] = df[n][0]; sf[hw][2 * n + 1][g] = df[n][1]; }
            wave_lds_sync();
            // lf_re = beta * intgrtrs(viscous - stabilisation fluxes) (rsdl.cpp:490-497)
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int o = g + 32 * r;
                if (o < NO) {
                    const int n = o / TM, k = o - n * TM;
                    T s = T(0.0);
#pragma unroll
                    for (int q = 0; q < G; ++q)
                        s += sops[D::OP_IR + q * 16 + k] * sf[hw][2 * n][q] + sops[D::OP_IS + q * 16 + k] * sf[hw][2 * n + 1][q];
                    lr[r] = s * T(a.beta);
                }
            }
        }

        // element-major: the sum lf_im + beta lf_re and beta lf_re, in FP64.  The element
        // whose colour touches a coefficient first adds the two parts one by one, the
        // others their FP32 sum, the roundings of a scatter colour by colour (one form for all
        // moves the iterates by 1e-3 at p = 4, 230 x 230, 2e-4 at p <= 2)
        if (valid) {
            const int col = a.tcol[t];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int o = g + 32 * r;
                if (o >= NO) continue;
                const int n = o / TM, k = o - n * TM;
                int kind;
                double sg;
                const int off = mode_offset<P, NVC>(k, t, vtx, seg, sgn, a.sm0, a.im0, kind, sg) + n;
                const T vli = T(sg) * li[r], vlr = T(sg) * lr[r];
                if (kind < 2) {
                    const bool first = (kind == 0 ? a.fcv[sel3(vtx, k)] : a.fcs[sel3(seg, (k - 3) / SMD)]) == col;
                    double* d = a.eres + ((size_t)t * D::BM + k) * (FULL ? 2 * NVC : NVC) + n;
                    d[0] = first ? (double)vlr + (double)vli : (double)(vlr + vli);
                    if constexpr (FULL) d[NVC] = vlr;
                } else {
                    const double r0 = a.keep == 0.0 ? 0.0 : a.keep * a.rri[off];
                    if (FULL || a.keep != 1.0) a.rri[off] = r0 + vlr;
                    a.resi[off] = r0 + vlr + vli + (a.srci ? a.srci[off] * a.sfac[0] : 0.0);
                }
            }
        }
    }
}

template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_cns32(CnsElemArgs32 a, CnsEdgeArgs e, int eblk) {
    if ((int)blockIdx.x < eblk) {
        edge_cns_body<P>(e, blockIdx.x * 256 + threadIdx.x);
        return;
    }
    elem_cns_lane_body<P, FULL>(a, (a.end - a.begin + 7) / 8, (int)blockIdx.x - eblk, (int)gridDim.x - eblk);
}

// Element Jacobians of a batch, as k_elem_ins_jac
template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_cns_jac(CnsElemArgs a) {
    elem_cns_body<P, FULL, true>(a);
}

// ---------------------------------------------------------------------------------
// setup_preconditioner (tri_hp/cns/setup_preconditioner.cpp:7-239, diagonal branch,
// straight elements): per element the low-Mach preconditioner inverse scaled by the
// inverse pseudo-time step, tprcn = jcb; then per-vertex / per-side sums
struct CnsSetupArgs {
    const double* pnts;
    const int* tri_pnt;
    const int* tri_seg;
    const int* tri_sgn;
    const double* ugv;
    const double* ugs;
    const double* ugi;
    const double* Pmat;  // G x tm
    double* tprcn;       // ntri x 4
    double* tpc;         // ntri x 16
    int* err;
    int ntri, sm0, im0;
    CnsPhys ph;
};

template <int P>
__global__ __launch_bounds__(128) void k_setup_elem_cns(CnsSetupArgs a) {
    constexpr int TM = Dims<P>::TM, SM = Dims<P>::SM, G = Dims<P>::G;
    const int t = xcd_block() * blockDim.x + threadIdx.x;
    if (t >= a.ntri) return;
    int vtx[3], seg[3], sgn[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        vtx[k] = a.tri_pnt[3 * t + k];
        seg[k] = a.tri_seg[3 * t + k];
        sgn[k] = a.tri_sgn[3 * t + k];
    }
    double uh[NVC][TM];
#pragma unroll
    for (int k = 0; k < TM; ++k) {
        int kind;
        double sg;
        const int off = mode_offset<P, NVC>(k, t, vtx, seg, sgn, a.sm0, a.im0, kind, sg);
        const double* src = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
#pragma unroll
        for (int n = 0; n < NVC; ++n) uh[n][k] = sg * src[off + n];
    }
    double qmax = 0.0, umax[NVC] = {0.0, 0.0, 0.0, 0.0};
    for (int g = 0; g < G; ++g) {
        double w[NVC] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < TM; ++k) {
            const double pv = a.Pmat[g * TM + k];
#pragma unroll
            for (int n = 0; n < NVC; ++n) w[n] += pv * uh[n][k];
        }
        const double q = w[1] * w[1] + w[2] * w[2];
        qmax = (qmax > q) ? qmax : q;  // MAX of sys/param.h
#pragma unroll
        for (int n = 0; n < NVC; ++n) {
            const double f = fabs(w[n]);
            umax[n] = (umax[n] > f) ? umax[n] : f;
        }
    }
    const double X[3] = {a.pnts[2 * vtx[0]], a.pnts[2 * vtx[1]], a.pnts[2 * vtx[2]]};
    const double Y[3] = {a.pnts[2 * vtx[0] + 1], a.pnts[2 * vtx[1] + 1], a.pnts[2 * vtx[2] + 1]};
    const double dx1 = X[0] - X[2], dy1 = Y[0] - Y[2], dx2 = X[1] - X[0], dy2 = Y[1] - Y[0];
    const double jcb = 0.25 * (dx1 * dy2 - dy1 * dx2);
    double hmax = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int j1 = (j + 1) % 3;
        const double hh = (X[j] - X[j1]) * (X[j] - X[j1]) + (Y[j] - Y[j1]) * (Y[j] - Y[j1]);
        hmax = hh > hmax ? hh : hmax;
    }
    hmax = sqrt(hmax);
    const double pf = 0.25 * (P + 1) * (P + 1);
    const double h = 4. * jcb / (pf * hmax);
    hmax = hmax / pf;
    if (!(h > 0.0) || qmax != qmax) {
        atomicOr(a.err, 1);
#pragma unroll
        for (int n = 0; n < NVC; ++n) a.tprcn[NVC * t + n] = 1.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) a.tpc[16 * t + k] = (k % 5 == 0) ? 1.0 : 0.0;
        return;
    }
    double Pinv[4][4], tau[4][4], tstep;
    cns_tau(a.ph, umax[0], umax[1], umax[2], umax[3], hmax, Pinv, tau, &tstep);
    const double dtstari = 1.0 / tstep;
#pragma unroll
    for (int n = 0; n < NVC; ++n) a.tprcn[NVC * t + n] = jcb;
#pragma unroll
    for (int k = 0; k < 16; ++k) a.tpc[16 * t + k] = Pinv[k / 4][k % 4] * dtstari;
}

// vprcn = 1/(vdiag sum jcb), vpc = sum tpc*jcb over the incident elements (ascending)
__global__ __launch_bounds__(256) void k_setup_vrtx_cns(int npnt, const int* ptr, const int* tri, const double* tprcn, const double* tpc,
                                 double* vprcn, double* vpc, double vdiag) {
    const int v = xcd_block() * blockDim.x + threadIdx.x;
    if (v >= npnt) return;
    double s[NVC] = {0.0, 0.0, 0.0, 0.0}, m[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) m[k] = 0.0;
    for (int j = ptr[v]; j < ptr[v + 1]; ++j) {
        const int t = tri[j];
        const double jcb = tprcn[NVC * t];
#pragma unroll
        for (int n = 0; n < NVC; ++n) s[n] += tprcn[NVC * t + n];
#pragma unroll
        for (int k = 0; k < 16; ++k) m[k] += tpc[16 * t + k] * jcb;
    }
#pragma unroll
    for (int n = 0; n < NVC; ++n) vprcn[NVC * v + n] = 1.0 / (vdiag * s[n]);
#pragma unroll
    for (int k = 0; k < 16; ++k) vpc[16 * v + k] = m[k];
}

// sprcn = 1/sum jcb, spc = sum tpc over the (one or two) elements of each side
__global__ __launch_bounds__(256) void k_setup_side_cns(int nseg, const int* st_tri, const double* tprcn, const double* tpc, double* sprcn,
                                 double* spc) {
    const int s = xcd_block() * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    double a[NVC] = {0.0, 0.0, 0.0, 0.0}, m[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) m[k] = 0.0;
    for (int j = 0; j < 2; ++j) {
        const int t = st_tri[2 * s + j];
        if (t < 0) continue;
#pragma unroll
        for (int n = 0; n < NVC; ++n) a[n] += tprcn[NVC * t + n];
#pragma unroll
        for (int k = 0; k < 16; ++k) m[k] += tpc[16 * t + k];
    }
#pragma unroll
    for (int n = 0; n < NVC; ++n) sprcn[NVC * s + n] = 1.0 / a[n];
#pragma unroll
    for (int k = 0; k < 16; ++k) spc[16 * s + k] = m[k];
}

// ---------------------------------------------------------------------------------
// inflow boundaries: the conservative momentum and energy residuals follow from the
// mass residual and the prescribed u, v, RT (tri_hp/cns/bdry.cpp:247-340)
struct CnsBcArgs {
    double* resv;
    double* ress;
    const int* verts;  // inflow boundary vertices (each once)
    const int* sides;  // inflow boundary sides
    int nverts, nsides;
    const int* seg_pnt;
    const double* g1;
    const double* w1;
    const double* sdiag1d;  // upper band factor, kd = 2
    int sm0;
    double bu, bv, benergy;  // u, v, RT/(gamma-1) + |u|^2/2 of the boundary state
};

__global__ void k_mbr_vrtx(CnsBcArgs a) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nverts) return;
    const int v = a.verts[k];
    const double r0 = a.resv[v * NVC];
    a.resv[v * NVC + 1] = r0 * a.bu;
    a.resv[v * NVC + 2] = r0 * a.bv;
    a.resv[v * NVC + 3] = r0 * a.benergy;
}

// banded U^T U x = b, U upper band with bandwidth 2 stored per column (3 per row)
template <int N>
__device__ __forceinline__ void band2_solve(const double* ab, double b[N]) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
        double s = b[j];
#pragma unroll
        for (int k = (j - 2 > 0 ? j - 2 : 0); k < j; ++k) s -= ab[j * 3 + 2 + k - j] * b[k];
        b[j] = s / ab[j * 3 + 2];
    }
#pragma unroll
    for (int j = N - 1; j >= 0; --j) {
        const double s = b[j] / ab[j * 3 + 2];
        b[j] = s;
#pragma unroll
        for (int k = (j - 2 > 0 ? j - 2 : 0); k < j; ++k) b[k] -= ab[j * 3 + 2 + k - j] * s;
    }
}

template <int P>
__global__ __launch_bounds__(256) void k_mbr_side(CnsBcArgs a) {
    constexpr int SM = Dims<P>::SM, N1 = SM + 2, GPX = P + 1;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nsides) return;
    const int s = a.sides[k];
    const int v0 = a.seg_pnt[2 * s], v1 = a.seg_pnt[2 * s + 1];
    double rc[N1];
    rc[0] = a.resv[v0 * NVC];
    rc[1] = a.resv[v1 * NVC];
#pragma unroll
    for (int m = 0; m < SM; ++m) rc[m + 2] = a.ress[(s * a.sm0 + m) * NVC];
    const double bval[NVC] = {0.0, a.bu, a.bv, a.benergy};
#pragma unroll
    for (int n = 1; n < NVC; ++n) {
        double lf[N1];
#pragma unroll
        for (int m = 0; m < N1; ++m) lf[m] = 0.0;
        const double e0 = a.resv[v0 * NVC + n], e1 = a.resv[v1 * NVC + n];
#pragma unroll
        for (int i = 0; i < GPX; ++i) {
            const double* g = a.g1 + i * N1;
            double r1 = 0.0;
#pragma unroll
            for (int m = 0; m < N1; ++m) r1 += rc[m] * g[m];
            const double f = (e0 * g[0] + e1 * g[1]) - r1 * bval[n];
#pragma unroll
            for (int m = 0; m < N1; ++m) lf[m] += g[m] * a.w1[i] * f;
        }
        double x[SM];
#pragma unroll
        for (int m = 0; m < SM; ++m) x[m] = lf[m + 2];
        band2_solve<SM>(a.sdiag1d, x);
#pragma unroll
        for (int m = 0; m < SM; ++m) a.ress[(s * a.sm0 + m) * NVC + n] = -x[m];
    }
}

// ---------------------------------------------------------------------------------
// project_new_variables (tri_hp/cns/update.cpp:5-245): the conservative correction
// becomes a primitive one, r <- L^-1 dpdc(u) r with L the lower triangle of the
// vertex block preconditioner (interpolated linearly along sides and over elements),
// projected back onto the side and interior modes.
struct CnsProjArgs {
    const double* ugv;
    const double* ugs;
    double* ugi;          // interiors: the stage update ug = ug0 - cfa * correction included
    const double* ug0i;
    double cfa;
    double* resv;
    double* ress;
    double* resi;
    double* rtv;  // copies of the conservative correction (res_temp)
    double* rts;
    const double* vpc;
    const unsigned char* vess;
    const unsigned char* sess;
    const int* seg_pnt;
    const int* tri_pnt;
    const int* tri_seg;
    const int* tri_sgn;
    const double* g1;
    const double* w1;
    const double* sdiag1d;
    const double* ops;    // PDims<P> pack
    int npnt, nseg, ntri, sm0, im0;
    double gamma;
};

__global__ __launch_bounds__(256) void k_pnv_vrtx(CnsProjArgs a) {
    const int v = xcd_block() * blockDim.x + threadIdx.x;
    if (v >= a.npnt) return;
    double w[NVC], r[NVC];
#pragma unroll
    for (int n = 0; n < NVC; ++n) {
        w[n] = a.ugv[v * NVC + n];
        r[n] = a.resv[v * NVC + n];
        a.rtv[v * NVC + n] = r[n];
    }
    switch_vars(w, r, a.gamma - 1.0);
    double L[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) L[k] = a.vpc[16 * v + k];
    lower4(L, r);
    const unsigned msk = a.vess[v];
#pragma unroll
    for (int n = 0; n < NVC; ++n) a.resv[v * NVC + n] = ((msk >> n) & 1) ? 0.0 : r[n];
}

template <int P>
__global__ __launch_bounds__(256) void k_pnv_side(CnsProjArgs a) {
    constexpr int SM = Dims<P>::SM, N1 = SM + 2, GPX = P + 1;
    const int s = xcd_block() * blockDim.x + threadIdx.x;
    if (s >= a.nseg) return;
    const int p0 = a.seg_pnt[2 * s], p1 = a.seg_pnt[2 * s + 1];
    const double gm1 = a.gamma - 1.0;
    double uc[NVC][N1], rc[NVC][N1], tv0[NVC], tv1[NVC];
#pragma unroll
    for (int n = 0; n < NVC; ++n) {
        uc[n][0] = a.ugv[p0 * NVC + n]; uc[n][1] = a.ugv[p1 * NVC + n];
        rc[n][0] = a.rtv[p0 * NVC + n]; rc[n][1] = a.rtv[p1 * NVC + n];
        tv0[n] = a.resv[p0 * NVC + n]; tv1[n] = a.resv[p1 * NVC + n];
#pragma unroll
        for (int m = 0; m < SM; ++m) {
            uc[n][m + 2] = a.ugs[(s * a.sm0 + m) * NVC + n];
            rc[n][m + 2] = a.ress[(s * a.sm0 + m) * NVC + n];
        }
    }
    double lf[NVC][N1];
#pragma unroll
    for (int n = 0; n < NVC; ++n)
#pragma unroll
        for (int m = 0; m < N1; ++m) lf[n][m] = 0.0;
#pragma unroll
    for (int i = 0; i < GPX; ++i) {
        const double* g = a.g1 + i * N1;
        double w[NVC], r[NVC], L[16];
#pragma unroll
        for (int n = 0; n < NVC; ++n) {
            double su = 0.0, sr = 0.0;
#pragma unroll
            for (int m = 0; m < N1; ++m) { su += uc[n][m] * g[m]; sr += rc[n][m] * g[m]; }
            w[n] = su; r[n] = sr;
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) L[k] = a.vpc[16 * p0 + k] * g[0] + a.vpc[16 * p1 + k] * g[1];
        switch_vars(w, r, gm1);
        lower4(L, r);
#pragma unroll
        for (int n = 0; n < NVC; ++n) {
            const double f = (tv0[n] * g[0] + tv1[n] * g[1]) - r[n];
#pragma unroll
            for (int m = 0; m < N1; ++m) lf[n][m] += g[m] * a.w1[i] * f;
        }
    }
    const unsigned msk = a.sess[s];
#pragma unroll
    for (int n = 0; n < NVC; ++n) {
        double x[SM];
#pragma unroll
        for (int m = 0; m < SM; ++m) x[m] = lf[n][m + 2];
        band2_solve<SM>(a.sdiag1d, x);
#pragma unroll
        for (int m = 0; m < SM; ++m) {
            const int ix = (s * a.sm0 + m) * NVC + n;
            a.rts[ix] = rc[n][m + 2];
            a.ress[ix] = ((msk >> n) & 1) ? 0.0 : -x[m];
        }
    }
}

// operators of the interior projection: P as lane-ready K-steps, then per Gauss point the
// three vertex functions and the three interior rows of S I (S the interior band solve, I
// the integration), then per mode the interior rows of S I P
template <int P>
struct PDims {
    static constexpr int PROJ = Dims<P>::PROJ, OP_V = PROJ, OP_I = OP_V + 32 * 3, OP_IP = OP_I + 32 * 3;
    static constexpr int SIZE = OP_IP + 16 * 3;
};

// interiors (IM = 3, p = 4): r <- S I (tt - L^-1 dpdc(u) r) with tt the primitive correction
// of the element's vertices and sides.  16 elements per wave: u and r are projected on the
// FP64 matrix cores, the lower-triangular solve runs in the lane that holds the point, and
// the integration, with the band solve and the projection of tt folded into its operators,
// is 33 products per lane and variable, summed over the four lanes of an element.
// Stage update of the interior state included (only this element reads it).  105 800
// elements: 77 us, against 154 us with an element per half-wave and its transforms
// through LDS.
template <int P>
__global__ __launch_bounds__(256, 2) void k_pnv_int(CnsProjArgs a) {
    using D = Dims<P>;
    using Q = PDims<P>;
    constexpr int GT = D::GT, KT = D::KT, IM = D::IM;
    static_assert(IM == 3, "interior modes of an element: one per lane group");
    __shared__ double so[Q::SIZE];
    for (int k = threadIdx.x; k < Q::SIZE; k += blockDim.x) so[k] = a.ops[k];
    __syncthreads();
    const int lane = threadIdx.x & 63, e = lane & 15, q = lane >> 4;
    const int WX = ((int)gridDim.x >> 3) * 4, rank = ((int)blockIdx.x >> 3) * 4 + (threadIdx.x >> 6);
    const int xcd = blockIdx.x & 7, ng = (a.ntri + 15) >> 4, gpx = (ng + 7) >> 3;
    const int g0 = xcd * gpx + rank, gend = min(ng, (xcd + 1) * gpx);
    if (g0 >= gend) return;
    const double gm1 = a.gamma - 1.0;
    auto elem = [&](int g) { const int t = g * 16 + e; return g < gend && t < a.ntri ? t : -1; };
    ElemConn cn = elem_conn(a, elem(g0));
    for (int g = g0; g < gend; g += WX) {
        const ElemConn c = cn;
        cn = elem_conn(a, elem(g + WX));
        const bool valid = c.t >= 0;
        double u[NVC][KT], r[NVC][KT], x[IM][NVC];
#pragma unroll
        for (int m = 0; m < IM; ++m)
#pragma unroll
            for (int n = 0; n < NVC; ++n) x[m][n] = 0.0;
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = 4 * s + q;
            const bool live = valid && k < D::TM;
            int kind;
            double sg;
            const int off = mode_offset<P, NVC>(k, valid ? c.t : 0, c.vtx, c.seg, c.sgn, a.sm0, a.im0, kind, sg);
            const double* pu = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
            const double* pr = kind == 0 ? a.rtv : (kind == 1 ? a.rts : a.resi);
            const double* pt = kind == 0 ? a.resv : a.ress;
            double ip[IM];
#pragma unroll
            for (int m = 0; m < IM; ++m) ip[m] = so[Q::OP_IP + k * 3 + m];
#pragma unroll
            for (int n = 0; n < NVC; ++n) {
                u[n][s] = live ? sg * pu[off + n] : 0.0;
                r[n][s] = live ? sg * pr[off + n] : 0.0;
                const double t = live && kind < 2 ? sg * pt[off + n] : 0.0;
#pragma unroll
                for (int m = 0; m < IM; ++m) x[m][n] += ip[m] * t;
            }
        }
        // lower triangles of the vertices' 4 x 4 blocks
        double L[3][10];
#pragma unroll
        for (int v = 0; v < 3; ++v)
#pragma unroll
            for (int i = 0, o = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j <= i; ++j, ++o) L[v][o] = valid ? a.vpc[(long)16 * c.vtx[v] + 4 * i + j] : (i == j ? 1.0 : 0.0);
#pragma unroll
        for (int kt = 0; kt < GT; ++kt) {
            const d4 z = {0.0, 0.0, 0.0, 0.0};
            d4 cu[NVC] = {z, z, z, z}, cr[NVC] = {z, z, z, z};
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const double av = so[(kt * KT + s) * 64 + lane];
#pragma unroll
                for (int n = 0; n < NVC; ++n) {
                    cu[n] = mfma(av, u[n][s], cu[n]);
                    cr[n] = mfma(av, r[n][s], cr[n]);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (16 * kt + 4 * i >= D::G) continue;
                __builtin_amdgcn_sched_barrier(0);  // one point at a time (registers)
                const int pt = 16 * kt + 4 * i + q;
                const bool in = valid && pt < D::G;
                const double b0 = so[Q::OP_V + pt * 3], b1 = so[Q::OP_V + pt * 3 + 1], b2 = so[Q::OP_V + pt * 3 + 2];
                double w[NVC], f[NVC], M[16];
#pragma unroll
                for (int n = 0; n < NVC; ++n) { w[n] = in ? cu[n][i] : 1.0; f[n] = cr[n][i]; }
#pragma unroll
                for (int ii = 0, o = 0; ii < 4; ++ii)
#pragma unroll
                    for (int j = 0; j <= ii; ++j, ++o)
                        M[4 * ii + j] = in ? L[0][o] * b0 + L[1][o] * b1 + L[2][o] * b2 : (ii == j ? 1.0 : 0.0);
                switch_vars(w, f, gm1);
                lower4(M, f);
#pragma unroll
                for (int m = 0; m < IM; ++m) {
                    const double wi = so[Q::OP_I + pt * 3 + m];
#pragma unroll
                    for (int n = 0; n < NVC; ++n) x[m][n] -= wi * (in ? f[n] : 0.0);
                }
            }
        }
        // sum over the element's four lanes; lane group m stores interior mode m
#pragma unroll
        for (int m = 0; m < IM; ++m)
#pragma unroll
            for (int n = 0; n < NVC; ++n) {
                x[m][n] += __shfl_xor(x[m][n], 16, 64);
                x[m][n] += __shfl_xor(x[m][n], 32, 64);
            }
        if (valid && q < IM) {
            const long o = ((long)c.t * a.im0 + q) * NVC;
#pragma unroll
            for (int n = 0; n < NVC; ++n) {
                const double d = -(q == 0 ? x[0][n] : (q == 1 ? x[1][n] : x[2][n]));
                a.resi[o + n] = d;
                a.ugi[o + n] = a.ug0i[o + n] - a.cfa * d;
            }
        }
    }
}

}  // namespace hpg
