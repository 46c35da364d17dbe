// HIP kernels of the tri_hp / tri_hp_ins residual and relaxation path (gfx950).
//
// Element residual: 16 elements per wave64, every basis transform a dense
// contraction on v_mfma_f64_16x16x4f64.  Rows of an MFMA tile are Gauss points
// (or modes), columns are the 16 elements of the wave.  Operands: A (16x4) lane l
// holds A[l%16][l/16], B (4x16) lane l holds B[l/16][l%16]; the f64 accumulator
// register i of lane l holds D[4*i + l/16][l%16] (checked on the device by
// hpg_selftest_mfma).  Accumulators are fed straight back as the B operand of the
// next contraction: the operator matrices are stored with their K index permuted
// so that K-step (tile t, register i) reads row 16t + 4*i + l/16, which is exactly
// what lane l holds.  No data moves between lanes from the modal gather to the
// modal scatter.
#include <hip/hip_runtime.h>
#include "tri_kernels.h"

namespace hpg {

typedef double d4 __attribute__((ext_vector_type(4)));

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// v_mfma_f32_16x16x4f32: accumulator register i of lane l holds D[4*(l/16) + i][l%16]
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// v_mfma_f64_4x4x4f64: four 4 x 4 blocks; lane l holds A[l % 4][l / 16] (the same for the
// four blocks here), B[l / 16][l % 16] and the result D[l / 16][l % 16].  16 cycles against 64
// of the 16x16x4 form: the same rate per product without its 16-row tiles.  FP64 vector and
// matrix instructions share one unit at one rate (measured: neither overlaps the other), so
// what an FP64 kernel pays for is its number of products, padding included.
__device__ __forceinline__ double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
// keeps the compiler from moving operand loads (all loop invariants) and flux sums across the
// phases of an element group: hoisted, they spill
__device__ __forceinline__ void group_phase() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// the same for values: what is computed from x after this is computed anew (fluxes kept from
// the pass before would not fit the registers)
template <int N>
__device__ __forceinline__ void group_opaque(double (&x)[N]) {
    group_phase();
#pragma unroll
    for (int k = 0; k < N; ++k) asm volatile("" : "+v"(x[k]));
}
template <typename T> struct Vec4;
template <> struct Vec4<double> { typedef d4 type; };
template <> struct Vec4<float> { typedef f4 type; };

// ---------------------------------------------------------------------------------
// tri_hp::ugtouht / lftog index map for mode k of element t (tri_hp/gtol.cpp:14-55,
// 364-402): returns the offset of the NV-vector and the side sign sgn^m.
// a[i] for a lane-varying i < 3 without dynamic register indexing (which would spill
// the array to scratch)
__device__ __forceinline__ int sel3(const int* a, int i) { return i == 0 ? a[0] : (i == 1 ? a[1] : a[2]); }

template <int P, int NVn = NV>
__device__ __forceinline__ int mode_offset(int k, int t, const int* vtx, const int* seg, const int* sgn,
                                           int sm0, int im0, int& kind, double& sign) {
    using D = Dims<P>;
    sign = 1.0;
    if (k < 3) { kind = 0; return sel3(vtx, k) * NVn; }
    if (k < D::BM) {
        constexpr int SMD = D::SM > 0 ? D::SM : 1;
        const int i = (k - 3) / SMD, m = (k - 3) - i * SMD;
        kind = 1;
        sign = ((m & 1) && sel3(sgn, i) < 0) ? -1.0 : 1.0;
        return (sel3(seg, i) * sm0 + m) * NVn;
    }
    kind = 2;
    return (t * im0 + (k - D::BM)) * NVn;
}

// Per-lane gather state of one element, loaded one group ahead of its use.
// Slot s of lane l is mode 4s + l/16 of element l%16: the K-step of the projection
// that reads it and the accumulator register that returns its residual.
struct ElemConn {
    int t;  // element, -1 for a padding lane
    int vtx[3], seg[3], sgn[3];
};

template <int P>
struct ElemSlots {
    static constexpr int KT = Dims<P>::KT;
    int t;
    int off[KT];   // offset of the slot's NV-vector, bitwise-negated for a side sign of -1
    int first;     // bit s: the slot's first visit in this stage
    double x[3], y[3];
};

// kind of mode k: 0 vertex, 1 side, 2 interior (mode_offset's classification)
template <int P>
__device__ __forceinline__ int mode_kind(int k) { return k < 3 ? 0 : (k < Dims<P>::BM ? 1 : 2); }

// element of lane e in 16-element group g; a null order walks the elements in their
// own (mesh) order, which keeps neighbouring elements in one group
template <bool JAC = false, class A>
__device__ __forceinline__ int elem_of_group(const A& a, int g, int gend, int e) {
    const int idx = a.begin + g * 16 + e;
    if (!(g < gend && idx < a.end)) return -1;
    if constexpr (JAC) return a.order[idx / a.jcols];
    return a.order ? a.order[idx] : idx;
}

template <class A>
__device__ __forceinline__ ElemConn elem_conn(const A& a, int t) {
    ElemConn c;
    c.t = t;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        c.vtx[k] = t >= 0 ? a.tri_pnt[3 * t + k] : 0;
        c.seg[k] = t >= 0 ? a.tri_seg[3 * t + k] : 0;
        c.sgn[k] = t >= 0 ? a.tri_sgn[3 * t + k] : 1;
    }
    return c;
}

template <int P, int NVn = NV, class A>
__device__ __forceinline__ ElemSlots<P> elem_slots(const A& a, const ElemConn& c, int q) {
    using D = Dims<P>;
    constexpr int SMD = D::SM > 0 ? D::SM : 1;
    ElemSlots<P> S;
    S.t = c.t;
    const bool valid = c.t >= 0;
    // padding lanes compute on the reference triangle with a zero state
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        S.x[k] = valid ? a.pnts[2 * c.vtx[k]] : (k == 1 ? 1.0 : 0.0);
        S.y[k] = valid ? a.pnts[2 * c.vtx[k] + 1] : (k == 2 ? 1.0 : 0.0);
    }
#pragma unroll
    for (int s = 0; s < D::KT; ++s) {
        const int k = 4 * s + q;
        int kind;
        double sg;
        const int off = mode_offset<P, NVn>(k, valid ? c.t : 0, c.vtx, c.seg, c.sgn, a.sm0, a.im0, kind, sg);
        S.off[s] = sg < 0.0 ? ~off : off;
        const bool live = valid && k < D::TM;
        const bool first = live && (kind == 2 || (kind == 0 ? a.fcv[sel3(c.vtx, k)]
                                                             : a.fcs[sel3(c.seg, (k - 3) / SMD)]) == a.colour);
        if (s == 0) S.first = 0;
        S.first |= first ? (1 << s) : 0;
    }
    return S;
}

// tri_hp_ins::element_rsdl, straight branch (tri_hp/ins/rsdl.cpp:259-433), steady,
// for the elements order[begin:end) (one colour: no two share a vertex or side).
// Persistent: each wave walks 16-element groups of its XCD's contiguous share of the
// colour and keeps a three-deep load pipeline (element ids three groups ahead,
// connectivity two ahead, modes/geometry/first-visit flags one ahead; the old
// residual values of the current group are requested before its contractions), so
// the dependent gathers overlap the MFMA work of earlier groups.  The grid is a
// multiple of 8 blocks of 4 waves.
// CURV: the curved branch (tri_hp/ins/rsdl.cpp:83-257) for the elements order[begin:end)
// that own a curved boundary side: the coordinate derivatives dcrd are projected to
// every Gauss point from the element's coordinate modes (tri_hp/metric.cpp:12-21:
// crdtocht + proj_bdry), so the metric terms, the Jacobian and tau vary per point.
// JAC: the forward-difference element Jacobian (tri_hp/nstage.cpp:131-165): entry idx is
// the element order[idx / jcols] with its own copy of column idx % jcols's coefficient
// moved by dw, so the columns of all elements are independent entries of one launch.
template <typename T, int P, bool FULL, bool EM = false, bool CURV = false, bool JAC = false>
__device__ __forceinline__ void elem_ins_body(const ElemArgsT<T>& a, T* __restrict__ eres = nullptr, int eblk = 0) {
    using D = Dims<P>;
    using V4 = typename Vec4<T>::type;
    constexpr int GT = D::GT, KT = D::KT;
    __shared__ T sops[D::PACK];
    for (int k = threadIdx.x; k < D::PACK; k += blockDim.x) sops[k] = a.ops[k];
    __syncthreads();

    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = lane & 15, q = lane >> 4;
    // XCD-aware split: hardware deals consecutive blocks round-robin to the 8 XCDs;
    // XCD x owns groups [x*gpx, (x+1)*gpx) so neighbouring elements share its L2
    // eblk: leading blocks of the launch that do other work (a multiple of 8)
    const int WX = (((int)gridDim.x - eblk) >> 3) * 4;
    const int rank = (((int)blockIdx.x - eblk) >> 3) * 4 + w;
    const int xcd = blockIdx.x & 7;
    const int ng = (a.end - a.begin + 15) >> 4;
    const int gpx = (ng + 7) >> 3;
    const int g0 = xcd * gpx + rank;
    const int gend = min(ng, (xcd + 1) * gpx);
    if (g0 >= gend) return;

    ElemSlots<P> S = elem_slots<P>(a, elem_conn(a, elem_of_group<JAC>(a, g0, gend, e)), q);
    ElemConn cnext = elem_conn(a, elem_of_group<JAC>(a, g0 + WX, gend, e));
    int tnext2 = elem_of_group<JAC>(a, g0 + 2 * WX, gend, e);

    for (int g = g0; g < gend; g += WX) {
        // old residual values of this group, consumed by the scatter at the end and
        // requested late (register pressure): before the last contraction of the full
        // residual, after the contractions of the inviscid one
        T ro[NV][KT], io[NV][KT];
        auto load_old = [&]() {
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int k = 4 * s + q, kind = mode_kind<P>(k);
                const bool live = S.t >= 0 && k < D::TM;
                const int off = S.off[s] < 0 ? ~S.off[s] : S.off[s];
                const T* di = kind == 0 ? a.resv : (kind == 1 ? a.ress : a.resi);
                const T* dr = kind == 0 ? a.rrv : (kind == 1 ? a.rrs : a.rri);
                // element-major output (EM) reads back only the interior modes, which
                // this element owns; the gathers read the carried parts of the others
                const bool own = !EM || kind == 2;
#pragma unroll
                for (int n = 0; n < NV; ++n) {
                    ro[n][s] = (live && own && (FULL || a.keep != T(0))) ? dr[off + n] : T(0);
                    io[n][s] = (live && !EM && !((S.first >> s) & 1)) ? di[off + n] : T(0);
                }
            }
        };
        // prefetch: next group's slots, connectivity two ahead, element ids three ahead
        const ElemSlots<P> Sn = elem_slots<P>(a, cnext, q);
        const ElemConn cn2 = elem_conn(a, tnext2);
        const int tn3 = elem_of_group<JAC>(a, g + 3 * WX, gend, e);

        // modal coefficients of this group: K-step s of lane l is mode 4s + l/16
        T b[NV][KT];
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = 4 * s + q, kind = mode_kind<P>(k);
            const bool live = S.t >= 0 && k < D::TM;
            const int off = S.off[s] < 0 ? ~S.off[s] : S.off[s];
            const T sg = S.off[s] < 0 ? T(-1) : T(1);
            const T* src = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
#pragma unroll
            for (int n = 0; n < NV; ++n) b[n][s] = live ? sg * src[off + n] : T(0);
        }
        // Jacobian column of this entry: dw(var) = eps_r * sum of |uht(var)| over the vertex
        // modes (lane groups 0..2 of K-step 0) + eps_a, added to uht(var)(mode)
        int jcol = 0, jel = 0;
        T jdw = T(1);
        if constexpr (JAC) {
            const int idx = a.begin + g * 16 + e;
            jel = idx / a.jcols;
            jcol = idx - jel * a.jcols;
            if (a.jK) {
                const int jm = jcol / NV, jn = jcol - jm * NV;
#pragma unroll
                for (int n = 0; n < NV; ++n) {
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
        // ldcrd(n,0) = dx_n/dr, ldcrd(n,1) = dx_n/ds (rsdl.cpp:44-47)
        const T l00 = T(0.5 * (x2 - x1)), l01 = T(0.5 * (x0 - x1));
        const T l10 = T(0.5 * (y2 - y1)), l11 = T(0.5 * (y0 - y1));

        const V4 z = {T(0), T(0), T(0), T(0)};
        // curved: dx/dr, dx/ds, dy/dr, dy/ds at the Gauss points.  The coordinate modes
        // are taken relative to vertex 1 (the derivatives of a constant vanish), which
        // keeps the FP32 form free of the cancellation of absolute coordinates.
        V4 Xr[CURV ? GT : 1], Xs[CURV ? GT : 1], Yr[CURV ? GT : 1], Ys[CURV ? GT : 1];
        if constexpr (CURV) {
            constexpr int SMD = D::SM > 0 ? D::SM : 1;
            const int cidx = a.begin + g * 16 + e;
            T bx[KT], by[KT];
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int k = 4 * s + q;
                T cx = T(0), cy = T(0);
                if (k == 0) { cx = T(x0 - x1); cy = T(y0 - y1); }
                else if (k == 2) { cx = T(x2 - x1); cy = T(y2 - y1); }
                else if (k >= 3 && k < D::BM && S.t >= 0) {
                    const int i = (k - 3) / SMD, m = (k - 3) - i * SMD;
                    const double* cr = a.crv + ((size_t)(cidx * 3 + i) * a.sm0 + m) * 2;
                    cx = T(cr[0]); cy = T(cr[1]);
                }
                bx[s] = cx; by[s] = cy;
            }
#pragma unroll
            for (int mt = 0; mt < GT; ++mt) {
                V4 c1 = z, c2 = z, c3 = z, c4 = z;
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    const T ar = sops[D::OFF_PR + (mt * KT + s) * 64 + lane];
                    const T as = sops[D::OFF_PS + (mt * KT + s) * 64 + lane];
                    c1 = mfma(ar, bx[s], c1); c2 = mfma(as, bx[s], c2);
                    c3 = mfma(ar, by[s], c3); c4 = mfma(as, by[s], c4);
                }
                Xr[mt] = c1; Xs[mt] = c2; Yr[mt] = c3; Ys[mt] = c4;
            }
        }
        // metric terms of Gauss point (mt, i): the element constants of a straight
        // element, the projected derivatives of a curved one.  The padding rows of the
        // tiles (points beyond the G Gauss points) have zero operator rows, hence a zero
        // Jacobian; they keep the straight metric so that their values stay finite (the
        // integrations weight them by zero, and 0 x inf would reach every mode).
        auto metric = [&](int mt, int i, T& m00, T& m01, T& m10, T& m11) {
            if constexpr (CURV) {
                m00 = Xr[mt][i]; m01 = Xs[mt][i]; m10 = Yr[mt][i]; m11 = Ys[mt][i];
                if (m00 * m11 - m10 * m01 == T(0)) { m00 = l00; m01 = l01; m10 = l10; m11 = l11; }
            } else {
                m00 = l00; m01 = l01; m10 = l10; m11 = l11;
            }
        };
        V4 U[GT], V[GT], Pp[GT];
#pragma unroll
        for (int mt = 0; mt < GT; ++mt) {
            V4 cu = z, cv = z, cp = z;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const T av = sops[D::OFF_P + (mt * KT + s) * 64 + lane];
                cu = mfma(av, b[0][s], cu);
                cv = mfma(av, b[1][s], cv);
                cp = mfma(av, b[2][s], cp);
            }
            U[mt] = cu; V[mt] = cv; Pp[mt] = cp;
        }

        // inviscid fluxes (rsdl.cpp:262-291): continuity C, momentum A
        V4 C0[GT], C1[GT], A00[GT], A01[GT], A10[GT], A11[GT];
        const T rho = a.rho;
#pragma unroll
        for (int mt = 0; mt < GT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                T m00, m01, m10, m11;
                metric(mt, i, m00, m01, m10, m11);
                const T u = U[mt][i], v = V[mt][i], pr = Pp[mt][i];
                const T fx = rho * u, fy = rho * v;
                const T c0 = +m11 * fx - m01 * fy;
                const T c1 = -m10 * fx + m00 * fy;
                C0[mt][i] = c0; C1[mt][i] = c1;
                A00[mt][i] = u * c0 + m11 * pr;
                A01[mt][i] = u * c1 - m10 * pr;
                A10[mt][i] = v * c0 - m01 * pr;
                A11[mt][i] = v * c1 + m00 * pr;
            }

        // lf_im = intgrtrs of the inviscid fluxes (rsdl.cpp:292-294)
        V4 LI0 = z, LI1 = z, LI2 = z;
#pragma unroll
        for (int kt = 0; kt < GT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // f64 layout: K-step (tile kt, register i) holds points 16 kt + 4 i .. + 3;
                // a step of padding points only (past the G Gauss points) adds nothing
                if (sizeof(T) == 8 && 16 * kt + 4 * i >= D::G) continue;
                const int kk = kt * 4 + i;
                const T ar = sops[D::OFF_IR + kk * 64 + lane];
                const T as = sops[D::OFF_IS + kk * 64 + lane];
                LI0 = mfma(ar, A00[kt][i], LI0); LI0 = mfma(as, A01[kt][i], LI0);
                LI1 = mfma(ar, A10[kt][i], LI1); LI1 = mfma(as, A11[kt][i], LI1);
                LI2 = mfma(ar, C0[kt][i], LI2);  LI2 = mfma(as, C1[kt][i], LI2);
            }

        V4 LR0 = z, LR1 = z, LR2 = z;
        if constexpr (FULL) {
            // derivatives of u, v at the Gauss points (proj with r/s derivatives)
            V4 Ur[GT], Us[GT], Vr[GT], Vs[GT];
#pragma unroll
            for (int mt = 0; mt < GT; ++mt) {
                V4 c1 = z, c2 = z, c3 = z, c4 = z;
#pragma unroll
                for (int s = 0; s < KT; ++s) {
                    const T ar = sops[D::OFF_PR + (mt * KT + s) * 64 + lane];
                    const T as = sops[D::OFF_PS + (mt * KT + s) * 64 + lane];
                    c1 = mfma(ar, b[0][s], c1); c2 = mfma(as, b[0][s], c2);
                    c3 = mfma(ar, b[1][s], c3); c4 = mfma(as, b[1][s], c4);
                }
                Ur[mt] = c1; Us[mt] = c2; Vr[mt] = c3; Vs[mt] = c4;
            }
            // viscous stress tensor (rsdl.cpp:303-326, curved :139-159 per point); steady
            // so rhobd0 = 0
            const T cjcb = l00 * l11 - l10 * l01;
            const T cjcbi = a.mu / cjcb;
            T v0000 = -cjcbi * (T(2) * l11 * l11 + l01 * l01);
            T v0011 = -cjcbi * (T(2) * l10 * l10 + l00 * l00);
            T v0001 = cjcbi * (T(2) * l11 * l10 + l01 * l00);
            T v1100 = -cjcbi * (l11 * l11 + T(2) * l01 * l01);
            T v1111 = -cjcbi * (l10 * l10 + T(2) * l00 * l00);
            T v1101 = cjcbi * (l11 * l10 + T(2) * l01 * l00);
            T v0100 = cjcbi * l01 * l11;
            T v0111 = cjcbi * l00 * l10;
            T v0101 = -cjcbi * l01 * l10;
            T v0110 = -cjcbi * l00 * l11;
            V4 F00[GT], F01[GT], F10[GT], F11[GT];
#pragma unroll
            for (int mt = 0; mt < GT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (CURV) {
                        T m00, m01, m10, m11;
                        metric(mt, i, m00, m01, m10, m11);
                        const T cji = a.mu / (m00 * m11 - m10 * m01);
                        v0000 = -cji * (T(2) * m11 * m11 + m01 * m01);
                        v0011 = -cji * (T(2) * m10 * m10 + m00 * m00);
                        v0001 = cji * (T(2) * m11 * m10 + m01 * m00);
                        v1100 = -cji * (m11 * m11 + T(2) * m01 * m01);
                        v1111 = -cji * (m10 * m10 + T(2) * m00 * m00);
                        v1101 = cji * (m11 * m10 + T(2) * m01 * m00);
                        v0100 = cji * m01 * m11;
                        v0111 = cji * m00 * m10;
                        v0101 = -cji * m01 * m10;
                        v0110 = -cji * m00 * m11;
                    }
                    const T ur = Ur[mt][i], us = Us[mt][i], vr = Vr[mt][i], vs = Vs[mt][i];
                    const T f00 = v0000 * ur + v0100 * vr + v0001 * us + v0101 * vs;
                    const T f01 = v0001 * ur + v0110 * vr + v0011 * us + v0111 * vs;
                    const T f10 = v0100 * ur + v1100 * vr + v0110 * us + v1101 * vs;
                    const T f11 = v0101 * ur + v1101 * vr + v0111 * us + v1111 * vs;
                    F00[mt][i] = f00; F01[mt][i] = f01; F10[mt][i] = f10; F11[mt][i] = f11;
                    A00[mt][i] += f00; A01[mt][i] += f01; A10[mt][i] += f10; A11[mt][i] += f11;
                }
            // strong residual: derivr/derivs of the total fluxes (rsdl.cpp:369-375)
            V4 R0[GT], R1[GT], R2[GT];
#pragma unroll
            for (int mt = 0; mt < GT; ++mt) {
                V4 r0 = z, r1 = z, r2 = z;
#pragma unroll
                for (int kt = 0; kt < GT; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (sizeof(T) == 8 && 16 * kt + 4 * i >= D::G) continue;  // padding points only
                        const int kk = (mt * GT + kt) * 4 + i;
                        const T dr = sops[D::OFF_DR + kk * 64 + lane];
                        const T ds = sops[D::OFF_DS + kk * 64 + lane];
                        r0 = mfma(dr, A00[kt][i], r0); r0 = mfma(ds, A01[kt][i], r0);
                        r1 = mfma(dr, A10[kt][i], r1); r1 = mfma(ds, A11[kt][i], r1);
                        r2 = mfma(dr, C0[kt][i], r2);  r2 = mfma(ds, C1[kt][i], r2);
                    }
                R0[mt] = r0; R1[mt] = r1; R2[mt] = r2;
            }
            if (sizeof(T) == 8 && a.lin) {
                // linearisation data of this 16-element group, coalesced per (field, tile, reg)
                float* L = a.lin + (size_t)(a.gbase + g) * (5 * GT * 4 * 64);
#pragma unroll
                for (int mt = 0; mt < GT; ++mt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int o = (mt * 4 + i) * 64 + lane;
                        L[0 * GT * 256 + o] = (float)U[mt][i];
                        L[1 * GT * 256 + o] = (float)V[mt][i];
                        L[2 * GT * 256 + o] = (float)R0[mt][i];
                        L[3 * GT * 256 + o] = (float)R1[mt][i];
                        L[4 * GT * 256 + o] = (float)R2[mt][i];
                    }
            }
            // per-point tau (CALC_TAU2, rsdl.cpp:377-395) and the stabilisation (:397-421)
            const T dx1 = T(x0 - x2), dy1 = T(y0 - y2), dx2 = T(x1 - x0), dy2 = T(y1 - y0);
            const T ar2 = dx1 * dy2 - dy1 * dx2;
            const T perim = sqrt(dx1 * dx1 + dy1 * dy1) + sqrt(dx2 * dx2 + dy2 * dy2) +
                            sqrt((dx1 + dx2) * (dx1 + dx2) + (dy1 + dy2) * (dy1 + dy2));
            const T h = (ar2 / perim) / (T(0.25) * (P + 1) * (P + 1));
            const T nu = a.mu / rho;
            const T gv = T(2) * nu / h;
            const T gvis = gv * gv;
            const T tfac = a.adis * h / cjcb;
#pragma unroll
            for (int mt = 0; mt < GT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    T m00, m01, m10, m11;
                    metric(mt, i, m00, m01, m10, m11);
                    const T u = U[mt][i], v = V[mt][i];
                    const T qq = u * u + v * v;
                    T gam = T(3) * qq + gvis;
                    if (a.mu == T(0)) gam = fmax(gam, T(0.1));
                    // curved: cjcb of this Gauss point (rsdl.cpp:385)
                    const T tf = CURV ? a.adis * h / (m00 * m11 - m10 * m01) : tfac;
                    const T tau0 = tf / sqrt(gam);
                    const T tau2 = sqrt(qq) * tau0;
                    const T t0 = tau0 * R0[mt][i], t1 = tau0 * R1[mt][i], t2 = tau2 * R2[mt][i];
                    F00[mt][i] -= (m11 * (T(2) * u) - m01 * v) * t0 - m01 * u * t1 + m11 * t2;
                    F01[mt][i] -= (-m10 * (T(2) * u) + m00 * v) * t0 + m00 * u * t1 - m10 * t2;
                    F10[mt][i] -= +m11 * v * t0 + (m11 * u - m01 * (T(2) * v)) * t1 - m01 * t2;
                    F11[mt][i] -= -m10 * v * t0 + (-m10 * u + m00 * (T(2) * v)) * t1 + m00 * t2;
                    C0[mt][i] = -(m11 * t0 - m01 * t1);
                    C1[mt][i] = -(-m10 * t0 + m00 * t1);
                }
            if constexpr (!JAC) load_old();
            // lf_re = intgrtrs of viscous - stabilisation fluxes (rsdl.cpp:424-426)
#pragma unroll
            for (int kt = 0; kt < GT; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (sizeof(T) == 8 && 16 * kt + 4 * i >= D::G) continue;  // padding points only
                    const int kk = kt * 4 + i;
                    const T ar = sops[D::OFF_IR + kk * 64 + lane];
                    const T as = sops[D::OFF_IS + kk * 64 + lane];
                    LR0 = mfma(ar, F00[kt][i], LR0); LR0 = mfma(as, F01[kt][i], LR0);
                    LR1 = mfma(ar, F10[kt][i], LR1); LR1 = mfma(as, F11[kt][i], LR1);
                    LR2 = mfma(ar, C0[kt][i], LR2);  LR2 = mfma(as, C1[kt][i], LR2);
                }
        }


        if constexpr (!FULL && !JAC) load_old();
        if constexpr (JAC) {
            constexpr int N = D::TM * NV;
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int k = 4 * s + q;
                if (S.t < 0 || k >= D::TM) continue;
                const T li[3] = {LI0[s], LI1[s], LI2[s]}, lr[3] = {LR0[s], LR1[s], LR2[s]};
#pragma unroll
                for (int n = 0; n < NV; ++n) {
                    const T R = FULL ? lr[n] * a.beta + li[n] : li[n];
                    const size_t r = (size_t)jel * N + (k * NV + n);
                    if (a.jK) a.jK[r * N + jcol] = (R - a.jbase[r]) / jdw;
                    else a.jbase[r] = R;
                }
            }
            S = Sn;
            cnext = cn2;
            tnext2 = tn3;
            continue;
        }
        if constexpr (EM) {
            // element-major output of the vertex and side modes, side sign applied:
            // eres[(t*BM + k)*2*NV + n] = lf_im, [... + NV + n] = beta lf_re; without the real
            // part (FULL = false) eres[(t*BM + k)*NV + n] = lf_im (half the bytes); the gather kernels add the carried real part and sum over
            // the elements.  Interior modes belong to this element: final here, started
            // from keep * res_r as on a first visit.
#pragma unroll
            for (int s = 0; s < KT; ++s) {
                const int k = 4 * s + q, kind = mode_kind<P>(k);
                if (S.t < 0 || k >= D::TM) continue;
                const T sg = S.off[s] < 0 ? T(-1) : T(1);
                const T li[3] = {sg * LI0[s], sg * LI1[s], sg * LI2[s]};
                T lr[3] = {T(0), T(0), T(0)};
                if constexpr (FULL) {
                    const T bt = a.beta;
                    lr[0] = sg * (LR0[s] * bt);
                    lr[1] = sg * (LR1[s] * bt);
                    lr[2] = sg * (LR2[s] * bt);
                }
                if (kind < 2) {
                    T* o = eres + ((size_t)S.t * D::BM + k) * (FULL ? 2 * NV : NV);
#pragma unroll
                    for (int n = 0; n < NV; ++n) {
                        o[n] = li[n];
                        if constexpr (FULL) o[NV + n] = lr[n];
                    }
                } else {
                    const int off = S.off[s];
#pragma unroll
                    for (int n = 0; n < NV; ++n) {
                        const T r0 = a.keep == T(0) ? T(0) : a.keep * ro[n][s];
                        if (FULL || a.keep != T(1)) a.rri[off + n] = r0 + lr[n];
                        if (sizeof(T) == 4 && a.srci)
                            a.resi[off + n] = r0 + lr[n] + li[n] + T(a.srci[off + n] * a.sfac[0]);
                        else
                            a.resi[off + n] = r0 + lr[n] + li[n];
                    }
                }
            }
            S = Sn;
            cnext = cn2;
            tnext2 = tn3;
            continue;
        }
        // lftog: res = sum lf_im + res_r,  res_r = (1-beta) res_r + beta sum lf_re
        // (tri_hp/nstage.cpp:21-82).  The first colour that touches a coefficient
        // starts both sums from keep * res_r; interiors belong to one element.
#pragma unroll
        for (int s = 0; s < KT; ++s) {
            const int k = 4 * s + q, kind = mode_kind<P>(k);
            if (S.t < 0 || k >= D::TM) continue;
            const int off = S.off[s] < 0 ? ~S.off[s] : S.off[s];
            const T sg = S.off[s] < 0 ? T(-1) : T(1);
            T* di = kind == 0 ? a.resv : (kind == 1 ? a.ress : a.resi);
            T* dr = kind == 0 ? a.rrv : (kind == 1 ? a.rrs : a.rri);
            const T li[3] = {sg * LI0[s], sg * LI1[s], sg * LI2[s]};
            T lr[3] = {T(0), T(0), T(0)};
            if constexpr (FULL) {
                const T bt = a.beta;
                lr[0] = sg * (LR0[s] * bt);
                lr[1] = sg * (LR1[s] * bt);
                lr[2] = sg * (LR2[s] * bt);
            }
            if ((S.first >> s) & 1) {
                // FP32 inner solve: the constant source sfac * R64(u0) enters once, on
                // the first visit (null in the FP64 kernel)
                const double* sr = kind == 0 ? a.srcv : (kind == 1 ? a.srcs : a.srci);
#pragma unroll
                for (int n = 0; n < NV; ++n) {
                    const T r0 = a.keep == T(0) ? T(0) : a.keep * ro[n][s];
                    if (FULL || a.keep != T(1)) dr[off + n] = r0 + lr[n];
                    if (sizeof(T) == 4 && sr)
                        di[off + n] = r0 + lr[n] + li[n] + T(sr[off + n] * a.sfac[0]);
                    else
                        di[off + n] = r0 + lr[n] + li[n];
                }
            } else {
#pragma unroll
                for (int n = 0; n < NV; ++n) {
                    if constexpr (FULL) dr[off + n] = ro[n][s] + lr[n];
                    di[off + n] = io[n][s] + lr[n] + li[n];
                }
            }
        }
        S = Sn;
        cnext = cn2;
        tnext2 = tn3;
    }
}

template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_ins(ElemArgs a) {
    elem_ins_body<double, P, FULL>(a);
}

// ---------------------------------------------------------------------------------
// Mode-array helpers over v(nent, mstride, NV) with the first nm modes active.
// op 0: x = 0, y *= c           (rsdl start, tri_hp/nstage.cpp:21-49)
// op 1: x += y                  (rsdl end, nstage.cpp:76-82; mg_source later visits)
// op 2: y = c*z - x, x += y     (mg_source first visit, nstage.cpp:113-128)
// op 3: y = x                   (mg_restrict, movco.cpp:18-37)
// op 4: x = y - c*z             (update, nstage.cpp:387-409)
// Up to three arrays (vertex, side, interior modes) as one index range, one launch.
struct ModeSpan {
    long end[3];      // running counts of active values
    int per[3];       // active values per entity: nm * NV
    int stride[3];    // values per entity in memory: mstride * NV
    double *x[3], *y[3];
    const double* z[3];
};
__global__ __launch_bounds__(256) void k_modes(int op, ModeSpan m, double c) {
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m.end[2]) return;
    const int i = k < m.end[0] ? 0 : (k < m.end[1] ? 1 : 2);
    if (i) k -= i == 1 ? m.end[0] : m.end[1];
    const int per = i == 0 ? m.per[0] : (i == 1 ? m.per[1] : m.per[2]);
    const int stride = i == 0 ? m.stride[0] : (i == 1 ? m.stride[1] : m.stride[2]);
    double* x = i == 0 ? m.x[0] : (i == 1 ? m.x[1] : m.x[2]);
    double* y = i == 0 ? m.y[0] : (i == 1 ? m.y[1] : m.y[2]);
    const double* z = i == 0 ? m.z[0] : (i == 1 ? m.z[1] : m.z[2]);
    const long ent = k / per, ix = ent * stride + (k - ent * per);
    switch (op) {
        case 0: x[ix] = 0.0; y[ix] *= c; break;
        case 1: x[ix] += y[ix]; break;
        case 2: { const double d = c * z[ix] - x[ix]; y[ix] = d; x[ix] += d; } break;
        case 3: y[ix] = x[ix]; break;
        case 4: x[ix] = y[ix] - c * z[ix]; break;
    }
}

// edge-boundary flux residual, tri_hp/hp_boundary.cpp:973-1049 with bdry_ins::generic::flux
// S: storage type of the state and residual (double, or float for the FP32 inner
// solve of the defect correction); the flux arithmetic is FP64 in both
template <typename S>
struct EdgeArgsT {
    const int* eseg;
    int begin, end;
    const int* seg_pnt;
    const double* pnts;
    const S* ugv;
    const S* ugs;
    S* resv;
    S* ress;
    const double* g1;   // gpx x (sm+2)
    const double* dg1;
    const double* w1;
    int gpx, sm, sm0;
    double rho, bc_pressure;
    // curved boundary sides (may be null): row of each edge idx in scrd, -1 if straight;
    // scrd rows hold the side's coordinate modes (sm0 modes, x/y) in the side's direction
    const int* ecrv;
    const double* scrd;
    // flux type of each edge idx (may be null: all generic), the freestream velocity of
    // the euler and characteristic fluxes (the freestream pressure is bc_pressure), mu
    // for the characteristic's gam
    const unsigned char* etype;
    double ub0, ub1, mu;
};
typedef EdgeArgsT<double> EdgeArgs;

enum EdgeFlux : unsigned char { EDGE_GENERIC = 0, EDGE_EULER = 1, EDGE_CHARACTERISTIC = 2 };

// boundary flux of tri_hp_ins at one Gauss point (steady, mesh velocity zero), unit
// normal (nx, ny), jcb the point's length factor |dx/dxi|:
//   generic (inflow, outflow, symmetry), bdry_ins.h:34-49: mass flux with the interior
//     velocity, the freestream pressure pb on the momentum;
//   euler, bdry_ins.h:96-113: mass flux and momentum with the freestream velocity, the
//     interior pressure;
//   characteristic, tri_hp/ins/bdry.cpp:245-320: the boundary state from the
//     characteristic swap between the interior and the freestream (its natural fluxes
//     zero), then the euler-form flux of that state.
template <int P>
__device__ __forceinline__ void edge_flux_ins(int type, const double* u, double nx, double ny, double jcb,
                                              double rho, double mu, double ub0, double ub1, double pb,
                                              double* fl) {
    if (type == EDGE_GENERIC) {
        const double f2 = rho * (u[0] * nx + u[1] * ny);
        fl[0] = f2 * u[0] + pb * nx;
        fl[1] = f2 * u[1] + pb * ny;
        fl[2] = f2;
        return;
    }
    double b0 = ub0, b1 = ub1, b2 = u[2];
    if (type == EDGE_CHARACTERISTIC) {
        const double rhoi = 1. / rho, nu = mu / rho;
        const double hmax = jcb * 2.0 / (0.25 * (P + 1) * (P + 1));
        const double qmax = u[0] * u[0] + u[1] * u[1];
        const double gv = 2. * nu / hmax;
        const double gam = 3.0 * qmax + gv * gv;
        const double ul = u[0] * nx + u[1] * ny, vl = -u[0] * ny + u[1] * nx, pl = u[2];
        const double ur = ub0 * nx + ub1 * ny, vr = -ub0 * ny + ub1 * nx, pr = pb;
        const double cl = sqrt(ul * ul + gam), cr = sqrt(ur * ur + gam);
        const double c = 0.5 * (cl + cr), sn = 0.5 * (ul + ur), vt = 0.5 * (vl + vr);
        const double den = 1. / (2 * c);
        const double lam0 = sn, lam1 = sn + c, lam2 = sn - c;
        const double w0 = ((pl - pr) * rhoi + (ul * lam1 - ur * lam2)) * den;
        const double w1 = lam0 > 0.0 ? vt * ((pr - pl) * rhoi + lam2 * (ur - ul)) * den / (lam0 - lam2) + vl
                                     : vt * ((pr - pl) * rhoi + lam1 * (ur - ul)) * den / (lam0 - lam1) + vr;
        const double w2 = (rho * (ul - ur) * gam - lam2 * pl + lam1 * pr) * den;
        b0 = w0 * nx - w1 * ny;
        b1 = w0 * ny + w1 * nx;
        b2 = w2;
    }
    const double f2 = rho * (b0 * nx + b1 * ny);
    fl[0] = f2 * b0 + b2 * nx;
    fl[1] = f2 * b1 + b2 * ny;
    fl[2] = f2;
}

// P fixes the edge's mode count (p + 1) and Gauss points (p + 1), so the per-lane
// arrays stay in registers
// EM: element-major output eout[(idx*(SM+2) + k)*NV + n], k the two ends then the side
// modes, summed by the gathers, instead of the RMW scatter (the linearisation's path)
template <int P, typename S, bool EM>
__device__ __forceinline__ void edge_ins_body(const EdgeArgsT<S>& a, S* __restrict__ eout, int idx) {
    constexpr int SM = P - 1, N1 = SM + 2, GPX = P + 1;
    if (idx >= a.end) return;
    const int sind = a.eseg[idx];
    const int v0 = a.seg_pnt[2 * sind], v1 = a.seg_pnt[2 * sind + 1];
    double uh[NV][N1];
#pragma unroll
    for (int n = 0; n < NV; ++n) {
        uh[n][0] = a.ugv[v0 * NV + n];
        uh[n][1] = a.ugv[v1 * NV + n];
#pragma unroll
        for (int m = 0; m < SM; ++m) uh[n][m + 2] = a.ugs[(sind * a.sm0 + m) * NV + n];
    }
    const double X0 = a.pnts[2 * v0], Y0 = a.pnts[2 * v0 + 1], X1 = a.pnts[2 * v1], Y1 = a.pnts[2 * v1 + 1];
    // crdtocht1d (tri_hp/gtol.cpp:296-320): the side modes of a curved side's coordinates
    double cx[SM > 0 ? SM : 1], cy[SM > 0 ? SM : 1];
    const int crow = a.ecrv ? a.ecrv[idx] : -1;
    const int etype = a.etype ? a.etype[idx] : EDGE_GENERIC;
#pragma unroll
    for (int m = 0; m < SM; ++m) {
        cx[m] = crow >= 0 ? a.scrd[((size_t)crow * a.sm0 + m) * 2] : 0.0;
        cy[m] = crow >= 0 ? a.scrd[((size_t)crow * a.sm0 + m) * 2 + 1] : 0.0;
    }
    double lf[NV][N1];
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int k = 0; k < N1; ++k) lf[n][k] = 0.0;
#pragma unroll
    for (int ip = 0; ip < GPX; ++ip) {
        const double* g = a.g1 + ip * N1;
        const double* dg = a.dg1 + ip * N1;
        double dxc = X0 * dg[0] + X1 * dg[1];
        double dyc = Y0 * dg[0] + Y1 * dg[1];
        if (crow >= 0) {
#pragma unroll
            for (int m = 0; m < SM; ++m) {
                dxc += cx[m] * dg[m + 2];
                dyc += cy[m] * dg[m + 2];
            }
        }
        double u[NV];
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < N1; ++k) s += uh[n][k] * g[k];
            u[n] = s;
        }
        double nx = dyc, ny = -dxc;
        const double jcb = sqrt(nx * nx + ny * ny);
        nx /= jcb; ny /= jcb;
        double fl[NV];
        edge_flux_ins<P>(etype, u, nx, ny, jcb, a.rho, a.mu, a.ub0, a.ub1, a.bc_pressure, fl);
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const double r = fl[n] * jcb * a.w1[ip];
#pragma unroll
            for (int k = 0; k < N1; ++k) lf[n][k] += g[k] * r;
        }
    }
    if constexpr (EM) {
#pragma unroll
        for (int n = 0; n < NV; ++n)
#pragma unroll
            for (int k = 0; k < N1; ++k) eout[((long)idx * N1 + k) * NV + n] = (S)lf[n][k];
        return;
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
        a.resv[v0 * NV + n] += (S)lf[n][0];
        a.resv[v1 * NV + n] += (S)lf[n][1];
#pragma unroll
        for (int m = 0; m < SM; ++m) a.ress[(sind * a.sm0 + m) * NV + n] += (S)lf[n][m + 2];
    }
}

template <int P>
__global__ __launch_bounds__(64) void k_edge_ins(EdgeArgs a) {
    edge_ins_body<P, double, false>(a, nullptr, a.begin + blockIdx.x * blockDim.x + threadIdx.x);
}

// Element-major residual (no colouring, mesh order): the element body with its EM
// output, persistent over all elements; k_gather_vs then sums the vertex and side
// modes in a fixed order.  At p = 2 the bound of 256 registers keeps two waves per
// SIMD without spilling (272 otherwise, one wave).
// The first eblk blocks (a multiple of 8) compute the boundary-edge fluxes into eout: one
// launch instead of three, and on small meshes the edges' latency hides behind the
// elements' (two edge launches were 10 us of a 31 us stage at 33 x 33, p = 2).
template <int P, bool FULL>
__global__ __launch_bounds__(256, 2) void k_elem_ins_em(ElemArgs a, double* eres, EdgeArgs e,
                                                                     double* eout, int eblk) {
    if ((int)blockIdx.x < eblk) {
        edge_ins_body<P, double, true>(e, eout, blockIdx.x * 256 + threadIdx.x);
        return;
    }
    elem_ins_body<double, P, FULL, true>(a, eres, eblk);
}

// ---------------------------------------------------------------------------------
// The FP64 residual of straight elements at p = 4 on v_mfma_f64_4x4x4f64 (see mfma4): 16
// elements per wave, lane l = 16 q + e.  Point layout, 28 places for the 5 x 5 Gauss grid
// (i, j): register r < 5 of row q is (r, q), register 5 is (q, 4), register 6 is (4, 4)
// (rows 1-3 repeat it, their weights are zero).  So the x lines j < 4 lie in a lane's
// registers, and their derivative is a 5-term sum on the vector unit; only the line j = 4 and
// the y derivatives are products.  The strong residual of a variable takes 23 blocks and 60
// multiply-adds, 620 cycles, against 1 792 of the dense 25 x 25 operators in 16-row tiles.
// Fluxes are formed when they are consumed: 256 registers, two waves per SIMD (the 16x16x4
// form kept all of them, 482 registers and one wave, and waited for every load).
// The next group's data are loaded a group ahead (without: 367 and 190 us).
// Bound by the FP64 unit.  512 x 512: full 482 -> 332 us, inviscid 190 -> 151 us a launch.
struct TI4 {
    static constexpr int P = 0;      // 28: values at register r from K-step s, [4 r + s]
    static constexpr int PR = 28;    // 28: r derivatives
    static constexpr int PS = 56;    // 28: s derivatives
    static constexpr int IR = 84;    // 28: tests, [4 r + row block]
    static constexpr int IS = 112;   // 28
    static constexpr int LA = 140;   // 4: n0 Lx on the line j = 4, [2 out + in] (registers 5, 6)
    static constexpr int LX = 144;   // 4: n0 x0 Lx there
    static constexpr int LB = 148;   // y derivative among j < 4
    static constexpr int LB4 = 149;  // 4: from (i, 4) to (i, j), column i
    static constexpr int LB5 = 153;  // 4: from (i, j) to (i, 4), row i
    static constexpr int N0 = 157;   // n0 of row q (not an operand)
    static constexpr int COUNT = 158;
};
struct TriLines {
    double lx[25], x0[5], ly44;
};

// collapsed-coordinate derivatives of one variable's fluxes (derivr of fr + derivs of fs)
__device__ __forceinline__ void tri_lines(const TriLines& ln, const double* op, const double fr[7], const double fs[7],
                                          double R[7]) {
    const double n0 = op[16 * TI4::N0];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        double t = ln.lx[5 * i] * fr[0], t2 = ln.lx[5 * i] * fs[0];
#pragma unroll
        for (int n = 1; n < 5; ++n) { t += ln.lx[5 * i + n] * fr[n]; t2 += ln.lx[5 * i + n] * fs[n]; }
        R[i] = n0 * (t + ln.x0[i] * t2);
    }
    const double lb = op[16 * TI4::LB];
#pragma unroll
    for (int i = 0; i < 5; ++i) R[i] = mfma4(lb, fs[i], R[i]);
#pragma unroll
    for (int i = 0; i < 5; ++i) R[i] = mfma4(op[16 * (TI4::LB4 + (i & 3))], i < 4 ? fs[5] : fs[6], R[i]);
#pragma unroll
    for (int o = 0; o < 2; ++o) {
        double s = ln.ly44 * fs[5 + o];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            s = mfma4(op[16 * (TI4::LA + 2 * o + i)], fr[5 + i], s);
            s = mfma4(op[16 * (TI4::LX + 2 * o + i)], fs[5 + i], s);
        }
        R[5 + o] = s;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) R[5] = mfma4(op[16 * (TI4::LB5 + i)], fs[i], R[5]);
    R[6] = mfma4(op[16 * TI4::LB5], fs[4], R[6]);
}

template <bool FULL>
__device__ __forceinline__ void elem_ins4_body(const ElemArgs& a, const double* __restrict__ ops, const TriLines& ln,
                                               double* __restrict__ eres, int eblk) {
    using D = Dims<4>;
    constexpr int REC = FULL ? 2 * NV : NV;
    __shared__ double sops[TI4::COUNT * 16];
    for (int k = threadIdx.x; k < TI4::COUNT * 16; k += blockDim.x) sops[k] = ops[k];
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = lane & 15, q = lane >> 4;
    const double* op = sops + (lane & 3) + 4 * q;  // this lane's element of block b: op[16 b]
    // groups of 16 elements per XCD and wave as in elem_ins_body
    const int WX = (((int)gridDim.x - eblk) >> 3) * 4;
    const int rank = (((int)blockIdx.x - eblk) >> 3) * 4 + w;
    const int xcd = blockIdx.x & 7;
    const int ng = (a.end - a.begin + 15) >> 4;
    const int gpx = (ng + 7) >> 3;
    const int g0 = xcd * gpx + rank;
    const int gend = min(ng, (xcd + 1) * gpx);
    if (g0 >= gend) return;
    // the state and coordinates of a group are loaded while the group before it is computed
    // (ahead of its stores, which the loads would otherwise wait for), its indices one earlier
    ElemConn cnext = elem_conn(a, elem_of_group(a, g0, gend, e));
    ElemSlots<4> Sn;
    double raw[NV][4];
    auto ahead = [&](int g) {  // g: the group whose indices cnext holds
        Sn = elem_slots<4>(a, cnext, q);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = 4 * s + q, kind = mode_kind<4>(k);
            const int off = Sn.off[s] < 0 ? ~Sn.off[s] : Sn.off[s];
            const double* src = kind == 0 ? a.ugv : (kind == 1 ? a.ugs : a.ugi);
            const bool live = Sn.t >= 0 && k < D::TM;
#pragma unroll
            for (int n = 0; n < NV; ++n) raw[n][s] = live ? src[off + n] : 0.0;
        }
        cnext = elem_conn(a, elem_of_group(a, g + WX, gend, e));
    };
    ahead(g0);
    for (int g = g0; g < gend; g += WX) {
        group_phase();
        const ElemSlots<4> S = Sn;
        // modal coefficients: K-step s of lane l is mode 4 s + q
        double b[NV][4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int n = 0; n < NV; ++n) b[n][s] = S.off[s] < 0 ? -raw[n][s] : raw[n][s];
        // ldcrd(n,0) = dx_n/dr, ldcrd(n,1) = dx_n/ds (rsdl.cpp:44-47): l00, l01, l10, l11
        double l[4] = {0.5 * (S.x[2] - S.x[1]), 0.5 * (S.x[0] - S.x[1]), 0.5 * (S.y[2] - S.y[1]),
                       0.5 * (S.y[0] - S.y[1])};
        const double rho = a.rho;
        group_phase();
        if constexpr (!FULL) ahead(g + WX);
        double U[NV][7];
#pragma unroll
        for (int r = 0; r < 7; ++r) {
            if (r == 3 || r == 5) group_phase();
#pragma unroll
            for (int n = 0; n < NV; ++n) U[n][r] = 0.0;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const double av = op[16 * (TI4::P + 4 * r + s)];
#pragma unroll
                for (int n = 0; n < NV; ++n) U[n][r] = mfma4(av, b[n][s], U[n][r]);
            }
        }
        // inviscid fluxes at register r (rsdl.cpp:262-291): mass c, momentum f[n], directions r, s
        auto inviscid = [&](int r, double c[2], double f0[2], double f1[2]) {
            const double u = U[0][r], v = U[1][r], pr = U[2][r];
            const double fx = rho * u, fy = rho * v;
            c[0] = l[3] * fx - l[1] * fy;
            c[1] = l[0] * fy - l[2] * fx;
            f0[0] = u * c[0] + l[3] * pr;
            f0[1] = u * c[1] - l[2] * pr;
            f1[0] = v * c[0] - l[1] * pr;
            f1[1] = v * c[1] + l[0] * pr;
        };
        auto test = [&](int r, const double f0[2], const double f1[2], const double c[2], double L[NV][4]) {
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const double ar = op[16 * (TI4::IR + 4 * r + rb)], as = op[16 * (TI4::IS + 4 * r + rb)];
                L[0][rb] = mfma4(ar, f0[0], L[0][rb]); L[1][rb] = mfma4(ar, f1[0], L[1][rb]);
                L[2][rb] = mfma4(ar, c[0], L[2][rb]);  L[0][rb] = mfma4(as, f0[1], L[0][rb]);
                L[1][rb] = mfma4(as, f1[1], L[1][rb]); L[2][rb] = mfma4(as, c[1], L[2][rb]);
            }
        };
        auto store = [&](const double L[NV][4], int at, double f) {
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const int k = 4 * s + q;
                if (S.t < 0) continue;
                const double sg = S.off[s] < 0 ? -f : f;
                double* o = eres + ((size_t)S.t * D::BM + k) * REC + at;
#pragma unroll
                for (int n = 0; n < NV; ++n) o[n] = sg * L[n][s];
            }
        };
        static_assert(D::BM == 12, "row blocks 0-2 hold the vertex and side modes");
        // lf_im = intgrtrs of the inviscid fluxes (rsdl.cpp:292-294); li: interior modes
        double li[NV];
        {
            double L[NV][4];
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int rb = 0; rb < 4; ++rb) L[n][rb] = 0.0;
#pragma unroll
            for (int r = 0; r < 7; ++r) {
                group_phase();
                double c[2], f0[2], f1[2];
                inviscid(r, c, f0, f1);
                test(r, f0, f1, c, L);
            }
            store(L, 0, 1.0);
#pragma unroll
            for (int n = 0; n < NV; ++n) li[n] = L[n][3];
        }
        double lr[NV] = {0.0, 0.0, 0.0};
        if constexpr (FULL) {
            group_opaque(l);
            const double cjcb = l[0] * l[3] - l[2] * l[1];
            // viscous fluxes (rsdl.cpp:303-326) F[r] = {f00, f01, f10, f11}
            double F[7][4];
            {
                const double cj = a.mu / cjcb;
                const double v0000 = -cj * (2.0 * l[3] * l[3] + l[1] * l[1]), v0011 = -cj * (2.0 * l[2] * l[2] + l[0] * l[0]);
                const double v0001 = cj * (2.0 * l[3] * l[2] + l[1] * l[0]);
                const double v1100 = -cj * (l[3] * l[3] + 2.0 * l[1] * l[1]), v1111 = -cj * (l[2] * l[2] + 2.0 * l[0] * l[0]);
                const double v1101 = cj * (l[3] * l[2] + 2.0 * l[1] * l[0]);
                const double v0100 = cj * l[1] * l[3], v0111 = cj * l[0] * l[2];
                const double v0101 = -cj * l[1] * l[2], v0110 = -cj * l[0] * l[3];
#pragma unroll
                for (int r = 0; r < 7; ++r) {
                    group_phase();
                    double ur = 0.0, us = 0.0, vr = 0.0, vs = 0.0;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const double ar = op[16 * (TI4::PR + 4 * r + s)], as = op[16 * (TI4::PS + 4 * r + s)];
                        ur = mfma4(ar, b[0][s], ur); us = mfma4(as, b[0][s], us);
                        vr = mfma4(ar, b[1][s], vr); vs = mfma4(as, b[1][s], vs);
                    }
                    F[r][0] = v0000 * ur + v0100 * vr + v0001 * us + v0101 * vs;
                    F[r][1] = v0001 * ur + v0110 * vr + v0011 * us + v0111 * vs;
                    F[r][2] = v0100 * ur + v1100 * vr + v0110 * us + v1101 * vs;
                    F[r][3] = v0101 * ur + v1101 * vr + v0111 * us + v1111 * vs;
                }
            }
            // strong residual: derivr/derivs of the total fluxes (rsdl.cpp:369-375)
            double R[NV][7], fr[7], fs[7];
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                group_opaque(l);
#pragma unroll
                for (int r = 0; r < 7; ++r) {
                    double c[2], f0[2], f1[2];
                    inviscid(r, c, f0, f1);
                    fr[r] = n == 0 ? f0[0] + F[r][0] : (n == 1 ? f1[0] + F[r][2] : c[0]);
                    fs[r] = n == 0 ? f0[1] + F[r][1] : (n == 1 ? f1[1] + F[r][3] : c[1]);
                }
                group_phase();
                tri_lines(ln, op, fr, fs, R[n]);
            }
            ahead(g + WX);
            // per-point tau (CALC_TAU2, rsdl.cpp:377-395) and the stabilisation (:397-421)
            group_opaque(l);
            const double dx1 = -2.0 * (l[0] - l[1]), dy1 = -2.0 * (l[2] - l[3]), dx2 = -2.0 * l[1], dy2 = -2.0 * l[3];
            const double ar2 = dx1 * dy2 - dy1 * dx2;
            const double perim = sqrt(dx1 * dx1 + dy1 * dy1) + sqrt(dx2 * dx2 + dy2 * dy2) +
                                 sqrt((dx1 + dx2) * (dx1 + dx2) + (dy1 + dy2) * (dy1 + dy2));
            const double h = (ar2 / perim) / (0.25 * 5 * 5);
            const double gv = 2.0 * (a.mu / rho) / h, gvis = gv * gv, tfac = a.adis * h / cjcb;
            double L[NV][4];
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int rb = 0; rb < 4; ++rb) L[n][rb] = 0.0;
#pragma unroll
            for (int r = 0; r < 7; ++r) {
                group_phase();
                const double u = U[0][r], v = U[1][r];
                const double qq = u * u + v * v;
                double gam = 3.0 * qq + gvis;
                if (a.mu == 0.0) gam = fmax(gam, 0.1);
                const double tau0 = tfac / sqrt(gam);
                const double tau2 = sqrt(qq) * tau0;
                const double t0 = tau0 * R[0][r], t1 = tau0 * R[1][r], t2 = tau2 * R[2][r];
                // with q_d = the contravariant velocity and t_d = the contravariant t:
                // (q_d t_n + u_n t_d + cofactor t2), and t_d
                const double q0 = l[3] * u - l[1] * v, q1 = l[0] * v - l[2] * u;
                const double s0 = l[3] * t0 - l[1] * t1, s1 = l[0] * t1 - l[2] * t0;
                const double c[2] = {-s0, -s1};
                const double f0[2] = {F[r][0] - (q0 * t0 + u * s0 + l[3] * t2), F[r][1] - (q1 * t0 + u * s1 - l[2] * t2)};
                const double f1[2] = {F[r][2] - (q0 * t1 + v * s0 - l[1] * t2), F[r][3] - (q1 * t1 + v * s1 + l[0] * t2)};
                test(r, f0, f1, c, L);
            }
            store(L, NV, a.beta);
#pragma unroll
            for (int n = 0; n < NV; ++n) lr[n] = a.beta * L[n][3];
        }
        // interior modes belong to this element: final here, started from keep * res_r
        if (S.t >= 0 && q < 3) {
            const int off = S.off[3];
#pragma unroll
            for (int n = 0; n < NV; ++n) {
                const double r0 = a.keep == 0.0 ? 0.0 : a.keep * a.rri[off + n];
                if (FULL || a.keep != 1.0) a.rri[off + n] = r0 + lr[n];
                a.resi[off + n] = r0 + lr[n] + li[n];
            }
        }
    }
}

template <bool FULL>
__global__ __launch_bounds__(256, 2) void k_elem_ins4_em(ElemArgs a, const double* __restrict__ ops, TriLines ln,
                                                                    double* eres, EdgeArgs e, double* eout, int eblk) {
    if ((int)blockIdx.x < eblk) {
        edge_ins_body<4, double, true>(e, eout, blockIdx.x * 256 + threadIdx.x);
        return;
    }
    elem_ins4_body<FULL>(a, ops, ln, eres, eblk);
}

// FP32 (the inner solve of the defect correction): the same residual in single precision
// on v_mfma_f32_16x16x4f32; its operator pack permutes the output rows of Ir/Is so that
// register s of lane group q again holds mode 4s + q
// EDGES: the first eblk blocks are the boundary edges, as in k_elem_ins_em.  At p = 4 their
// body costs registers (104 bytes a lane in scratch against 44 in the full residual, 174
// registers against 124 in the inviscid one; 255 x 255: 70 -> 81 us and 30 -> 36 us); launches
// without it take the edges from k_edge_ins32_em (OWN_EDGES says when).
template <int P, bool FULL, bool EDGES>
__global__ __launch_bounds__(256, 2) void k_elem_ins32_em(ElemArgs32 a, float* eres, EdgeArgsT<float> e, float* eout,
                                                          int eblk) {
    if constexpr (EDGES)
        if ((int)blockIdx.x < eblk) {
            edge_ins_body<P, float, true>(e, eout, blockIdx.x * 256 + threadIdx.x);
            return;
        }
    elem_ins_body<float, P, FULL, true>(a, eres, eblk);
}

template <int P>
__global__ __launch_bounds__(256) void k_edge_ins32_em(EdgeArgsT<float> e, float* eout) {
    edge_ins_body<P, float, true>(e, eout, blockIdx.x * 256 + threadIdx.x);
}

// Element Jacobians of a batch: every (element, column) pair is an entry of one launch,
// its residual and difference formed in the lanes that hold it; 16 neighbouring lanes
// write 16 neighbouring columns of a row of K.  4 000 elements at p = 4 (180 000 entries):
// 0.2 ms, against 46 perturb / residual / collect launches per colour, 10.6 ms.
template <int P, bool FULL>
__global__ __launch_bounds__(256, P == 4 ? 1 : 2) void k_elem_ins_jac(ElemArgs a) {
    elem_ins_body<double, P, FULL, false, false, true>(a);
}

// the curved elements (order[begin:end), a.crv per entry) in element-major form: a
// launch of its own after the straight elements' launch, over the few elements that
// own a curved boundary side
template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_ins_em_curved(ElemArgs a, double* eres) {
    elem_ins_body<double, P, FULL, true, true>(a, eres);
}

template <int P, bool FULL>
__global__ __launch_bounds__(256) void k_elem_ins32_em_curved(ElemArgs32 a, float* eres) {
    elem_ins_body<float, P, FULL, true, true>(a, eres);
}

// lftog of the element-major vertex and side modes (tri_hp/nstage.cpp:21-82): one lane
// per (vertex, variable), then one per (side, mode, variable).  Each sum starts from
// keep * res_r and adds the elements' (beta lf_re, lf_im) in a fixed order (ascending
// element at a vertex, the side's two elements in ascending order), as the first
// colour and the later colours of the scatter do.  FP32 (the defect correction's inner
// solve): the constant source sfac[0] * src enters with the first element, as on the
// scatter's first visit.
// summed: the elements' first entry already is lf_im + beta lf_re.  The boundary-edge
// results follow the elements (eout, written by the element launch's edge
// blocks): a vertex adds its edges' end entries in list order, a boundary side its own.
template <typename T>
struct GatherArgsT {
    int npnt, nseg, sm, sm0, bm;
    const int* vt_ptr;
    const int* vt_tri;
    const int* vt_loc;
    const int* st_tri;
    const int* st_loc;
    const T* eres;
    const int* vb_ptr;   // boundary-edge ends at each vertex: 2 * edge + end
    const int* vb_ent;
    const int* sedge;    // first edge of a side in the boundary lists (-1: none) and
    const int* enext;    // the edge's next entry for the same side
    const T* eout;       // (edge, 2 ends then the side modes, NV)
    T* resv;
    T* rrv;
    T* ress;
    T* rrs;
    T keep;
    int full, summed;
    const double* srcv;  // defect source, may be null
    const double* srcs;
    const double* sfac;
};

template <typename T, int NVn>
__device__ __forceinline__ void gather_sum(const GatherArgsT<T>& a, const T* e, int n, T sign, T& acc, T& accr) {
    const T li = sign * e[n];
    if (a.full) {
        const T lr = sign * e[NVn + n];
        accr += lr;
        acc = (a.summed ? acc : acc + lr) + li;
    } else {
        acc = acc + li;
    }
}

template <typename T, int NVn>
__global__ __launch_bounds__(256) void k_gather_vs(GatherArgsT<T> a) {
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nvl = (long)a.npnt * NVn;
    const T keep = a.keep;
    const int ne = a.sm + 2;  // entries of a boundary edge
    const int rec = a.full ? 2 * NVn : NVn;  // inviscid stages: records of the imaginary part only
    if (g < nvl) {
        const int v = (int)(g / NVn), n = (int)(g - (long)v * NVn);
        const T r0 = keep == T(0) ? T(0) : keep * a.rrv[g];
        T acc = r0, accr = r0;
        for (int k = a.vt_ptr[v]; k < a.vt_ptr[v + 1]; ++k) {
            gather_sum<T, NVn>(a, a.eres + ((long)a.vt_tri[k] * a.bm + a.vt_loc[k]) * rec, n, T(1), acc, accr);
            if (k == a.vt_ptr[v] && a.srcv) acc = acc + T(a.srcv[g] * a.sfac[0]);
        }
        for (int k = a.vb_ptr[v]; k < a.vb_ptr[v + 1]; ++k) {
            const int ent = a.vb_ent[k];
            acc += a.eout[((long)(ent >> 1) * ne + (ent & 1)) * NVn + n];
        }
        if (a.full || keep != T(1)) a.rrv[g] = accr;
        a.resv[g] = acc;
        return;
    }
    const long h = g - nvl;
    const long per = (long)a.sm * NVn;
    if (h >= (long)a.nseg * per) return;
    const int s = (int)(h / per);
    const int r = (int)(h - (long)s * per);
    const int m = r / NVn, n = r - m * NVn;
    const long o = ((long)s * a.sm0 + m) * NVn + n;
    const T r0 = keep == T(0) ? T(0) : keep * a.rrs[o];
    T acc = r0, accr = r0;
    bool first = true;
    for (int slot = 0; slot < 2; ++slot) {
        const int t = a.st_tri[2 * s + slot];
        if (t < 0) continue;
        // st_loc bit 2: the element is a periodic partner's, whose side runs the other
        // way: its odd modes change sign in this side's frame
        const int sl = a.st_loc[2 * s + slot];
        const int mode = 3 + (sl & 3) * a.sm + m;
        gather_sum<T, NVn>(a, a.eres + ((long)t * a.bm + mode) * rec, n, ((sl & 4) && (m & 1)) ? T(-1) : T(1),
                              acc, accr);
        if (first && a.srcs) acc = acc + T(a.srcs[o] * a.sfac[0]);
        first = false;
    }
    for (int ed = a.sedge[s]; ed >= 0; ed = a.enext[ed]) acc += a.eout[((long)ed * ne + 2 + m) * NVn + n];
    if (a.full || keep != T(1)) a.rrs[o] = accr;
    a.ress[o] = acc;
}

// p = 1 element residual on the vector ALU, one thread per element (mesh order), the
// element-major output of k_elem_ins_em (at p = 1, eres[(t*3 + k)*2*NV + n]).  At p = 1
// the 16 x 16 x 4 MFMA tiles are
// mostly padding (4 Gauss points, 3 modes: 80 matrix instructions per 16 elements for
// about 1.2 kflop of work per element), so the residual is written out as scalar
// loops over the dense operators (uniform across the wave: scalar loads).  The same
// sequence as elem_ins_body: proj, inviscid fluxes, intgrtrs (tri_hp/ins/rsdl.cpp:
// 262-294); derivatives, viscous tensor, strong residual, tau and stabilisation,
// intgrtrs of the real part (:296-426).
// Dense p = 1 operators: P, Pr, Ps [4][3] | Ir, Is [3][4] | Dr, Ds [4][4]
constexpr int OP1_P = 0, OP1_PR = 12, OP1_PS = 24, OP1_IR = 36, OP1_IS = 48, OP1_DR = 60, OP1_DS = 76, OP1_SIZE = 92;

template <bool FULL>
__global__ __launch_bounds__(256) void k_elem_ins1_valu(ElemArgs a, const double* __restrict__ op,
                                                        double* __restrict__ eres, EdgeArgs e,
                                                        double* __restrict__ eout, int egrid) {
    if ((int)blockIdx.x >= egrid) {
        edge_ins_body<1, double, true>(e, eout, e.begin + ((int)blockIdx.x - egrid) * (int)blockDim.x + (int)threadIdx.x);
        return;
    }
    const int t = a.begin + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= a.end) return;
    constexpr int G = 4, M = 3;
    int vtx[3];
    double x[3], y[3], b[NV][M];
#pragma unroll
    for (int k = 0; k < 3; ++k) vtx[k] = a.tri_pnt[3 * t + k];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        x[k] = a.pnts[2 * vtx[k]];
        y[k] = a.pnts[2 * vtx[k] + 1];
#pragma unroll
        for (int n = 0; n < NV; ++n) b[n][k] = a.ugv[vtx[k] * NV + n];
    }
    const double l00 = 0.5 * (x[2] - x[1]), l01 = 0.5 * (x[0] - x[1]);
    const double l10 = 0.5 * (y[2] - y[1]), l11 = 0.5 * (y[0] - y[1]);
    double U[G], V[G], Pp[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        double u = 0.0, v = 0.0, pr = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const double w = op[OP1_P + g * M + m];
            u += w * b[0][m]; v += w * b[1][m]; pr += w * b[2][m];
        }
        U[g] = u; V[g] = v; Pp[g] = pr;
    }
    const double rho = a.rho;
    double C0[G], C1[G], A00[G], A01[G], A10[G], A11[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const double fx = rho * U[g], fy = rho * V[g];
        const double c0 = +l11 * fx - l01 * fy;
        const double c1 = -l10 * fx + l00 * fy;
        C0[g] = c0; C1[g] = c1;
        A00[g] = U[g] * c0 + l11 * Pp[g];
        A01[g] = U[g] * c1 - l10 * Pp[g];
        A10[g] = V[g] * c0 - l01 * Pp[g];
        A11[g] = V[g] * c1 + l00 * Pp[g];
    }
    double LI[NV][M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const double ar = op[OP1_IR + m * G + g], as = op[OP1_IS + m * G + g];
            s0 += ar * A00[g] + as * A01[g];
            s1 += ar * A10[g] + as * A11[g];
            s2 += ar * C0[g] + as * C1[g];
        }
        LI[0][m] = s0; LI[1][m] = s1; LI[2][m] = s2;
    }
    double* o = eres + (size_t)t * M * (FULL ? 2 * NV : NV);
    if constexpr (FULL) {
        double Ur[G], Us[G], Vr[G], Vs[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            double c1 = 0.0, c2 = 0.0, c3 = 0.0, c4 = 0.0;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const double ar = op[OP1_PR + g * M + m], as = op[OP1_PS + g * M + m];
                c1 += ar * b[0][m]; c2 += as * b[0][m];
                c3 += ar * b[1][m]; c4 += as * b[1][m];
            }
            Ur[g] = c1; Us[g] = c2; Vr[g] = c3; Vs[g] = c4;
        }
        const double cjcb = l00 * l11 - l10 * l01;
        const double cjcbi = a.mu / cjcb;
        const double v0000 = -cjcbi * (2.0 * l11 * l11 + l01 * l01);
        const double v0011 = -cjcbi * (2.0 * l10 * l10 + l00 * l00);
        const double v0001 = cjcbi * (2.0 * l11 * l10 + l01 * l00);
        const double v1100 = -cjcbi * (l11 * l11 + 2.0 * l01 * l01);
        const double v1111 = -cjcbi * (l10 * l10 + 2.0 * l00 * l00);
        const double v1101 = cjcbi * (l11 * l10 + 2.0 * l01 * l00);
        const double v0100 = cjcbi * l01 * l11;
        const double v0111 = cjcbi * l00 * l10;
        const double v0101 = -cjcbi * l01 * l10;
        const double v0110 = -cjcbi * l00 * l11;
        double F00[G], F01[G], F10[G], F11[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const double ur = Ur[g], us = Us[g], vr = Vr[g], vs = Vs[g];
            F00[g] = v0000 * ur + v0100 * vr + v0001 * us + v0101 * vs;
            F01[g] = v0001 * ur + v0110 * vr + v0011 * us + v0111 * vs;
            F10[g] = v0100 * ur + v1100 * vr + v0110 * us + v1101 * vs;
            F11[g] = v0101 * ur + v1101 * vr + v0111 * us + v1111 * vs;
            A00[g] += F00[g]; A01[g] += F01[g]; A10[g] += F10[g]; A11[g] += F11[g];
        }
        double R0[G], R1[G], R2[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            double r0 = 0.0, r1 = 0.0, r2 = 0.0;
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const double dr = op[OP1_DR + g * G + h], ds = op[OP1_DS + g * G + h];
                r0 += dr * A00[h] + ds * A01[h];
                r1 += dr * A10[h] + ds * A11[h];
                r2 += dr * C0[h] + ds * C1[h];
            }
            R0[g] = r0; R1[g] = r1; R2[g] = r2;
        }
        const double dx1 = x[0] - x[2], dy1 = y[0] - y[2], dx2 = x[1] - x[0], dy2 = y[1] - y[0];
        const double ar2 = dx1 * dy2 - dy1 * dx2;
        const double perim = sqrt(dx1 * dx1 + dy1 * dy1) + sqrt(dx2 * dx2 + dy2 * dy2) +
                             sqrt((dx1 + dx2) * (dx1 + dx2) + (dy1 + dy2) * (dy1 + dy2));
        const double h = (ar2 / perim) / (0.25 * 2 * 2);
        const double nu = a.mu / rho;
        const double gv = 2.0 * nu / h;
        const double gvis = gv * gv;
        const double tfac = a.adis * h / cjcb;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const double u = U[g], v = V[g];
            const double qq = u * u + v * v;
            double gam = 3.0 * qq + gvis;
            if (a.mu == 0.0) gam = fmax(gam, 0.1);
            const double tau0 = tfac / sqrt(gam);
            const double tau2 = sqrt(qq) * tau0;
            const double t0 = tau0 * R0[g], t1 = tau0 * R1[g], t2 = tau2 * R2[g];
            F00[g] -= (l11 * (2.0 * u) - l01 * v) * t0 - l01 * u * t1 + l11 * t2;
            F01[g] -= (-l10 * (2.0 * u) + l00 * v) * t0 + l00 * u * t1 - l10 * t2;
            F10[g] -= +l11 * v * t0 + (l11 * u - l01 * (2.0 * v)) * t1 - l01 * t2;
            F11[g] -= -l10 * v * t0 + (-l10 * u + l00 * (2.0 * v)) * t1 + l00 * t2;
            C0[g] = -(l11 * t0 - l01 * t1);
            C1[g] = -(-l10 * t0 + l00 * t1);
        }
        const double bt = a.beta;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const double ar = op[OP1_IR + m * G + g], as = op[OP1_IS + m * G + g];
                s0 += ar * F00[g] + as * F01[g];
                s1 += ar * F10[g] + as * F11[g];
                s2 += ar * C0[g] + as * C1[g];
            }
            double* om = o + m * (2 * NV);
            om[0] = LI[0][m]; om[1] = LI[1][m]; om[2] = LI[2][m];
            om[NV + 0] = s0 * bt; om[NV + 1] = s1 * bt; om[NV + 2] = s2 * bt;
        }
    } else {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            double* om = o + m * NV;
            om[0] = LI[0][m]; om[1] = LI[1][m]; om[2] = LI[2][m];
        }
    }
}

// ---------------------------------------------------------------------------------
// XCD-aware block index: launches use a multiple of 8 blocks; consecutive hardware
// blocks go round-robin to the 8 XCDs, so XCD x is given the contiguous logical
// range [x * per, (x + 1) * per) and neighbouring entities share one L2
__device__ __forceinline__ int xcd_block() {
    const int per = gridDim.x >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

// setup_preconditioner, element part (tri_hp/ins/setup_preconditioner.cpp:33-219,
// diagonal branch, REFINED_WAY, straight elements, steady)
struct SetupArgs {
    const double* pnts;
    const int* tri_pnt;
    const int* tri_seg;
    const int* tri_sgn;
    const double* ugv;
    const double* ugs;
    const double* ugi;
    const double* Pmat;  // G x tm
    double* tprcn;
    int* err;
    int ntri, p, sm, im, tm, G, sm0, im0;
    double rho, mu, adis;
    // curved elements (k_setup_elem_curved): list, coordinate side modes per entry
    // (the layout of ElemArgsT::crv), dense d/dr and d/ds projections (G x tm)
    const int* clist;
    int ncurv;
    const double* crv;
    const double* PRmat;
    const double* PSmat;
};

template <int P>
__global__ __launch_bounds__(128) void k_setup_elem(SetupArgs a) {
    constexpr int TM = Dims<P>::TM, SM = Dims<P>::SM, G = Dims<P>::G;
    const int t = xcd_block() * blockDim.x + threadIdx.x;
    if (t >= a.ntri) return;
    int vtx[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) vtx[k] = a.tri_pnt[3 * t + k];
    double uh[2][TM];
#pragma unroll
    for (int k = 0; k < TM; ++k) {
        int off;
        double sg = 1.0;
        const double* src;
        if (k < 3) { off = vtx[k] * NV; src = a.ugv; }
        else if (k < 3 * P) {
            const int i = (k - 3) / SM, m = (k - 3) - i * SM;
            const int sgn = a.tri_sgn[3 * t + i];
            sg = ((m & 1) && sgn < 0) ? -1.0 : 1.0;
            off = (a.tri_seg[3 * t + i] * a.sm0 + m) * NV;
            src = a.ugs;
        } else { off = (t * a.im0 + (k - 3 * P)) * NV; src = a.ugi; }
        uh[0][k] = sg * src[off];
        uh[1][k] = sg * src[off + 1];
    }
    double qmax = 0.0;
    for (int g = 0; g < G; ++g) {
        double u = 0.0, v = 0.0;
#pragma unroll
        for (int k = 0; k < TM; ++k) {
            const double pv = a.Pmat[g * TM + k];
            u += pv * uh[0][k];
            v += pv * uh[1][k];
        }
        const double q = u * u + v * v;
        qmax = (qmax > q) ? qmax : q;  // MAX of sys/param.h, as the reference
    }
    const double X[3] = {a.pnts[2 * vtx[0]], a.pnts[2 * vtx[1]], a.pnts[2 * vtx[2]]};
    const double Y[3] = {a.pnts[2 * vtx[0] + 1], a.pnts[2 * vtx[1] + 1], a.pnts[2 * vtx[2] + 1]};
    const double dx1 = X[0] - X[2], dy1 = Y[0] - Y[2], dx2 = X[1] - X[0], dy2 = Y[1] - Y[0];
    double jcb = 0.25 * (dx1 * dy2 - dy1 * dx2);
    double hmax = 0.0;
    for (int j = 0; j < 3; ++j) {
        const int j1 = (j + 1) % 3;
        const double hh = (X[j] - X[j1]) * (X[j] - X[j1]) + (Y[j] - Y[j1]) * (Y[j] - Y[j1]);
        hmax = hh > hmax ? hh : hmax;
    }
    hmax = sqrt(hmax);
    const double pf = 0.25 * (a.p + 1) * (a.p + 1);
    const double h = 4. * jcb / (pf * hmax);
    hmax = hmax / pf;
    if (!(h > 0.0) || qmax != qmax) {
        atomicOr(a.err, 1);
        a.tprcn[3 * t + 0] = a.tprcn[3 * t + 1] = a.tprcn[3 * t + 2] = 1.0;
        return;
    }
    const double nu = a.mu / a.rho;
    double gam = 3.0 * qmax + (2. * nu / hmax) * (2. * nu / hmax);
    if (a.mu == 0.0) gam = fmax(gam, 0.1);
    const double qs = sqrt(qmax);
    const double lam1 = qs + sqrt(qmax + gam);
    jcb *= 2. * nu * (1. / (hmax * hmax) + 1. / (h * h)) + 3 * lam1 / h;
    a.tprcn[3 * t + 0] = a.rho * jcb;
    a.tprcn[3 * t + 1] = a.rho * jcb;
    a.tprcn[3 * t + 2] = jcb / gam;
}

// the curved branch of the same (tri_hp/ins/setup_preconditioner.cpp:44-90) for the
// elements clist[0:ncurv), after k_setup_elem: h from the smallest Jacobian over the
// Gauss points and hmax from the longest projected side tangent, both through the
// coordinate derivatives at every point; tprcn overwritten
template <int P>
__global__ __launch_bounds__(64) void k_setup_elem_curved(SetupArgs a) {
    constexpr int TM = Dims<P>::TM, SM = Dims<P>::SM, BM = Dims<P>::BM, G = Dims<P>::G;
    const int ci = blockIdx.x * blockDim.x + threadIdx.x;
    if (ci >= a.ncurv) return;
    const int t = a.clist[ci];
    int vtx[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) vtx[k] = a.tri_pnt[3 * t + k];
    double uh[2][TM], cx[BM], cy[BM];
#pragma unroll
    for (int k = 0; k < TM; ++k) {
        int off;
        double sg = 1.0;
        const double* src;
        if (k < 3) { off = vtx[k] * NV; src = a.ugv; }
        else if (k < BM) {
            const int i = (k - 3) / SM, m = (k - 3) - i * SM;
            const int sgn = a.tri_sgn[3 * t + i];
            sg = ((m & 1) && sgn < 0) ? -1.0 : 1.0;
            off = (a.tri_seg[3 * t + i] * a.sm0 + m) * NV;
            src = a.ugs;
        } else { off = (t * a.im0 + (k - BM)) * NV; src = a.ugi; }
        uh[0][k] = sg * src[off];
        uh[1][k] = sg * src[off + 1];
    }
    const double X[3] = {a.pnts[2 * vtx[0]], a.pnts[2 * vtx[1]], a.pnts[2 * vtx[2]]};
    const double Y[3] = {a.pnts[2 * vtx[0] + 1], a.pnts[2 * vtx[1] + 1], a.pnts[2 * vtx[2] + 1]};
    // coordinate modes relative to vertex 1 (crdtocht, tri_hp/gtol.cpp:204-245)
    cx[0] = X[0] - X[1]; cy[0] = Y[0] - Y[1];
    cx[1] = 0.0; cy[1] = 0.0;
    cx[2] = X[2] - X[1]; cy[2] = Y[2] - Y[1];
#pragma unroll
    for (int k = 3; k < BM; ++k) {
        const int i = (k - 3) / SM, m = (k - 3) - i * SM;
        cx[k] = a.crv[(((size_t)ci * 3 + i) * a.sm0 + m) * 2];
        cy[k] = a.crv[(((size_t)ci * 3 + i) * a.sm0 + m) * 2 + 1];
    }
    const double dx1 = X[0] - X[2], dy1 = Y[0] - Y[2], dx2 = X[1] - X[0], dy2 = Y[1] - Y[0];
    double jcb = 0.25 * (dx1 * dy2 - dy1 * dx2);
    double jcbmin = jcb, hmax = 0.0, qmax = 0.0;
    for (int g = 0; g < G; ++g) {
        double u = 0.0, v = 0.0, xr = 0.0, xs = 0.0, yr = 0.0, ys = 0.0;
#pragma unroll
        for (int k = 0; k < TM; ++k) {
            const double pv = a.Pmat[g * TM + k];
            u += pv * uh[0][k];
            v += pv * uh[1][k];
        }
#pragma unroll
        for (int k = 0; k < BM; ++k) {
            const double pr = a.PRmat[g * TM + k], ps = a.PSmat[g * TM + k];
            xr += pr * cx[k]; xs += ps * cx[k];
            yr += pr * cy[k]; ys += ps * cy[k];
        }
        jcbmin = fmin(jcbmin, xr * ys - yr * xs);
        double hh = xr * xr + yr * yr;
        hmax = hh > hmax ? hh : hmax;
        hh = xs * xs + ys * ys;
        hmax = hh > hmax ? hh : hmax;
        hh = (xs - xr) * (xs - xr) + (ys - yr) * (ys - yr);
        hmax = hh > hmax ? hh : hmax;
        const double q = u * u + v * v;
        qmax = (qmax > q) ? qmax : q;
    }
    hmax = 2. * sqrt(hmax);
    const double pf = 0.25 * (a.p + 1) * (a.p + 1);
    const double h = 4. * jcbmin / (pf * hmax);
    hmax = hmax / pf;
    if (!(h > 0.0) || qmax != qmax) {
        atomicOr(a.err, 1);
        a.tprcn[3 * t + 0] = a.tprcn[3 * t + 1] = a.tprcn[3 * t + 2] = 1.0;
        return;
    }
    const double nu = a.mu / a.rho;
    double gam = 3.0 * qmax + (2. * nu / hmax) * (2. * nu / hmax);
    if (a.mu == 0.0) gam = fmax(gam, 0.1);
    const double qs = sqrt(qmax);
    const double lam1 = qs + sqrt(qmax + gam);
    jcb *= 2. * nu * (1. / (hmax * hmax) + 1. / (h * h)) + 3 * lam1 / h;
    a.tprcn[3 * t + 0] = a.rho * jcb;
    a.tprcn[3 * t + 1] = a.rho * jcb;
    a.tprcn[3 * t + 2] = jcb / gam;
}

// vprcn = 1/(vdiag * sum of incident tprcn) (setup_preconditioner.cpp:213-219 and
// tri_hp/setup_preconditioner.cpp:68-76); incident elements in ascending order
__global__ void k_setup_vrtx(int npnt, const int* ptr, const int* tri, const double* tprcn, double* vprcn, double vdiag) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= npnt) return;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int k = ptr[v]; k < ptr[v + 1]; ++k) {
        const int t = tri[k];
        s0 += tprcn[3 * t]; s1 += tprcn[3 * t + 1]; s2 += tprcn[3 * t + 2];
    }
    vprcn[3 * v] = 1.0 / (vdiag * s0);
    vprcn[3 * v + 1] = 1.0 / (vdiag * s1);
    vprcn[3 * v + 2] = 1.0 / (vdiag * s2);
}

__global__ void k_setup_side(int nseg, const int* st_tri, const double* tprcn, double* sprcn) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nseg) return;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int k = 0; k < 2; ++k) {
        const int t = st_tri[2 * s + k];
        if (t < 0) continue;
        a0 += tprcn[3 * t]; a1 += tprcn[3 * t + 1]; a2 += tprcn[3 * t + 2];
    }
    sprcn[3 * s] = 1.0 / a0; sprcn[3 * s + 1] = 1.0 / a1; sprcn[3 * s + 2] = 1.0 / a2;
}

// ---------------------------------------------------------------------------------
// periodic boundaries.  The reference keeps a partial residual on each copy of a
// periodic vertex or side and averages the preconditioned values across the pair
// (tri_hp/setup_preconditioner.cpp:24-36, 171-176, 255-258, 331-334 with the comm of
// tri_mesh/tri_boundary.h:113-148), with the preconditioner sums averaged too, which
// equals assembling the pair as one set of unknowns.  Here every copy holds the
// assembled values: the vertex residual of each copy is summed over the group after
// the residual (k_periodic_combine), the side and vertex sweeps read the union of the
// copies' adjacency, and the state copies are kept equal (k_periodic_sync).
// Vertex groups: copies pg_v[pg_ptr[g]:pg_ptr[g+1]] (ascending); one lane per (group, n).
template <typename T, int NVn>
__global__ void k_periodic_combine(int ngrp, const int* __restrict__ ptr, const int* __restrict__ pv, T* res) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngrp * NVn) return;
    const int grp = g / NVn, n = g - grp * NVn;
    T sum = T(0);
    for (int k = ptr[grp]; k < ptr[grp + 1]; ++k) sum += res[pv[k] * NVn + n];
    for (int k = ptr[grp]; k < ptr[grp + 1]; ++k) res[pv[k] * NVn + n] = sum;
}

// r += fl32(sfac[0] * src): the FP32 inner solve's constant source on the vertices of a
// periodic mesh, added after the copies are summed
__global__ void k_add_src32(long n, const double* __restrict__ src, const double* __restrict__ sfac, float* r) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) r[i] = r[i] + float(src[i] * sfac[0]);
}

// state copies from the first copy of each vertex group and from side a of each pair
// (side b = o^m side a); one lane per (group, n), then per (pair, mode, n)
template <typename T, int NVn>
__global__ void k_periodic_sync(int ngrp, const int* __restrict__ ptr, const int* __restrict__ pv, int npair,
                                const int* __restrict__ sa, const int* __restrict__ sb, const int* __restrict__ so,
                                int sm, int sm0, T* v, T* sd) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < ngrp * NVn) {
        const int grp = g / NVn, n = g - grp * NVn;
        const T x = v[pv[ptr[grp]] * NVn + n];
        for (int k = ptr[grp] + 1; k < ptr[grp + 1]; ++k) v[pv[k] * NVn + n] = x;
        return;
    }
    const int h = g - ngrp * NVn;
    if (h >= npair * sm * NVn) return;
    const int pr = h / (sm * NVn), r = h - pr * (sm * NVn), m = r / NVn, n = r - m * NVn;
    const T x = sd[((long)sa[pr] * sm0 + m) * NVn + n];
    sd[((long)sb[pr] * sm0 + m) * NVn + n] = (so[pr] < 0 && (m & 1)) ? -x : x;
}

// ---------------------------------------------------------------------------------
// minvrt, tri_hp/setup_preconditioner.cpp:102-373 (diagonal preconditioner)
template <typename T>
struct MinvArgsT {
    const int* tri_pnt;
    const int* tri_seg;
    const int* tri_sgn;
    const int* vs_ptr;
    const int* vs_side;
    const int* vs_end;
    const int* vt_ptr;
    const int* vt_tri;
    const int* vt_loc;
    const int* st_tri;
    const int* st_loc;
    const unsigned char* vess;
    const unsigned char* sess;
    T* resv;
    T* ress;
    T* resi;
    const T* vprcn;
    const T* sprcn;
    // element scalings of the side rows (side assembly couplings) and of the interior
    // rows; both are tprcn for the analytic preconditioner, the learned one scales them
    // by mode type
    const T* tprcn_s;
    const T* tprcn_i;
    const T* lump;  // sfmv | ifmb | vfms | sdiag | sfms | bfmi | idiag
    int npnt, nseg, ntri, sm, im, bm, sm0, im0;
    int o_sfmv, o_ifmb, o_vfms, o_sdiag, o_sfms, o_bfmi, o_idiag;
    // p = 4: work planes of the side sweeps, one per mode, (mode, side, variable).  A sweep
    // reads one mode of four neighbouring sides: from the (side, mode, variable) records it
    // would fetch all three
    T* pl;
    // the solved side and interior values go to ress / resi (always, unless another stage
    // of the same update overwrites them unread)
    int store;
    // fused stage update ug = ug0 - cfa * res (tri_hp/nstage.cpp:387-409) when ug != null
    T* ugv;
    T* ugs;
    T* ugi;
    const T* ug0v;
    const T* ug0s;
    const T* ug0i;
    T cfa;
};


// The minvrt sweeps run one lane per (entity, variable): the diagonal preconditioner
// never couples the variables, so lane (e, n) carries variable n of entity e through
// every subtraction in the same order as the per-entity loop.  Consecutive lanes then
// read consecutive doubles of the (entity, mode, variable) records, and the gathers of
// neighbouring records touch a third of the cache lines a lane-per-entity sweep does.
template <typename T, int NVn>
__device__ __forceinline__ bool minv_lane(int count, int& e, int& n) {
    const long g = (long)xcd_block() * blockDim.x + threadIdx.x;
    e = (int)(g / NVn);
    n = (int)(g - (long)e * NVn);
    return e < count;
}

// vertices: subtract side and interior couplings (:110-135), scale (:151-152),
// vertex Dirichlet (:179-183)
template <typename T, int P, int NVn>
__global__ __launch_bounds__(256) void k_minv_vrtx(MinvArgsT<T> a) {
    constexpr int SM = Dims<P>::SM, IM = Dims<P>::IM;
    int v, n;
    if (!minv_lane<T, NVn>(a.npnt, v, n)) return;
    T r = a.resv[v * NVn + n];
    if constexpr (SM > 0) {
        for (int k = a.vs_ptr[v]; k < a.vs_ptr[v + 1]; ++k) {
            const int s = a.vs_side[k], i = a.vs_end[k];
#pragma unroll
            for (int m = 0; m < SM; ++m) r -= a.lump[a.o_sfmv + i * SM + m] * a.ress[(s * a.sm0 + m) * NVn + n];
        }
        if constexpr (IM > 0)
            for (int k = a.vt_ptr[v]; k < a.vt_ptr[v + 1]; ++k) {
                const int t = a.vt_tri[k], i = a.vt_loc[k];
#pragma unroll
                for (int m = 0; m < IM; ++m) r -= a.lump[a.o_ifmb + i * IM + m] * a.resi[(t * a.im0 + m) * NVn + n];
            }
    }
    // every load before the first store: the stores could alias later loads
    const T x = (a.vess[v] >> n) & 1 ? T(0) : r * a.vprcn[v * NVn + n];
    const T u0 = a.ugv ? a.ug0v[v * NVn + n] : T(0);
    a.resv[v * NVn + n] = x;
    if (a.ugv) a.ugv[v * NVn + n] = u0 - a.cfa * x;
}

// p = 1 stage on the vertices, one lane per (vertex, variable): the lftog sums of the
// element-major element and edge results in a fixed order (tri_hp/nstage.cpp:21-82,
// hp_boundary.cpp:973-1049), the multigrid source (nstage.cpp:76-82, 113-128) and,
// with `ug` set, the vertex minvrt (setup_preconditioner.cpp:151-152, 179-183) and the
// stage update ug = ug0 - cfa * res (nstage.cpp:387-409).  At p = 1 every mode is a
// vertex mode, so this is the whole stage after the element residual.
struct VStageArgs {
    int npnt;
    const int* vt_ptr;
    const int* vt_tri;
    const int* vt_loc;
    const int* vb_ptr;  // boundary-edge endpoints at each vertex: entries 2*idx + k of eout
    const int* vb_ent;
    const double* eres;  // (ntri, 3, 2, NV), (ntri, 3, NV) without the real part
    const double* eout;  // (neseg, 2, NV)
    double* resv;
    double* rrv;
    double keep;
    int full;           // the stage evaluates the real part (beta > 0)
    int mg;             // 0 none, 1 res += dres, 2 dres = fadd r0 - res, res += dres
    double* dres;
    const double* r0;
    double fadd;
    const unsigned char* vess;
    const double* vprcn;
    double* ug;         // null: residual only
    double* ug0;
    double cfa;
    int save_u0;        // first stage: ug0 = ug
};

template <int NVn>
__global__ __launch_bounds__(256) void k_vstage1(VStageArgs a) {
    int v, n;
    if (!minv_lane<double, NVn>(a.npnt, v, n)) return;
    const long o = (long)v * NVn + n;
    const double keep = a.keep;
    const double r0 = (keep == 0.0 || !(a.full || keep != 0.0)) ? 0.0 : keep * a.rrv[o];
    double acc = r0, accr = r0;
    for (int k = a.vt_ptr[v]; k < a.vt_ptr[v + 1]; ++k) {
        const double* e = a.eres + ((long)a.vt_tri[k] * 3 + a.vt_loc[k]) * (a.full ? 2 * NVn : NVn);
        const double li = e[n];
        if (a.full) {
            const double lr = e[NVn + n];
            accr += lr;
            acc = (acc + lr) + li;
        } else {
            acc = acc + li;
        }
    }
    for (int k = a.vb_ptr[v]; k < a.vb_ptr[v + 1]; ++k) acc += a.eout[(long)a.vb_ent[k] * NVn + n];
    if (a.mg == 1) {
        acc += a.dres[o];
    } else if (a.mg == 2) {
        const double d = a.fadd * a.r0[o] - acc;
        a.dres[o] = d;
        acc += d;
    }
    if (a.full || keep != 1.0) a.rrv[o] = accr;
    if (a.ug) {
        const double x = (a.vess[v] >> n) & 1 ? 0.0 : acc * a.vprcn[o];
        const double u = a.save_u0 ? a.ug[o] : a.ug0[o];
        if (a.save_u0) a.ug0[o] = u;
        a.resv[o] = x;
        a.ug[o] = u - a.cfa * x;
    } else {
        a.resv[o] = acc;
    }
}

// solved value of side mode `mode` from its residual r (:245-267, :331-343): scale, sdirichlet
template <typename T, int NVn>
__device__ __forceinline__ T side_solved(const MinvArgsT<T>& a, int s, int mode, int n, T r) {
    if ((a.sess[s] >> n) & 1) return T(0);
    return r * (a.sprcn[s * NVn + n] * a.lump[a.o_sdiag + mode]);
}

// sides: subtract interior couplings (:137-148), then the vertex solution (:192-214), and
// solve mode 0 (p = 2: the only one, stored with its stage update)
template <typename T, int P, int NVn>
__global__ __launch_bounds__(256) void k_minv_side(MinvArgsT<T> a) {
    constexpr int SM = Dims<P>::SM, IM = Dims<P>::IM;
    int s, n;
    if (!minv_lane<T, NVn>(a.nseg, s, n)) return;
    T r[SM];
#pragma unroll
    for (int m = 0; m < SM; ++m) r[m] = a.ress[(s * a.sm0 + m) * NVn + n];
    if constexpr (IM > 0)
        for (int k = 0; k < 2; ++k) {
            const int t = a.st_tri[2 * s + k];
            if (t < 0) continue;
            // a periodic partner's element (st_loc bit 2) sees this side reversed
            const int sl = a.st_loc[2 * s + k], i = sl & 3;
            const int sgn = (sl & 4) ? -a.tri_sgn[3 * t + i] : a.tri_sgn[3 * t + i];
            T bi[IM];
#pragma unroll
            for (int m = 0; m < IM; ++m) bi[m] = a.resi[(t * a.im0 + m) * NVn + n];
            T ms = T(1);
#pragma unroll
            for (int j = 0; j < SM; ++j) {
#pragma unroll
                for (int m = 0; m < IM; ++m) {
                    const T c = ms * a.lump[a.o_ifmb + (3 + i * SM + j) * IM + m];
                    r[j] -= c * bi[m];
                }
                ms *= sgn;
            }
        }
    for (int k = 0; k < 2; ++k) {
        const int t = a.st_tri[2 * s + k];
        if (t < 0) continue;
        const int sl = a.st_loc[2 * s + k], i = sl & 3;
        const int sgn = (sl & 4) ? -a.tri_sgn[3 * t + i] : a.tri_sgn[3 * t + i];
        const T tp = a.tprcn_s[NVn * t + n];
        T uh[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) uh[j] = a.resv[a.tri_pnt[3 * t + (i + j) % 3] * NVn + n] * tp;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            T ms = T(1);
#pragma unroll
            for (int m = 0; m < SM; ++m) {
                r[m] -= ms * a.lump[a.o_vfms + j * SM + m] * uh[j];
                ms *= sgn;
            }
        }
    }
    const T x0 = side_solved<T, NVn>(a, s, 0, n, r[0]);
    if constexpr (SM == 1) {
        const int ix = s * a.sm0 * NVn + n;
        const T u0 = a.ugs ? a.ug0s[ix] : T(0);
        if (a.store) a.ress[ix] = x0;
        if (a.ugs) a.ugs[ix] = u0 - a.cfa * x0;
    } else {
        a.pl[s * NVn + n] = x0;
#pragma unroll
        for (int m = 1; m < SM; ++m) a.pl[((long)m * a.nseg + s) * NVn + n] = r[m];
    }
}

// remove solved side mode MODE from the higher modes (:244-328) and solve mode MODE + 1.
// The last mode's sweep also stores the solved values and the stage update: 64 sides per
// block go through LDS so that the (side, mode, variable) records are read and written as
// one contiguous stream.  512 x 512, p = 4, FP64: 35 us for mode 0, 63 us for the last
template <typename T, int P, int MODE, int NVn>
__global__ __launch_bounds__(64 * NVn) void k_minv_sub(MinvArgsT<T> a) {
    constexpr int SM = Dims<P>::SM;
    constexpr bool LAST = MODE == SM - 2;
    __shared__ T sx[LAST ? 64 * SM * NVn : 1];
    const int blk = xcd_block();
    const int ls = threadIdx.x / NVn, n = threadIdx.x - ls * NVn;
    const int s = blk * 64 + ls;
    if (s < a.nseg) {
        T r[SM];
#pragma unroll
        for (int m = MODE + 1; m < SM; ++m) r[m] = a.pl[((long)m * a.nseg + s) * NVn + n];
        for (int k = 0; k < 2; ++k) {
            const int t = a.st_tri[2 * s + k];
            if (t < 0) continue;
            const int sl = a.st_loc[2 * s + k], i = sl & 3;
            const T tp = a.tprcn_s[NVn * t + n];
            T uh[3];
            int sign[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int jj = (i + j) % 3;
                const int sj = a.tri_seg[3 * t + jj];
                sign[j] = a.tri_sgn[3 * t + jj];
                const T sg = (MODE % 2) ? T(sign[j]) : T(1);
                uh[j] = sg * a.pl[((long)MODE * a.nseg + sj) * NVn + n] * tp;
            }
            // into this side's frame: a periodic partner's element (st_loc bit 2) has its
            // own copy of the side running the other way
            const int s0 = (sl & 4) ? -sign[0] : sign[0];
            T ms = ((MODE + 1) % 2) ? T(s0) : T(1);
#pragma unroll
            for (int m = MODE + 1; m < SM; ++m) {
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const T c = ms * a.lump[a.o_sfms + (MODE * SM + m) * 3 + j];
                    r[m] -= c * uh[j];
                }
                ms *= s0;
            }
        }
        const T x = side_solved<T, NVn>(a, s, MODE + 1, n, r[MODE + 1]);
        a.pl[((long)(MODE + 1) * a.nseg + s) * NVn + n] = x;
        if constexpr (LAST) {
#pragma unroll
            for (int m = 0; m < SM - 1; ++m) sx[(ls * SM + m) * NVn + n] = a.pl[((long)m * a.nseg + s) * NVn + n];
            sx[(ls * SM + SM - 1) * NVn + n] = x;
        } else {
#pragma unroll
            for (int m = MODE + 2; m < SM; ++m) a.pl[((long)m * a.nseg + s) * NVn + n] = r[m];
        }
    }
    if constexpr (LAST) {
        __syncthreads();
        const long o = (long)blk * 64 * SM * NVn;
        const int cnt = min(64, a.nseg - blk * 64) * SM * NVn;
        for (int k = threadIdx.x; k < cnt; k += 64 * NVn) {
            const T u0 = a.ugs ? a.ug0s[o + k] : T(0);
            if (a.store) a.ress[o + k] = sx[k];
            if (a.ugs) a.ugs[o + k] = u0 - a.cfa * sx[k];
        }
    }
}

// interiors: banded solve with the literal DPBTRSNU2 indexing (utilities/myblas.c:91-122),
// divide by tprcn, subtract the boundary solution through bfmi (:347-370)
template <typename T, int P, int NVn>
__global__ __launch_bounds__(256) void k_minv_int(MinvArgsT<T> a) {
    constexpr int SM = Dims<P>::SM, IM = Dims<P>::IM, BM = Dims<P>::BM;
    int t, n;
    if (!minv_lane<T, NVn>(a.ntri, t, n)) return;
    T b[IM];
#pragma unroll
    for (int k = 0; k < IM; ++k) b[k] = a.resi[(t * a.im0 + k) * NVn + n];
    const T* ab = a.lump + a.o_idiag;  // stride 2, ofdg 1
#pragma unroll
    for (int i = 0; i < IM; ++i) {
        const int frst = (1 - i > 0 ? 1 - i : 0), ba = -frst;
#pragma unroll
        for (int j = frst; j < 1; ++j) b[i] -= ab[i * 2 + j] * b[ba + j];
        b[i] /= ab[i * 2 + 1];
    }
#pragma unroll
    for (int i = IM - 1; i >= 0; --i) {
        b[i] /= ab[i * 2 + 1];
        const int frst = (1 - i > 0 ? 1 - i : 0), ba = -frst;
#pragma unroll
        for (int j = frst; j < 1; ++j) b[ba + j] -= ab[i * 2 + j] * b[i];
    }
    T uh[BM];
#pragma unroll
    for (int i = 0; i < 3; ++i) uh[i] = a.resv[a.tri_pnt[3 * t + i] * NVn + n];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int sd = a.tri_seg[3 * t + i], sgn = a.tri_sgn[3 * t + i];
        T ms = T(1);
#pragma unroll
        for (int m = 0; m < SM; ++m) {
            uh[3 + i * SM + m] = ms * a.pl[((long)m * a.nseg + sd) * NVn + n];
            ms *= sgn;
        }
    }
    const T tp = a.tprcn_i[NVn * t + n];
#pragma unroll
    for (int k = 0; k < IM; ++k) {
        b[k] /= tp;
#pragma unroll
        for (int i = 0; i < BM; ++i) b[k] -= a.lump[a.o_bfmi + i * IM + k] * uh[i];
    }
    T u0[IM];
#pragma unroll
    for (int k = 0; k < IM; ++k) u0[k] = a.ugi ? a.ug0i[(t * a.im0 + k) * NVn + n] : T(0);
#pragma unroll
    for (int k = 0; k < IM; ++k) {
        const int ix = (t * a.im0 + k) * NVn + n;
        if (a.store) a.resi[ix] = b[k];
        if (a.ugi) a.ugi[ix] = u0[k] - a.cfa * b[k];
    }
}

// ---------------------------------------------------------------------------------
// max |x| over (nent, nm active modes of mstride, NV), per variable, into out[NV] as
// ordered bit patterns of non-negative doubles; mask (optional) skips essential entries
template <int NVn>
__global__ void k_absmax(long nent, int nm, int mstride, const double* __restrict__ x,
                         const unsigned char* __restrict__ mask, unsigned long long* out) {
    __shared__ unsigned long long red[NVn][256];
    unsigned long long mx[NVn] = {};
    const long span = (long)nm;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < nent * span; k += (long)gridDim.x * blockDim.x) {
        const long ent = k / span, m = k - ent * span;
        const unsigned msk = mask ? mask[ent] : 0u;
        for (int n = 0; n < NVn; ++n) {
            if ((msk >> n) & 1) continue;
            const double v = fabs(x[(ent * mstride + m) * NVn + n]);
            const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
            mx[n] = bits > mx[n] ? bits : mx[n];
        }
    }
    for (int n = 0; n < NVn; ++n) red[n][threadIdx.x] = mx[n];
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st)
            for (int n = 0; n < NVn; ++n) {
                const unsigned long long o = red[n][threadIdx.x + st];
                red[n][threadIdx.x] = o > red[n][threadIdx.x] ? o : red[n][threadIdx.x];
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int n = 0; n < NVn; ++n) atomicMax(&out[n], red[n][0]);
}

// ---------------------------------------------------------------------------------
// h-multigrid transfers between a mesh and its coarse neighbour (tri_hp/movco.cpp:41-102,
// tri_hp/movfin.cpp:16-82), vertex values only (coarse levels run at p = 1)

// res0(coarse v) = sum over the fine vertices held by triangles of v, in ascending fine
// order, of weight x fine residual (ccnnct transposed into a gather)
template <int NVn>
__global__ void k_hrestrict(int nc, const int* __restrict__ ptr, const int* __restrict__ fidx,
                            const double* __restrict__ wt, const double* __restrict__ fres, double* __restrict__ res0) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nc) return;
    double s[NVn];
#pragma unroll
    for (int n = 0; n < NVn; ++n) s[n] = 0.0;
    for (int k = ptr[v]; k < ptr[v + 1]; ++k) {
        const int i = fidx[k];
        const double w = wt[k];
#pragma unroll
        for (int n = 0; n < NVn; ++n) s[n] += w * fres[i * NVn + n];
    }
#pragma unroll
    for (int n = 0; n < NVn; ++n) res0[v * NVn + n] = s[n];
}

// coarse ug = fine ug interpolated at the coarse vertices (fcnnct); vug_frst = ug
template <int NVn>
__global__ void k_hinterp(int nc, const int* __restrict__ fv, const double* __restrict__ w,
                          const double* __restrict__ fug, double* __restrict__ ug, double* __restrict__ vug) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nc) return;
    double s[NVn];
#pragma unroll
    for (int n = 0; n < NVn; ++n) s[n] = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int f = fv[3 * v + j];
        const double ww = w[3 * v + j];
#pragma unroll
        for (int n = 0; n < NVn; ++n) s[n] += ww * fug[f * NVn + n];
    }
#pragma unroll
    for (int n = 0; n < NVn; ++n) { ug[v * NVn + n] = s[n]; vug[v * NVn + n] = s[n]; }
}

// vug_frst -= ug: minus the coarse correction
__global__ void k_hcorr(long n, double* __restrict__ vug, const double* __restrict__ ug) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) vug[k] -= ug[k];
}

// fine res = interpolated coarse correction (ccnnct), fine ug += res
template <int NVn>
__global__ void k_hprolong(int nf, const int* __restrict__ cv, const double* __restrict__ w,
                           const double* __restrict__ vug, double* __restrict__ fres, double* __restrict__ fug) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nf) return;
    double r[NVn];
#pragma unroll
    for (int n = 0; n < NVn; ++n) r[n] = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int c = cv[3 * i + j];
        const double ww = w[3 * i + j];
#pragma unroll
        for (int n = 0; n < NVn; ++n) r[n] -= ww * vug[c * NVn + n];
    }
#pragma unroll
    for (int n = 0; n < NVn; ++n) {
        fres[i * NVn + n] = r[n];
        fug[i * NVn + n] += r[n];
    }
}

// MFMA lane-layout self test: D = A(16x4) * B(4x16) with the layout the element
// kernel assumes; out[lane*4+i] = D element held by (lane, register i)
__global__ void k_mfma_probe(const double* A, const double* B, double* out) {
    const int l = threadIdx.x;
    const double av = A[(l & 15) * 4 + (l >> 4)];
    const double bv = B[(l >> 4) * 16 + (l & 15)];
    d4 c = {0.0, 0.0, 0.0, 0.0};
    c = mfma(av, bv, c);
    for (int i = 0; i < 4; ++i) out[l * 4 + i] = c[i];
}

// same probe for v_mfma_f32_16x16x4f32 (FP32 inputs, FP32 accumulation)
__global__ void k_mfma_probe_f32(const float* A, const float* B, float* out) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int l = threadIdx.x;
    const float av = A[(l & 15) * 4 + (l >> 4)];
    const float bv = B[(l >> 4) * 16 + (l & 15)];
    f4 c = {0.f, 0.f, 0.f, 0.f};
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv, c, 0, 0, 0);
    for (int i = 0; i < 4; ++i) out[l * 4 + i] = c[i];
}

// explicit instantiations used by the host context
template __global__ void k_elem_ins<1, true>(ElemArgs);
template __global__ void k_elem_ins<1, false>(ElemArgs);
template __global__ void k_elem_ins<2, true>(ElemArgs);
template __global__ void k_elem_ins<2, false>(ElemArgs);
template __global__ void k_elem_ins<4, true>(ElemArgs);
template __global__ void k_elem_ins<4, false>(ElemArgs);


// grid-stride 16-byte copy (reference kernel for traffic counters)
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, long long n16) {
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n16; k += (long long)gridDim.x * blockDim.x)
        dst[k] = src[k];
}

}  // namespace hpg
