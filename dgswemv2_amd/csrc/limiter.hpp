// Cockburn-Shu slope limiter and trouble check, per element (FP64 arithmetic in every form).
//
// The arithmetic is FP64 and not contracted in any form (each function turns contraction off, whatever the
// translation unit's setting), so a limiter decision depends only on the state.  The one place with fused
// multiply-adds, written out, is the write-back of an FP32 state (sl_decide<true>).
//
// CS_slope_limiter_serial (problem_slope_limiter/swe_CS_sl_serial.hpp:9-23) as kernels:
//   barycentres         - of the linear part (slope_limiting_prepare_element_kernel,
//                         swe_CS_slope_limiter.hpp:8-20), written by the stage kernel, or by the limiter's
//                         first launch where the state may change in between (a stage in two calls);
//   sl_check_element    - the KXRCF-style indicator I of check_trouble (swe_trouble_check.hpp:13-104),
//                         written as the seed set;
//   sl_spread_seeds     - the six neighbour-dilation passes (:106-115), by the limit kernel;
//   sl_limit_core       - slope_limiting_kernel (swe_CS_slope_limiter.hpp:88-189) reading the
//                         neighbours' barycentres, then the NaN scan.
// The limit pass never reads the troubled flags: they are an output.
#pragma once

#include "engine.hpp"

namespace rkdg {

template <typename Real>
struct LimiterArgs {
    int ne, nedge;
    Real* q;                  // [3][ND][ne] state of the new stage, limited in place
    const Real* bath;         // [ND][ne]
    const int* nb;            // [3][ne] face slots (as in StageArgs)
    const int* edge;
    const uint32_t* meta;
    const Real* egeom;        // [3][nedge]
    const uint8_t* wet;       // [ne] flags after wetting-drying
    const double* bath_vrtx;  // [3][ne]
    const int* neighbor;      // [3][ne] by local face, -1 on a boundary
    const double* median;     // [6][ne]
    const double* alpha;      // [6][ne]
    const double* rsq;        // [3][ne]
    const double* len;        // [3][ne]
    const double* radius;     // [ne]
    const double* bath_bc;    // [ne]
    double* baryctr;          // [3][ne]
    uint8_t* seed;            // [ne] elements with I > 1
    uint8_t* troubled;        // [ne]
    uint8_t* limited;         // [3][ne]
    double g, M, nu;
    int p;
    int nan_check;
    unsigned long long* nan_key;
    unsigned long long stage_key;  // step * nstages + stage (the stage alone with step_ctr)
    const unsigned long long* step_ctr;  // device step counter of an ensemble, or null
    int key_ns;
};

// BARY: writes the barycentres too.  Only a wet element can be a seed; its own data and then its
// neighbours' are read together (two round trips; 190 B an element at p = 1 in FP64: 500k triangles
// 24.7 -> 16.6 us, 33k triangles 5.5 -> 4 us).
template <typename Real, int P, bool BARY>
RKDG_HD RKDG_FORCE_INLINE inline void sl_check_element(const LimiterArgs<Real>& L, const FaceTables<Real>& FT, int e) {
#pragma clang fp contract(off)
    using C = ConstTables<Real, P>;
    constexpr int ND = Sizes<P>::ND, NE = Sizes<P>::NE;
    const int ne = L.ne;
    uint8_t seed = 0;
    if (L.wet[e]) {
        double ze[ND], qx[ND], bath[ND], vrtx[3], len[3];
        int nb[3], ed[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) nb[s] = ldc(L.nb, ne, s, e), ed[s] = ldc(L.edge, ne, s, e);
        const uint32_t meta = ldc(L.meta, ne, 0, e);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            ze[d] = (double)ldc(L.q, ne, d, e);
            qx[d] = (double)ldc(L.q, ne, ND + d, e);
            bath[d] = (double)ldc(L.bath, ne, d, e);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) vrtx[k] = ldc(L.bath_vrtx, ne, k, e), len[k] = ldc(L.len, ne, k, e);
        const double r = ldc(L.radius, ne, 0, e);
        if constexpr (BARY) {
            stc(L.baryctr, ne, 0, e, barycentre(ze[0], ze[1], ze[2]));
            stc(L.baryctr, ne, 1, e, barycentre(qx[0], qx[1], qx[2]));
            stc(L.baryctr, ne, 2, e,
                barycentre((double)ldc(L.q, ne, 2 * ND, e), (double)ldc(L.q, ne, 2 * ND + 1, e), (double)ldc(L.q, ne, 2 * ND + 2, e)));
        }
        // check_trouble: interfaces of this element in (in, ex) order = face slots
        double I = 0.0, perimeter = 0.0;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            if (nb[s] < 0) continue;
            double zn[ND], bn[ND];
#pragma unroll
            for (int d = 0; d < ND; ++d) zn[d] = (double)ldc(L.q, ne, d, nb[s]), bn[d] = (double)ldc(L.bath, ne, d, nb[s]);
            const double nx = (double)ldc(L.egeom, L.nedge, 0, ed[s]), ny = (double)ldc(L.egeom, L.nedge, 1, ed[s]);
            const double sJ = (double)ldc(L.egeom, L.nedge, 2, ed[s]);
            const int f = (meta >> (4 * s)) & 3, fn = (meta >> (4 * s + 2)) & 3;
            const bool is_in = e < nb[s];
            const double onx = is_in ? nx : -nx, ony = is_in ? ny : -ny;
            const Real* pf = FT.phie + f * ND * NE;
            const Real* pn = FT.phie + fn * ND * NE;
            // sum of modes times the face's basis values at point g (the constant mode's value is one)
            auto trace = [](const double* m, const Real* ph) {
                double t = m[0];
#pragma unroll
                for (int d = 1; d < ND; ++d) t = t + m[d] * (double)ph[d];
                return t;
            };
            double ze_o[NE], integ = 0.0;
#pragma unroll
            for (int g = 0; g < NE; ++g) {
                ze_o[g] = trace(ze, pf + g * ND);
                // quirk kept: q_n is formed from rows 0/1 of q (ze, qx) (swe_trouble_check.hpp:29-35)
                const double qn = onx * ze_o[g] + ony * trace(qx, pf + g * ND);
                const double w = (double)C::we[0][g] * sJ;
                integ = (g == 0) ? qn * w : integ + qn * w;
            }
            if (integ < 0.0) {
                double hi = 0.0;
#pragma unroll
                for (int g = 0; g < NE; ++g) {
                    double hd = ze_o[g] + trace(bath, pf + g * ND);
                    hd -= trace(zn, pn + (NE - 1 - g) * ND) + trace(bn, pn + (NE - 1 - g) * ND);
                    const double w = (double)C::we[0][g] * sJ;
                    hi = (g == 0) ? hd * w : hi + hd * w;
                }
                perimeter += f == 0 ? len[0] : (f == 1 ? len[1] : len[2]);
                I += (hi < 0 ? -hi : hi);
            }
        }
        if (perimeter != 0.0) {
            double v[3], h_norm = 0.0;
            to_vertices(ze, v);
#pragma unroll
            for (int k = 0; k < 3; ++k) h_norm = rmax(h_norm, v[k] + vrtx[k]);
            using std::pow;
            I /= ((P == 1 ? r : pow(r, (L.p + 1.0) / 2.0)) * perimeter * h_norm);
            seed = I > 1.0 ? 1 : 0;
        }
    }
    L.seed[e] = seed;
    L.troubled[e] = seed;
}

RKDG_HD inline void mv3(const double A[3][3], const double* x, double* y) {
#pragma clang fp contract(off)
    for (int i = 0; i < 3; ++i) y[i] = (A[i][0] * x[0] + A[i][1] * x[1]) + A[i][2] * x[2];
}

// What slope_limiting_kernel decides for one element: may act (element and neighbours wet), the
// variables it writes back, and the 2-norm of each variable's vertex-value change.
struct SlOutcome {
    bool ok;
    unsigned mask;
    double del[3];
};

// What the decision reads of a wet element with wet neighbours: vertex values, barycentre values of
// the element and (or its own, across a boundary) its neighbours, and its geometry.
struct SlInput {
    double ql[3][3], bc[3], bcn[3][3];
    double med[3][2], alpha[3][2], rsq[3], bath_bc;
};
RKDG_HD RKDG_FORCE_INLINE inline void sl_geometry(const double* median, const double* alpha, const double* rsq, const double* bath_bc, int ne,
                                                  int e, SlInput& in) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        in.med[k][0] = ldc(median, ne, 2 * k, e), in.med[k][1] = ldc(median, ne, 2 * k + 1, e);
        in.alpha[k][0] = ldc(alpha, ne, 2 * k, e), in.alpha[k][1] = ldc(alpha, ne, 2 * k + 1, e);
        in.rsq[k] = ldc(rsq, ne, k, e);
    }
    in.bath_bc = ldc(bath_bc, ne, 0, e);
}

// The limiting step: out.mask and out.del, and the linear modes m of the written-back variables.
template <bool FUSED>
RKDG_HD RKDG_FORCE_INLINE inline void sl_decide(const SlInput& in, double g, double M, double nu, SlOutcome& out, double m[3][3]) {
#pragma clang fp contract(off)
    const double(&ql)[3][3] = in.ql;
    const double(&bc)[3] = in.bc;
    const double(&bcn)[3][3] = in.bcn;
    using std::copysign;
    using std::fabs;
    using std::signbit;
    using std::sqrt;
    const double chi[3][3] = {{0.0, 0.5, 0.5}, {0.5, 0.0, 0.5}, {0.5, 0.5, 0.0}};
    const double h = bc[0] + in.bath_bc;
    const double u = bc[1] / h, v = bc[2] / h;
    const double c = sqrt(g * h);
    const Quotient<double> by_2c(2 * c);
    double delta[3][3];  // [var][bound]
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const int e1 = b, e2 = (b + 1) % 3;
        const double mx = in.med[b][0], my = in.med[b][1];
        // R and invR along the median (problem_jacobian/swe_jacobian.hpp:462-480, 531-550)
        const double R[3][3] = {{1.0, 0.0, 1.0}, {u - c * mx, -my, u + c * mx}, {v - c * my, mx, v + c * my}};
        const double un = u * mx + v * my;
        const double iR[3][3] = {{by_2c(c + un), by_2c(-mx), by_2c(-my)},
                                 {u * my - v * mx, -my, mx},
                                 {by_2c(c - un), by_2c(mx), by_2c(my)}};
        double qm[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) qm[k] = (ql[k][0] * chi[0][b] + ql[k][1] * chi[1][b]) + ql[k][2] * chi[2][b];
        double wm[3], w0[3], w1[3], w2[3];
        mv3(iR, qm, wm);
        mv3(iR, bc, w0);
        mv3(iR, bcn[e1], w1);
        mv3(iR, bcn[e2], w2);
        const double Mr2 = M * in.rsq[b];
        double dc[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double wt = wm[k] - w0[k];
            const double wd = in.alpha[b][0] * (w1[k] - w0[k]) + in.alpha[b][1] * (w2[k] - w0[k]);
            if (fabs(wt) <= Mr2)
                dc[k] = wt;
            else if (signbit(wt) == signbit(wd))
                dc[k] = copysign(1.0, wt) * rmin(fabs(wt), fabs(nu * wd));
            else
                dc[k] = 0.0;
        }
        double col[3];
        mv3(R, dc, col);
#pragma unroll
        for (int k = 0; k < 3; ++k) delta[k][b] = col[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double sum = 0.0;
#pragma unroll
        for (int b = 0; b < 3; ++b) sum += delta[k][b];
        if (sum != 0.0) {
            double pos = 0.0, neg = 0.0;
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                pos += rmax(0.0, delta[k][b]);
                neg += rmax(0.0, -delta[k][b]);
            }
            const double tp = rmin(1.0, neg / pos);
            const double tn = rmin(1.0, pos / neg);
#pragma unroll
            for (int b = 0; b < 3; ++b) delta[k][b] = tp * rmax(0.0, delta[k][b]) - tn * rmax(0.0, -delta[k][b]);
        }
    }
    const double Tm[3][3] = {{-1.0, 1.0, 1.0}, {1.0, -1.0, 1.0}, {1.0, 1.0, -1.0}};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double qv[3];
#pragma unroll
        for (int vv = 0; vv < 3; ++vv)
            qv[vv] = bc[k] + ((delta[k][0] * Tm[0][vv] + delta[k][1] * Tm[1][vv]) + delta[k][2] * Tm[2][vv]);
        const double d0 = qv[0] - ql[k][0], d1 = qv[1] - ql[k][1], d2 = qv[2] - ql[k][2];
        const double del_norm = sqrt((d0 * d0 + d1 * d1) + d2 * d2);
        const double q_norm = sqrt((ql[k][0] * ql[k][0] + ql[k][1] * ql[k][1]) + ql[k][2] * ql[k][2]);
        out.del[k] = del_norm;
        if (del_norm / q_norm > 1.0e-12) {
            out.mask |= 1u << k;
            // from_vertices, rounded alike in every translation unit (the learned form limits in the gate's);
            // with fused multiply-adds for an FP32 state, as its write-back has always been
            if constexpr (FUSED) {
                m[k][0] = fma(qv[2], 1.0 / 3.0, fma(qv[0], 1.0 / 3.0, qv[1] * (1.0 / 3.0)));
                m[k][1] = fma(qv[2], 1.0 / 3.0, fma(qv[0], -1.0 / 6.0, qv[1] * (-1.0 / 6.0)));
            } else {
                m[k][0] = (qv[0] * (1.0 / 3.0) + qv[1] * (1.0 / 3.0)) + qv[2] * (1.0 / 3.0);
                m[k][1] = (qv[0] * (-1.0 / 6.0) + qv[1] * (-1.0 / 6.0)) + qv[2] * (1.0 / 3.0);
            }
            m[k][2] = (qv[0] * (-1.0 / 2.0) + qv[1] * (1.0 / 2.0)) + qv[2] * 0.0;
        }
    }
}

template <typename Real>
RKDG_HD inline void sl_record_nan(const LimiterArgs<Real>& L, int e) {
    const unsigned long long key = ((L.step_ctr ? *L.step_ctr * (unsigned long long)L.key_ns + L.stage_key : L.stage_key) << 32) | (unsigned long long)(unsigned)e;
#ifdef __HIP_DEVICE_COMPILE__
    atomicMin(L.nan_key, key);
#else
    if (key < *L.nan_key) *L.nan_key = key;
#endif
}

// WRITE: the limiter itself (writes the limited modes, the flags, the NaN scan); otherwise a dry
// run that only reports the decision (the learned indicator's judge and label pass).
//
// Bound by memory (p = 1: 310 B an element, 5.5 TB/s at 500k triangles): the element's own modes, wet
// flag and neighbours are read together, then everything a wet element needs, so a small mesh waits
// for two round trips and a dry one reads no geometry; the NaN scan uses the registers.
template <typename Real, int P, bool WRITE>
RKDG_HD RKDG_FORCE_INLINE inline SlOutcome sl_limit_core(const LimiterArgs<Real>& L, int e) {
#pragma clang fp contract(off)
    constexpr int ND = Sizes<P>::ND;
    const int ne = L.ne;
    SlOutcome out{false, 0u, {0.0, 0.0, 0.0}};
    Real lin[3][3];
    int nbr[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) nbr[k] = ldc(L.neighbor, ne, k, e);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int d = 0; d < 3; ++d) lin[k][d] = ldc(L.q, ne, k * ND + d, e);
    const bool wet = L.wet[e] != 0;
    if (wet) {
        bool wet_neigh = true;
        SlInput in;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int n = nbr[k] >= 0 ? nbr[k] : e;
            wet_neigh = wet_neigh && (L.wet[n] != 0);
#pragma unroll
            for (int v = 0; v < 3; ++v) in.bcn[k][v] = ldc(L.baryctr, ne, v, n);
            in.bc[k] = ldc(L.baryctr, ne, k, e);
        }
        sl_geometry(L.median, L.alpha, L.rsq, L.bath_bc, ne, e, in);
        out.ok = wet_neigh;
        if (wet_neigh) {
            double m[3][3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double lm[3] = {(double)lin[k][0], (double)lin[k][1], (double)lin[k][2]};
                to_vertices(lm, in.ql[k]);
            }
            sl_decide<sizeof(Real) == 4>(in, L.g, L.M, L.nu, out, m);
            if constexpr (WRITE)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (out.mask & (1u << k)) {
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            lin[k][d] = (Real)m[k][d];
                            stc(L.q, ne, k * ND + d, e, lin[k][d]);
                        }
#pragma unroll
                        for (int d = 3; d < ND; ++d) stc(L.q, ne, k * ND + d, e, Real(0.0));
                    }
        }
    }
    if constexpr (!WRITE) return out;
#pragma unroll
    for (int k = 0; k < 3; ++k) L.limited[(size_t)k * ne + e] = (out.mask >> k) & 1;
    if (L.nan_check) {
        bool has_nan = false;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
#pragma unroll
            for (int d = 0; d < 3; ++d) has_nan |= (lin[k][d] != lin[k][d]);
            if (ND > 3 && !((out.mask >> k) & 1))  // a written-back variable's higher modes are zero
#pragma unroll
                for (int d = 3; d < ND; ++d) {
                    const Real x = ldc(L.q, ne, k * ND + d, e);
                    has_nan |= (x != x);
                }
        }
        if (has_nan) sl_record_nan(L, e);
    }
    return out;
}

// Relative size of a write-back for the indicator's labels: the change of each variable's vertex
// values over that variable's physical scale (h_s for ze, h_s sqrt(g h_s) for qx, qy, with
// h_s = max(ze mode 0 + bathymetry at the barycentre, 0.01)); the largest over written-back variables.
template <typename Real>
RKDG_HD inline double sl_change(const LimiterArgs<Real>& L, const SlOutcome& o, int e, double h_floor) {
#pragma clang fp contract(off)
    double h = (double)L.q[e] + L.bath_bc[e];
    h = h > h_floor ? h : h_floor;
    using std::sqrt;
    const double sq = h * sqrt(L.g * h);
    double r = 0.0;
    for (int k = 0; k < 3; ++k)
        if (o.mask & (1u << k)) {
            const double c = o.del[k] / (k == 0 ? h : sq);
            r = c > r ? c : r;
        }
    return r;
}

}  // namespace rkdg
