// Device-side numerics of the FastS structured NS iteration for CDNA4 (gfx950).
//
// Every function reproduces the per-cell floating-point operation order of the reference
// kernel it cites, so that with floating-point contraction disabled the results are bit-for-bit
// those of the reference FastS kernels.  Layout: structure of arrays, i fastest, ghost layers
// included (Fast/FastS/FastS/formule_param.h: inddm).
#pragma once
#include <hip/hip_runtime.h>

namespace fm {

// Everything a kernel needs about one zone, passed by value as a kernel argument.
struct KZ {
    int ni, nj, nk;        // interior cells (IJKV)
    int nit, njt, nkt;     // storage cells per direction (NIJK)
    int nf, nfk;           // ghost layers
    long nd;               // NDIMDX
    long incj, inck;
    int typ;               // ITYPZONE: 0 3dfull, 2 3dcart
    long mi, mj, mk;       // metric strides (NIJK_MTR)
    int mf, mfk;
    long ndm;              // NDIMDX_MTR
    int xi, xj, xf, xfk;   // vertex grid (NIJK_XYZ)
    int kflu, slope, iflow, itypcp, dtloc, rk, nssiter, sensortype;
    // cache blocks of the reference's flux and gradient passes in j and k (CACHEBLCKJ/K and
    // the block counts max(1, n / size) of crsdm_scater.for; one block in i): they fix the
    // order in which a cell receives the fluxes of its max faces
    int cbj, cbk, nbj, nbk;
    double dtc, gam, cv, roinf, pinf, vinf, tinf, prandt, xmul0, temp0, cs, cfl, psiroe, wig_amp;
    // fields
    const double* x; const double* y; const double* z;
    double* ti; double* tj; double* tk; double* vol;
    double* xmut; double* drodm; double* coe; double* wig;
};

__host__ __device__ __forceinline__ long IDX(const KZ& z, int i, int j, int k) {
    return (long)(i + z.nf - 1) + (long)(j + z.nf - 1) * z.incj + (long)(k + z.nfk - 1) * z.inck;
}
__device__ __forceinline__ long MTR(const KZ& z, int i, int j, int k) {
    return (long)(i + z.mf - 1) * z.mi + (long)(j + z.mf - 1) * z.mj + (long)(k + z.mfk - 1) * z.mk;
}
__device__ __forceinline__ long XYZ(const KZ& z, int i, int j, int k) {
    return (long)(i + z.xf - 1) + (long)(j + z.xf - 1) * z.xi + (long)(k + z.xfk - 1) * (long)z.xi * z.xj;
}
// Fortran MAX/MIN as compiled by the reference: a > b ? a : b
__device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double dsign(double a, double b) { return copysign(fabs(a), b); }

// the value lane L + DI holds (DPP wave shifts; the last lanes of the wave get their own value)
template <int DI>
__device__ __forceinline__ double from_lane(double v) {
    static_assert(DI >= -1 && DI <= 1, "shift of a wave");
    if (DI == 0) return v;
    constexpr int ctl = DI > 0 ? 0x130 : 0x138;   // wave_shl:1 / wave_shr:1
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, ctl, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), ctl, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// A barrier that makes the LDS accesses of every wave before it visible after it.  Only LDS is ordered: a
// __syncthreads() may also wait for the wave's global stores and loads in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Constants of the flux template header (template_FluxAndBalance.for:100-190)
struct FluxConst {
    double gam, rgp, gam1, gam3, psiroe, tmin_1, c1, c2, c3, opt0, c4, c5, c6, cvisq, wig_cte;
    double tc[3], s[3], volinv;   // 3dcart metric
};

__device__ __forceinline__ FluxConst flux_const(const KZ& z) {
    FluxConst f;
    f.gam = z.gam;
    f.rgp = z.cv * (f.gam - 1.);
    f.gam1 = f.gam / (f.gam - 1.);
    f.gam3 = f.gam1 / z.prandt * f.rgp;
    f.psiroe = z.psiroe;
    f.tmin_1 = 100. / z.tinf;
    f.c1 = 0.02 * z.vinf;
    f.c2 = 0.02 / (z.vinf * z.roinf);
    f.c3 = -2.;
    f.opt0 = (double)z.sensortype;
    f.wig_cte = z.wig_amp;
    f.c6 = 1. / 6.; f.c4 = 5. * f.c6; f.c5 = 2. * f.c6; f.c6 = -1. * f.c6;
    f.cvisq = 1. / 3;
    if (z.typ == 2) {
        f.tc[0] = z.ti[0]; f.tc[1] = z.tj[0]; f.tc[2] = z.tk[0];
        f.s[0] = fabs(f.tc[0]); f.s[1] = fabs(f.tc[1]); f.s[2] = fabs(f.tc[2]);
        f.volinv = 0.5 / z.vol[0];
    } else {
        f.tc[0] = f.tc[1] = f.tc[2] = 0.; f.s[0] = f.s[1] = f.s[2] = 0.; f.volinv = 0.;
    }
    return f;
}

// Where a face flux reads its stencil from: values of the cell (DI, DJ, DK) away from the flux's own
// cell, and the face vectors and volumes at the same place of the metric grid.  MemCell reads all of
// them from memory.
struct MemCell {
    const KZ& z;
    const double* __restrict__ rop;
    long l, lt;
    __device__ __forceinline__ MemCell(const KZ& z_, const double* rop_, long l_, long lt_) : z(z_), rop(rop_), l(l_), lt(lt_) {}
    template <int DI, int DJ, int DK> __device__ __forceinline__ long at() const { return l + DI + DJ * z.incj + DK * z.inck; }
    template <int DI, int DJ, int DK> __device__ __forceinline__ double q(int e) const { return rop[at<DI, DJ, DK>() + e * z.nd]; }
    template <int DI, int DJ, int DK> __device__ __forceinline__ double mu() const { return z.xmut[at<DI, DJ, DK>()]; }
    __device__ __forceinline__ double wig(int d) const { return z.wig[l + d * z.nd]; }
    template <int DI, int DJ, int DK> __device__ __forceinline__ double met(const double* __restrict__ t, int m) const {
        return t[lt + DI * z.mi + DJ * z.mj + DK * z.mk + m * z.ndm];
    }
};

// the same with the neighbour's distance added last, as an index that is one for all lanes: k_residual on 3dcart,
// where the one sum of indexes spills 8 to 18 registers of the laminar kernels (128^3 AUSM+(P) 251 us; so 209),
// and SENSEUR Euler on 3dfull (128^3 225 us; so 203).  The others on 3dfull are 5 to 15 % faster with the sum.
struct MemCellApart : MemCell {
    using MemCell::MemCell;
    template <int DI, int DJ, int DK> __device__ __forceinline__ double q(int e) const {
        return (rop + (l + e * z.nd))[DI + DJ * z.incj + DK * z.inck];
    }
};

// value e of the cell M places along direction D (M = 0: the cell itself)
template <int D, int M, typename Cell>
__device__ __forceinline__ double along(const Cell& c, int e) {
    return c.template q<(D == 0 ? M : 0), (D == 1 ? M : 0), (D == 2 ? M : 0)>(e);
}

// MUSCL states (Slope/{o1,o3,minmod}_slope_var.for); qm right, qp left of face (l-inc, l)
template <int SLOPE, int D, typename Cell>
__device__ __forceinline__ void slope_state(const FluxConst& f, const Cell& cell, double qm[5], double qp[5]) {
    if (SLOPE == 1) {
#pragma unroll
        for (int e = 0; e < 5; e++) { qm[e] = along<D, 0>(cell, e); qp[e] = along<D, -1>(cell, e); }
    } else if (SLOPE == 2) {
#pragma unroll
        for (int e = 0; e < 5; e++) {
            double a = along<D, 0>(cell, e), b = along<D, -1>(cell, e);
            double c = along<D, 1>(cell, e), d = along<D, -2>(cell, e);
            qm[e] = f.c4 * a + f.c5 * b + f.c6 * c;
            qp[e] = f.c4 * b + f.c6 * d + f.c5 * a;
        }
    } else {
        double roff = .5 * dmax(0., dmin(along<D, 0>(cell, 4) * f.tmin_1 - .5, 1.));
#pragma unroll
        for (int e = 0; e < 5; e++) {
            double a = along<D, 0>(cell, e), b = along<D, -1>(cell, e);
            double c = along<D, 1>(cell, e), d = along<D, -2>(cell, e);
            double delm = a - b, delp = c - a, delq = b - d;
            double sg = dsign(1., delm);
            double slp = roff * (sg * dmax(0., dmin(fabs(delm), sg * delp)));
            sg = dsign(1., delq);
            double slq = roff * (sg * dmax(0., dmin(fabs(delq), sg * delm)));
            qm[e] = a - slp;
            qp[e] = b + slq;
        }
    }
}

// Inviscid face flux: Roe (etat_roe_GD.for + Vit_ent/fludiffer_*), AUSM+(P)
// (AUSM/fluFaceEuler.for) and SENSEUR (SENSOR/fluFaceEuler.for), 3dcart or 3dfull.
template <int KFLU, bool CART, int D, typename Cell>
__device__ __forceinline__ void inviscid_flux(const FluxConst& f, const Cell& cell, const double tn[3], double sn,
                                              const double qm[5], const double qp[5], double flu[5]) {
    if (KFLU == 5) {
        double gam = f.gam, rgp = f.rgp, gam1 = f.gam1, psiroe = f.psiroe;
        double r1 = qp[0];
        double p1 = r1 * qp[4] * rgp;
        double h1 = gam1 * qp[4] * rgp + .5 * (qp[1] * qp[1] + qp[2] * qp[2] + qp[3] * qp[3]);
        double r2 = qm[0];
        double p2 = r2 * qm[4] * rgp;
        double h2 = gam1 * qm[4] * rgp + .5 * (qm[1] * qm[1] + qm[2] * qm[2] + qm[3] * qm[3]);
        double sp1 = sqrt(r1), sm1 = sqrt(r2);
        double r = sp1 * sm1;
        double r_1 = 1. / (sp1 + sm1);
        double a[3];
        a[0] = (sp1 * qp[1] + sm1 * qm[1]) * r_1;
        a[1] = (sp1 * qp[2] + sm1 * qm[2]) * r_1;
        a[2] = (sp1 * qp[3] + sm1 * qm[3]) * r_1;
        double h = (sp1 * h1 + sm1 * h2) * r_1;
        double q = .5 * (a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
        double c = sqrt((gam - 1.) * fabs(h - q));
        double qn1, qn2;
        if (CART) { qn1 = qp[1 + D] * tn[D]; qn2 = qm[1 + D] * tn[D]; }
        else {
            qn1 = qp[1] * tn[0] + qp[2] * tn[1] + qp[3] * tn[2];
            qn2 = qm[1] * tn[0] + qm[2] * tn[1] + qm[3] * tn[2];
        }
        double du[3] = {(qm[1] - qp[1]) * sn, (qm[2] - qp[2]) * sn, (qm[3] - qp[3]) * sn};
        double dp = p2 - p1;
        double dqn = qn2 - qn1;
        double s_1 = 1. / dmax(sn, 1.e-30);
        double nn[3], qn;
        if (CART) { nn[0] = nn[1] = nn[2] = 0.; nn[D] = tn[D] * s_1; qn = a[D] * nn[D]; }
        else {
            nn[0] = tn[0] * s_1; nn[1] = tn[1] * s_1; nn[2] = tn[2] * s_1;
            qn = a[0] * nn[0] + a[1] * nn[1] + a[2] * nn[2];
        }
        double f1 = qn;
        double f4 = psiroe * (fabs(f1) + c);
        double f2 = .5 + dsign(.5, fabs(f1) - f4);
        double f3 = (f2 - 1.) * (f1 * f1 / f4 + f4) * 0.5 - f2 * fabs(f1);
        f1 = (r2 - r1 - dp / (c * c)) * sn;
        flu[0] = f3 * (f1);
#pragma unroll
        for (int m = 0; m < 3; m++) {
            bool dir = CART ? (m == D) : true;
            flu[1 + m] = f3 * (f1 * a[m] + r * (dir ? du[m] - nn[m] * dqn : du[m]));
        }
        flu[4] = f3 * (f1 * q + r * (a[0] * du[0] + a[1] * du[1] + a[2] * du[2] - qn * dqn));
        f1 = qn + c;
        f2 = .5 + dsign(.5, fabs(f1) - f4);
        f3 = (f2 - 1.) * (f1 * f1 / f4 + f4) * 0.5 - f2 * fabs(f1);
        f1 = (dp + r * c * dqn * s_1) / (2. * c * c) * sn * f3;
        flu[0] = flu[0] + f1;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            bool dir = CART ? (m == D) : true;
            flu[1 + m] = flu[1 + m] + f1 * (dir ? a[m] + nn[m] * c : a[m]);
        }
        flu[4] = flu[4] + f1 * (h + qn * c);
        f1 = qn - c;
        f2 = .5 + dsign(.5, fabs(f1) - f4);
        f3 = (f2 - 1.) * (f1 * f1 / f4 + f4) * 0.5 - f2 * fabs(f1);
        f1 = (dp - r * c * dqn * s_1) / (2. * c * c) * f3 * sn;
        flu[0] = flu[0] + f1;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            bool dir = CART ? (m == D) : true;
            flu[1 + m] = flu[1 + m] + f1 * (dir ? a[m] - nn[m] * c : a[m]);
        }
        flu[4] = flu[4] + f1 * (h - qn * c);
        double rou1 = r1 * qn1, rou2 = r2 * qn2, p1p2 = p1 + p2;
        flu[0] = (flu[0] + rou1 + rou2) * 0.5;
#pragma unroll
        for (int m = 0; m < 3; m++) {
            bool dir = CART ? (m == D) : true;
            flu[1 + m] = dir ? (flu[1 + m] + rou1 * qp[1 + m] + rou2 * qm[1 + m] + tn[m] * p1p2) * 0.5
                             : (flu[1 + m] + rou1 * qp[1 + m] + rou2 * qm[1 + m]) * 0.5;
        }
        flu[4] = (flu[4] + rou1 * h1 + rou2 * h2) * 0.5;
    } else {
        double rgp = f.rgp, gam1 = f.gam1;
        double r1 = qp[0];
        double rou1 = r1 * qp[1], rov1 = r1 * qp[2], row1 = r1 * qp[3];
        double p1 = r1 * qp[4] * rgp;
        double h1 = gam1 * p1 + .5 * (rou1 * qp[1] + rov1 * qp[2] + row1 * qp[3]);
        double r2 = qm[0];
        double rou2 = r2 * qm[1], rov2 = r2 * qm[2], row2 = r2 * qm[3];
        double p2 = r2 * qm[4] * rgp;
        double h2 = gam1 * p2 + .5 * (rou2 * qm[1] + rov2 * qm[2] + row2 * qm[3]);
        double qn1, qn2;
        if (CART) { qn1 = qp[1 + D] * tn[D]; qn2 = qm[1 + D] * tn[D]; }
        else {
            qn1 = qp[1] * tn[0] + qp[2] * tn[1] + qp[3] * tn[2];
            qn2 = qm[1] * tn[0] + qm[2] * tn[1] + qm[3] * tn[2];
        }
        double u, tdu;
        if (KFLU == 1) {
            double c = rgp * f.gam * cell.template q<0, 0, 0>(4);
            double son = sqrt(qn1 * qn1 / c);
            double tam = f.c3 * son + sn;
            double tam1 = dmax(0., tam) * f.c2;
            u = 0.25 * (qn1 + qn2) - tam1 * (p2 - p1);
            tdu = dmax(fabs(u), f.c1 * sn) * f.wig_cte;
        } else {
            double wg = cell.wig(D);
            u = 0.25 * (qn1 + qn2) - f.c2 * sn * (p2 - p1) * (f.opt0 * wg + 1. - f.opt0);
            tdu = dmax(fabs(u), f.c1 * sn) * wg;
        }
        double p1p2 = (p1 + p2) * 0.5;
        double mom1[3] = {rou1, rov1, row1}, mom2[3] = {rou2, rov2, row2};
        flu[0] = u * (r1 + r2) - tdu * (r2 - r1);
#pragma unroll
        for (int m = 0; m < 3; m++) {
            bool dir = CART ? (m == D) : true;
            flu[1 + m] = dir ? u * (mom1[m] + mom2[m]) - tdu * (mom2[m] - mom1[m]) + tn[m] * p1p2
                             : u * (mom1[m] + mom2[m]) - tdu * (mom2[m] - mom1[m]);
        }
        flu[4] = u * (h1 + h2) - tdu * (h2 - h1);
    }
}

// Centred viscous flux on a Cartesian zone (fluvisq_3dcart_{i,j,k}.for)
// gv (optional): the face gradients (u, v, w, T) x (x, y, z) the flux was built from, and the
// face's volinv in gv[12]; components this direction does not form stay as they were
template <int D, typename Cell>
__device__ __forceinline__ void visc_cart(const FluxConst& f, const Cell& cell, double flu[5],
                                          double* gv = nullptr) {
    double tcx = f.tc[0], tcy = f.tc[1], tcz = f.tc[2];
    double xmutvol, xktvol, fv, fv5, f1, f2, f3, f4, f5, f6, div, fvs;
    if constexpr (D == 0) {
        double tix = tcx, tjy = .25 * tcy, tkz = .25 * tcz;
        double gUx, gUy, gUz, gVx, gVy, gWx, gWz, gTx;
        f1 = cell.template q<-1, 0, 0>(1); f2 = cell.template q<0, 0, 0>(1); fvs = f1 + f2;
        f3 = fvs + cell.template q<-1, -1, 0>(1) + cell.template q<0, -1, 0>(1); f4 = fvs + cell.template q<-1, 1, 0>(1) + cell.template q<0, 1, 0>(1);
        f5 = fvs + cell.template q<-1, 0, -1>(1) + cell.template q<0, 0, -1>(1); f6 = fvs + cell.template q<-1, 0, 1>(1) + cell.template q<0, 0, 1>(1);
        gUx = (f2 - f1) * tix; gUy = (f4 - f3) * tjy; gUz = (f6 - f5) * tkz;
        f1 = cell.template q<-1, 0, 0>(2); f2 = cell.template q<0, 0, 0>(2); fvs = f1 + f2;
        f3 = fvs + cell.template q<-1, -1, 0>(2) + cell.template q<0, -1, 0>(2); f4 = fvs + cell.template q<-1, 1, 0>(2) + cell.template q<0, 1, 0>(2);
        gVx = (f2 - f1) * tix; gVy = (f4 - f3) * tjy;
        f1 = cell.template q<-1, 0, 0>(3); f2 = cell.template q<0, 0, 0>(3); fvs = f1 + f2;
        f5 = fvs + cell.template q<-1, 0, -1>(3) + cell.template q<0, 0, -1>(3); f6 = fvs + cell.template q<-1, 0, 1>(3) + cell.template q<0, 0, 1>(3);
        gWx = (f2 - f1) * tix; gWz = (f6 - f5) * tkz;
        f1 = cell.template q<-1, 0, 0>(4); f2 = cell.template q<0, 0, 0>(4);
        gTx = (f2 - f1) * tix;
        div = (gUx + gVy + gWz) * f.cvisq;
        f1 = gUx - div; f2 = gUy + gVx; f3 = gUz + gWx;
        xmutvol = (cell.template mu<0, 0, 0>() + cell.template mu<-1, 0, 0>()) * f.volinv;
        xktvol = xmutvol * f.gam3;
        fv = -(2. * f1 * tcx) * xmutvol; fv5 = fv * (cell.template q<0, 0, 0>(1) + cell.template q<-1, 0, 0>(1)); flu[1] = flu[1] + fv;
        fv = -(f2 * tcx) * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(2) + cell.template q<-1, 0, 0>(2)); flu[2] = flu[2] + fv;
        fv = -(f3 * tcx) * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(3) + cell.template q<-1, 0, 0>(3)); flu[3] = flu[3] + fv;
        fv = fv5 * 0.5 - (gTx * tcx) * xktvol; flu[4] = flu[4] + fv;
        if (gv) {
            gv[0] = gUx; gv[1] = gUy; gv[2] = gUz; gv[3] = gVx; gv[4] = gVy;
            gv[6] = gWx; gv[8] = gWz; gv[9] = gTx;
        }
    } else if constexpr (D == 1) {
        double tiy = tcy, tjz = .25 * tcz, tkx = .25 * tcx;
        double gUx, gUy, gVx, gVy, gVz, gWy, gWz, gTy;
        f1 = cell.template q<0, -1, 0>(1); f2 = cell.template q<0, 0, 0>(1); fvs = f1 + f2;
        f5 = fvs + cell.template q<-1, -1, 0>(1) + cell.template q<-1, 0, 0>(1); f6 = fvs + cell.template q<1, -1, 0>(1) + cell.template q<1, 0, 0>(1);
        gUx = (f6 - f5) * tkx; gUy = (f2 - f1) * tiy;
        f1 = cell.template q<0, -1, 0>(2); f2 = cell.template q<0, 0, 0>(2); fvs = f1 + f2;
        f3 = fvs + cell.template q<0, -1, -1>(2) + cell.template q<0, 0, -1>(2); f4 = fvs + cell.template q<0, -1, 1>(2) + cell.template q<0, 0, 1>(2);
        f5 = fvs + cell.template q<-1, -1, 0>(2) + cell.template q<-1, 0, 0>(2); f6 = fvs + cell.template q<1, -1, 0>(2) + cell.template q<1, 0, 0>(2);
        gVx = (f6 - f5) * tkx; gVy = (f2 - f1) * tiy; gVz = (f4 - f3) * tjz;
        f1 = cell.template q<0, -1, 0>(3); f2 = cell.template q<0, 0, 0>(3); fvs = f1 + f2;
        f3 = fvs + cell.template q<0, -1, -1>(3) + cell.template q<0, 0, -1>(3); f4 = fvs + cell.template q<0, -1, 1>(3) + cell.template q<0, 0, 1>(3);
        gWy = (f2 - f1) * tiy; gWz = (f4 - f3) * tjz;
        f1 = cell.template q<0, -1, 0>(4); f2 = cell.template q<0, 0, 0>(4);
        gTy = (f2 - f1) * tiy;
        div = (gUx + gVy + gWz) * f.cvisq;
        f2 = gUy + gVx; f4 = gVy - div; f5 = gVz + gWy;
        xmutvol = (cell.template mu<0, 0, 0>() + cell.template mu<0, -1, 0>()) * f.volinv;
        xktvol = xmutvol * f.gam3;
        fv = -(f2 * tcy) * xmutvol; fv5 = fv * (cell.template q<0, 0, 0>(1) + cell.template q<0, -1, 0>(1)); flu[1] = flu[1] + fv;
        fv = -(2. * f4 * tcy) * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(2) + cell.template q<0, -1, 0>(2)); flu[2] = flu[2] + fv;
        fv = -(f5 * tcy) * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(3) + cell.template q<0, -1, 0>(3)); flu[3] = flu[3] + fv;
        fv = fv5 * 0.5 - (gTy * tcy) * xktvol; flu[4] = flu[4] + fv;
        if (gv) {
            gv[0] = gUx; gv[1] = gUy; gv[3] = gVx; gv[4] = gVy; gv[5] = gVz;
            gv[7] = gWy; gv[8] = gWz; gv[10] = gTy;
        }
    } else {
        double tiz = tcz, tky = .25 * tcy, tjx = .25 * tcx;
        double gUx, gUz, gVy, gVz, gWx, gWy, gWz, gTz;
        f1 = cell.template q<0, 0, -1>(1); f2 = cell.template q<0, 0, 0>(1); fvs = f1 + f2;
        f3 = fvs + cell.template q<-1, 0, -1>(1) + cell.template q<-1, 0, 0>(1); f4 = fvs + cell.template q<1, 0, -1>(1) + cell.template q<1, 0, 0>(1);
        gUx = (f4 - f3) * tjx; gUz = (f2 - f1) * tiz;
        f1 = cell.template q<0, 0, -1>(2); f2 = cell.template q<0, 0, 0>(2); fvs = f1 + f2;
        f5 = fvs + cell.template q<0, -1, -1>(2) + cell.template q<0, -1, 0>(2); f6 = fvs + cell.template q<0, 1, -1>(2) + cell.template q<0, 1, 0>(2);
        gVy = (f6 - f5) * tky; gVz = (f2 - f1) * tiz;
        f1 = cell.template q<0, 0, -1>(3); f2 = cell.template q<0, 0, 0>(3); fvs = f1 + f2;
        f3 = fvs + cell.template q<-1, 0, -1>(3) + cell.template q<-1, 0, 0>(3); f4 = fvs + cell.template q<1, 0, -1>(3) + cell.template q<1, 0, 0>(3);
        f5 = fvs + cell.template q<0, -1, -1>(3) + cell.template q<0, -1, 0>(3); f6 = fvs + cell.template q<0, 1, -1>(3) + cell.template q<0, 1, 0>(3);
        gWx = (f4 - f3) * tjx; gWy = (f6 - f5) * tky; gWz = (f2 - f1) * tiz;
        f1 = cell.template q<0, 0, -1>(4); f2 = cell.template q<0, 0, 0>(4);
        gTz = (f2 - f1) * tiz;
        div = (gUx + gVy + gWz) * f.cvisq;
        f3 = gUz + gWx; f5 = gVz + gWy; f6 = gWz - div;
        xmutvol = (cell.template mu<0, 0, 0>() + cell.template mu<0, 0, -1>()) * f.volinv;
        xktvol = xmutvol * f.gam3;
        fv = -f3 * tcz * xmutvol; fv5 = fv * (cell.template q<0, 0, 0>(1) + cell.template q<0, 0, -1>(1)); flu[1] = flu[1] + fv;
        fv = -f5 * tcz * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(2) + cell.template q<0, 0, -1>(2)); flu[2] = flu[2] + fv;
        fv = -2. * f6 * tcz * xmutvol; fv5 = fv5 + fv * (cell.template q<0, 0, 0>(3) + cell.template q<0, 0, -1>(3)); flu[3] = flu[3] + fv;
        fv = fv5 * 0.5 - gTz * tcz * xktvol; flu[4] = flu[4] + fv;
        if (gv) {
            gv[0] = gUx; gv[2] = gUz; gv[4] = gVy; gv[5] = gVz;
            gv[6] = gWx; gv[7] = gWy; gv[8] = gWz; gv[11] = gTz;
        }
    }
    if (gv) gv[12] = f.volinv;
}

// Centred viscous flux on a curvilinear zone (fluvisq_3dfull_{i,j,k}.for)
template <int D, typename Cell>
__device__ __forceinline__ void visc_full(const FluxConst& f, const KZ& z, const Cell& cell, const double tn[3],
                                          double flu[5], double* gv = nullptr) {
    // (D, then the two directions after it) the face vectors of the cells on both sides, and the
    // neighbours of the two cells in those directions
    double t0[3], t1[3], u0[3], u1[3], w0[3], w1[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
        const double* ti = z.ti; const double* tj = z.tj; const double* tk = z.tk;
        if constexpr (D == 0) {
            const double a = cell.template met<0, 0, 0>(ti, m);
            t0[m] = .5 * (a + cell.template met<-1, 0, 0>(ti, m));
            t1[m] = .5 * (a + cell.template met<1, 0, 0>(ti, m));
            u0[m] = .125 * (cell.template met<0, 0, 0>(tj, m) + cell.template met<-1, 0, 0>(tj, m));
            u1[m] = .125 * (cell.template met<0, 1, 0>(tj, m) + cell.template met<-1, 1, 0>(tj, m));
            w0[m] = .125 * (cell.template met<0, 0, 0>(tk, m) + cell.template met<-1, 0, 0>(tk, m));
            w1[m] = .125 * (cell.template met<0, 0, 1>(tk, m) + cell.template met<-1, 0, 1>(tk, m));
        } else if constexpr (D == 1) {
            const double a = cell.template met<0, 0, 0>(tj, m);
            t0[m] = .5 * (a + cell.template met<0, -1, 0>(tj, m));
            t1[m] = .5 * (a + cell.template met<0, 1, 0>(tj, m));
            u0[m] = .125 * (cell.template met<0, 0, 0>(tk, m) + cell.template met<0, -1, 0>(tk, m));
            u1[m] = .125 * (cell.template met<0, 0, 1>(tk, m) + cell.template met<0, -1, 1>(tk, m));
            w0[m] = .125 * (cell.template met<0, 0, 0>(ti, m) + cell.template met<0, -1, 0>(ti, m));
            w1[m] = .125 * (cell.template met<1, 0, 0>(ti, m) + cell.template met<1, -1, 0>(ti, m));
        } else {
            const double a = cell.template met<0, 0, 0>(tk, m);
            t0[m] = .5 * (a + cell.template met<0, 0, -1>(tk, m));
            t1[m] = .5 * (a + cell.template met<0, 0, 1>(tk, m));
            u0[m] = .125 * (cell.template met<0, 0, 0>(ti, m) + cell.template met<0, 0, -1>(ti, m));
            u1[m] = .125 * (cell.template met<1, 0, 0>(ti, m) + cell.template met<1, 0, -1>(ti, m));
            w0[m] = .125 * (cell.template met<0, 0, 0>(tj, m) + cell.template met<0, 0, -1>(tj, m));
            w1[m] = .125 * (cell.template met<0, 1, 0>(tj, m) + cell.template met<0, 1, -1>(tj, m));
        }
    }
    // (the 33 face vectors are read and averaged before any state, which keeps both out of scratch)
    __builtin_amdgcn_sched_barrier(0);
    double ql[5], qr[5], g[4][3];
#pragma unroll
    for (int e = 1; e < 5; e++) {
        const double f1 = ql[e] = along<D, -1>(cell, e), f2 = qr[e] = along<D, 0>(cell, e);
        double n3a, n3b, n4a, n4b, n5a, n5b, n6a, n6b;
        if constexpr (D == 0) {
            n3a = cell.template q<-1, -1, 0>(e); n3b = cell.template q<0, -1, 0>(e);
            n4a = cell.template q<-1, 1, 0>(e); n4b = cell.template q<0, 1, 0>(e);
            n5a = cell.template q<-1, 0, -1>(e); n5b = cell.template q<0, 0, -1>(e);
            n6a = cell.template q<-1, 0, 1>(e); n6b = cell.template q<0, 0, 1>(e);
        } else if constexpr (D == 1) {
            n3a = cell.template q<0, -1, -1>(e); n3b = cell.template q<0, 0, -1>(e);
            n4a = cell.template q<0, -1, 1>(e); n4b = cell.template q<0, 0, 1>(e);
            n5a = cell.template q<-1, -1, 0>(e); n5b = cell.template q<-1, 0, 0>(e);
            n6a = cell.template q<1, -1, 0>(e); n6b = cell.template q<1, 0, 0>(e);
        } else {
            n3a = cell.template q<-1, 0, -1>(e); n3b = cell.template q<-1, 0, 0>(e);
            n4a = cell.template q<1, 0, -1>(e); n4b = cell.template q<1, 0, 0>(e);
            n5a = cell.template q<0, -1, -1>(e); n5b = cell.template q<0, -1, 0>(e);
            n6a = cell.template q<0, 1, -1>(e); n6b = cell.template q<0, 1, 0>(e);
        }
        double f3 = f2 + f1 + n3a + n3b;
        double f4 = f2 + f1 + n4a + n4b;
        double f5 = f2 + f1 + n5a + n5b;
        double f6 = f2 + f1 + n6a + n6b;
#pragma unroll
        for (int m = 0; m < 3; m++)
            g[e - 1][m] = (f2 * t1[m] - f1 * t0[m]) + (f4 * u1[m] - f3 * u0[m]) + (f6 * w1[m] - f5 * w0[m]);
    }
    constexpr int IL = D == 0 ? -1 : 0, JL = D == 1 ? -1 : 0, KL = D == 2 ? -1 : 0;
    double div = (g[0][0] + g[1][1] + g[2][2]) * f.cvisq;
    double f1 = g[0][0] - div, f2 = g[0][1] + g[1][0], f3 = g[0][2] + g[2][0];
    double f4 = g[1][1] - div, f5 = g[1][2] + g[2][1], f6 = g[2][2] - div;
    double volinv = 1. / (cell.template met<0, 0, 0>(z.vol, 0) + cell.template met<IL, JL, KL>(z.vol, 0));
    double xmutvol = (cell.template mu<0, 0, 0>() + cell.template mu<IL, JL, KL>()) * volinv;
    double xktvol = xmutvol * f.gam3;
    double tcx = tn[0], tcy = tn[1], tcz = tn[2], fv, fv5;
    fv = -(2. * f1 * tcx + f2 * tcy + f3 * tcz) * xmutvol;
    fv5 = fv * (qr[1] + ql[1]); flu[1] = flu[1] + fv;
    fv = -(f2 * tcx + 2. * f4 * tcy + f5 * tcz) * xmutvol;
    fv5 = fv5 + fv * (qr[2] + ql[2]); flu[2] = flu[2] + fv;
    fv = -(f3 * tcx + f5 * tcy + 2. * f6 * tcz) * xmutvol;
    fv5 = fv5 + fv * (qr[3] + ql[3]); flu[3] = flu[3] + fv;
    fv = fv5 * 0.5 - (g[3][0] * tcx + g[3][1] * tcy + g[3][2] * tcz) * xktvol;
    flu[4] = flu[4] + fv;
    if (gv) {
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int m = 0; m < 3; m++) gv[3 * e + m] = g[e][m];
        gv[12] = volinv;
    }
}

// Full face flux through the face (l - inc_D, l) of a cell
template <int KFLU, int SLOPE, bool LAMIN, bool CART, int D, typename Cell>
__device__ __forceinline__ void face_flux_at(const FluxConst& f, const KZ& z, const Cell& cell, double flu[5]) {
    double qm[5], qp[5], tn[3], sn;
    if (CART) {
        tn[0] = f.tc[0]; tn[1] = f.tc[1]; tn[2] = f.tc[2]; sn = f.s[D];
    } else {
        const double* t = D == 0 ? z.ti : D == 1 ? z.tj : z.tk;
#pragma unroll
        for (int m = 0; m < 3; m++) tn[m] = cell.template met<0, 0, 0>(t, m);
        sn = sqrt(tn[0] * tn[0] + tn[1] * tn[1] + tn[2] * tn[2]);
    }
    slope_state<SLOPE, D>(f, cell, qm, qp);
    inviscid_flux<KFLU, CART, D>(f, cell, tn, sn, qm, qp, flu);
    if constexpr (LAMIN) {
        if constexpr (CART) visc_cart<D>(f, cell, flu);
        else visc_full<D>(f, z, cell, tn, flu);
    }
}
// the same of cell (i, j, k), read from memory
template <int KFLU, int SLOPE, bool LAMIN, bool CART, int D, typename Cell = MemCell>
__device__ __forceinline__ void face_flux(const FluxConst& f, const KZ& z, const double* __restrict__ rop,
                                          int i, int j, int k, double flu[5]) {
    face_flux_at<KFLU, SLOPE, LAMIN, CART, D>(f, z, Cell(z, rop, IDX(z, i, j, k), CART ? 0 : MTR(z, i, j, k)), flu);
}

}  // namespace fm
