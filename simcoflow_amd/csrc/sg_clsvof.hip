// Coupled level-set / volume-of-fluid transport on gfx950 (Clsvof_Mod.f90).
//
// One call advances vof and phi over dt in nsub sub-steps (Coupled_LS_VOF,
// Clsvof_Mod.f90:730-959).  Each sub-step runs these launches:
//
//   k_recon      PLIC reconstruction (Interface_Reconstruct :1250-1321): find
//                the interface cells, then, packed one per lane, their normals,
//                plane constants and the PLIC face fluxes of the coming sweep
//   k_sweep      first sweep, implicit divergence (:798-823 / :862-888), with
//                the boundary copy (Boundary_Condition :961-973)
//   k_recon
//   k_sweep      second sweep, explicit divergence (:834-858 / :898-929)
//   k_recon (+ source list)
//   k_rd_scatter, k_redistance: level set from the PLIC segments (Redistance
//                :1525-1708)
//
// The reference's sweeps walk each row in order and update cells in place;
// every face flux they use depends only on data from before the sweep, so a
// sweep here is one thread per cell that recomputes the fluxes of its two
// faces and applies them in the reference's order.  Redistance scatters
// from interface cells into a 9x9 window.  For two- and three-phase targets
// the result is a minimum over the visits, taken here with one lane per
// (source, window offset) pair and an integer atomic minimum on the
// distance's bit pattern; full-solid targets, whose sign depends on the
// order of equal distances, replay their visits in the reference's order.
// Both give the reference's result bit for bit.
//
// This file is compiled with FP contraction off: every sum and product
// rounds as the reference writes it.
#include <type_traits>

#include "sg_internal.hpp"
#include "sg_poly.hpp"

namespace sg {

namespace {

constexpr double VOFEPS = 1.0e-14;   // Clsvof_Mod.f90:10
constexpr double TOLDENO = 1.0e-24;  // Clsvof_Mod.f90:10
constexpr int BAND = 4;              // Clsvof_Mod.f90:9 band_width

struct ClsGeo {
    int ni, nj;
    const double *dx, *dy, *xc, *yc;
    const double *vofS, *nxS, *nyS, *phiS;
    const double *aE, *aW, *aN, *aS;  // ghosted
    const int *uflag, *vflag;
    const double *u, *v;  // ghosted TVar%u, TVar%v
};

// 1-based cell index (the reference's (i,j)) -> cell array offset
__device__ __forceinline__ size_t cix(const ClsGeo& G, int i, int j) {
    return (size_t)(i - 1) + (size_t)(j - 1) * (size_t)G.ni;
}
__device__ __forceinline__ size_t gix(const ClsGeo& G, int i, int j) {
    return (size_t)i + (size_t)j * (size_t)(G.ni + 2);
}
__device__ __forceinline__ double fsign(double a, double b) { return copysign(fabs(a), b); }

// ---- PLIC geometry --------------------------------------------------------

// frac (:1371-1404): liquid fraction of a dx*dy box below |nx|x+|ny|y+d=0
__device__ double plic_frac(double nx, double ny, double d, double dx, double dy) {
    const double tnx = fabs(nx), tny = fabs(ny);
    if (d + 0.5 * (tnx * dx + tny * dy) <= 0.0) return 1.0;
    if (d - 0.5 * (tnx * dx + tny * dy) >= 0.0) return 0.0;
    if (tnx <= 1.0e-20) return 0.5 - d / dy;
    if (tny <= 1.0e-20) return 0.5 - d / dx;
    const double xx = (0.5 * tny * dy - d) / dx / tnx + 0.5;
    const double yy = (0.5 * tnx * dx - d) / dy / tny + 0.5;
    const double area = 0.5 * xx * yy;
    double top = 0.0, right = 0.0;
    if (yy > 1.0) {
        const double t = (yy - 1.0) / yy;
        top = t * t;
    }
    if (xx > 1.0) {
        const double t = (xx - 1.0) / xx;
        right = t * t;
    }
    return area * (1.0 - top - right);
}

// distance (:1323-1369): plane constant for volume fraction vf
__device__ double plic_distance(double vf, double nxx, double nyy, double dx, double dy) {
    const double nx = fabs(nxx), ny = fabs(nyy);
    if (nx < 1.0e-20) return (0.5 - vf) * dy;
    if (ny < 1.0e-20) return (0.5 - vf) * dx;
    const double dll = 0.5 * (nx * dx + ny * dy);
    double dul = 0.5 * (nx * dx - ny * dy);
    double dlr = -dul;
    const double dur = -dll;
    double vul = plic_frac(nx, ny, dul, dx, dy);
    double vlr = plic_frac(nx, ny, dlr, dx, dy);
    if (vf <= vul && vf <= vlr) {
        if (vul > vlr) {
            double t = vul; vul = vlr; vlr = t;
            t = dul; dul = dlr; dlr = t;
        }
        const double e = dul - dll;
        return dll - sqrt((e * e) * vf / vul);
    }
    if (vf >= vul && vf >= vlr) {
        if (vlr < vul) {
            double t = vul; vul = vlr; vlr = t;
            t = dul; dul = dlr; dlr = t;
        }
        const double e = dlr - dur;
        return dur + sqrt(e * e * (1.0 - vf) / (1.0 - vlr));
    }
    if (fabs(vlr - vul) < 1.0e-20) return 0.5 * (dul + dlr);
    const double th = (vf - vul) / (vlr - vul);
    return dlr * th + dul * (1.0 - th);
}

// Fluid part of a cell cut by the solid line, counter-clockwise from the SE
// corner (CellGeoCal :2170-2219, DistanceFluidCalculate :1966-2015): n <= 5
// vertices, x[n] repeats x[0], the rest are zero.  Every loop over the
// vertices is unrolled with a guard in place of a run-time bound, so each
// index is a compile-time constant and the polygon stays in registers.
struct Poly {
    double x[6], y[6];
    int n;
};

__device__ __forceinline__ void solid_poly(double nxs, double nys, double phis, double dx, double dy, Poly& P) {
#pragma unroll
    for (int k = 0; k < 6; ++k) P.x[k] = P.y[k] = 0.0;
    int n = 0;
    fluid_vertices(nxs, nys, phis, dx, dy, [&](double a, double b) {
        if (n < 5) {
#pragma unroll
            for (int s = 0; s < 5; ++s)
                if (s == n) {
                    P.x[s] = a;
                    P.y[s] = b;
                }
            ++n;
        }
    });
    const double x0 = P.x[0], y0 = P.y[0];
#pragma unroll
    for (int s = 1; s < 6; ++s)
        if (s == n) {
            P.x[s] = x0;
            P.y[s] = y0;
        }
    P.n = n;
}

// CellGeoCal (:2159-2253)
__device__ __forceinline__ void cell_geo(double nxs, double nys, double phis, double nxl, double nyl, double phil,
                                         double dx, double dy, double& vols, double& volf) {
    cut_cell_fractions(nxs, nys, phis, nxl, nyl, phil, dx, dy, vols, volf);
}

// LiqFuncVol (:2107-2155): volf less the fraction of the fluid polygon on
// the liquid side of the line through (xf, yf) with normal (nxf, nyf).  The
// reference takes the vertex count from the last non-zero vertex, nz - 1
// (the repeat of the first vertex makes that n), and closes the polygon at
// vertex nz - 1 with the first vertex's distance.  Inlined, so P stays in
// registers.
__device__ __forceinline__ double liq_func(double nxf, double nyf, double volf, double dx, double dy, const Poly& P, double xf,
                           double yf) {
    const double phil = -(nxf * xf + nyf * yf);
    // the reference counts vertices as the last non-zero node
    int nz = 0;
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (fabs(P.x[k]) > 1.0e-14 || fabs(P.y[k]) > 1.0e-14) nz = k + 1;
    if (nz == 0) return volf;
    const int n = nz - 1;
    double pdt[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) pdt[k] = P.x[k] * nxf + P.y[k] * nyf + phil;
    ShoelaceClip c;
#pragma unroll
    for (int k = 0; k < 5; ++k)
        if (k < n) c.edge(P.x[k], P.y[k], pdt[k], P.x[k + 1], P.y[k + 1], k + 1 == n ? pdt[0] : pdt[k + 1]);
    return volf - fabs(c.close() / (dx * dy));
}

// DistanceFluidCalculate + zriddr (:1957-2105).  Returns false when the
// reference leaves the plane constant unassigned.
__device__ bool distance_fluid(double nxs, double nys, double phis, double nxf, double nyf, double volf, double dx,
                               double dy, double& phif) {
    Poly P;
    solid_poly(nxs, nys, phis, dx, dy, P);
    const double diag = sqrt(dx * dx + dy * dy);
    double maxd = -2.0 * diag, mind = 2.0 * diag;
    double hx = 0.0, hy = 0.0, lx = 0.0, ly = 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        if (k >= P.n) break;
        const double t = nxf * P.x[k] + nyf * P.y[k];
        if (t > maxd) {
            maxd = t;
            hx = P.x[k];
            hy = P.y[k];
        }
        if (t < mind) {
            mind = t;
            lx = P.x[k];
            ly = P.y[k];
        }
    }
    hx = hx + hx * nxf * EPSI;
    hy = hy + hy * nyf * EPSI;
    lx = lx - lx * nxf * EPSI;
    ly = ly - ly * nyf * EPSI;
    // Ridders' method on the segment (lx,ly) -> (hx,hy), tol 1e-14, 1000 its
    const double tol = 1.0e-14;
    double fl = liq_func(nxf, nyf, volf, dx, dy, P, lx, ly);
    double fh = liq_func(nxf, nyf, volf, dx, dy, P, hx, hy);
    if ((fl > tol && fh < -tol) || (fl < -tol && fh > tol)) {
        double xlo = lx, ylo = ly, xhi = hx, yhi = hy;
        double ax = -1.11e-30, ay = -1.11e-30;
        for (int it = 0; it < 1000; ++it) {
            const double mx = 0.5 * (xlo + xhi), my = 0.5 * (ylo + yhi);
            const double fm = liq_func(nxf, nyf, volf, dx, dy, P, mx, my);
            const double s = sqrt(fm * fm - fl * fh);
            const double sg = fsign(1.0, fl - fh);
            const double nxw = mx + (mx - xlo) * sg * fm / s;
            const double nyw = my + (my - ylo) * sg * fm / s;
            const double e0 = nxw - ax, e1 = nyw - ay;
            if (sqrt(e0 * e0 + e1 * e1) <= tol) {
                phif = -(nxf * ax + nyf * ay);
                return true;
            }
            ax = nxw;
            ay = nyw;
            const double fn = liq_func(nxf, nyf, volf, dx, dy, P, ax, ay);
            if (fabs(fn) <= tol) {
                phif = -(nxf * ax + nyf * ay);
                return true;
            }
            if (fsign(fm, fn) != fm) {
                xlo = mx; ylo = my; fl = fm;
                xhi = ax; yhi = ay; fh = fn;
            } else if (fsign(fl, fn) != fl) {
                xhi = ax; yhi = ay; fh = fn;
            } else if (fsign(fh, fn) != fh) {
                xlo = ax; ylo = ay; fl = fn;
            }
            const double h0 = xhi - xlo, h1 = yhi - ylo;
            if (sqrt(h0 * h0 + h1 * h1) <= tol) {
                phif = -(nxf * ax + nyf * ay);
                return true;
            }
        }
        phif = -(nxf * ax + nyf * ay);
        return true;
    }
    if (fl < tol && fl > -tol) {
        phif = -(nxf * lx + nyf * ly);
        return true;
    }
    if (fh < tol && fh > -tol) {
        phif = -(nxf * hx + nyf * hy);
        return true;
    }
    return false;
}

// ---- normals ----------------------------------------------------------------

struct PhiView {
    const ClsGeo& G;
    const double* phi;
    __device__ double operator()(int i, int j) const { return phi[cix(G, i, j)]; }
    __device__ double X(int i) const { return G.xc[i - 1]; }
    __device__ double Y(int j) const { return G.yc[j - 1]; }
};

// The level set and the cell centres around an inner cell that its normal may
// ask for, loaded together before the first test: offsets are compile-time
// constants, so all of it stays in registers.  Two cells away is clamped to the
// grid; normal_irre does not use what lies beyond it.
struct Stencil {
    double v[13], x[5], y[5];
    static constexpr int at(int di, int dj) {
        return dj == 0 ? di + 2 : di == 0 ? 5 + (dj < 0 ? dj + 2 : dj + 1) : 9 + (di > 0 ? 1 : 0) + (dj > 0 ? 2 : 0);
    }
    __device__ __forceinline__ double operator()(int di, int dj) const { return v[at(di, dj)]; }
    __device__ __forceinline__ double X(int di) const { return x[di + 2]; }
    __device__ __forceinline__ double Y(int dj) const { return y[dj + 2]; }
};
__device__ __forceinline__ Stencil stencil(const ClsGeo& G, const double* __restrict__ phi, int i, int j) {
    Stencil s;
    const int im = max(i - 2, 1), ip = min(i + 2, G.ni), jm = max(j - 2, 1), jp = min(j + 2, G.nj);
#pragma unroll
    for (int d = -1; d <= 1; ++d) {
        s.v[Stencil::at(d, 0)] = phi[cix(G, i + d, j)];
        if (d) {
            s.v[Stencil::at(0, d)] = phi[cix(G, i, j + d)];
            s.v[Stencil::at(d, -1)] = phi[cix(G, i + d, j - 1)];
            s.v[Stencil::at(d, 1)] = phi[cix(G, i + d, j + 1)];
        }
        s.x[d + 2] = G.xc[i + d - 1];
        s.y[d + 2] = G.yc[j + d - 1];
    }
    s.v[Stencil::at(-2, 0)] = phi[cix(G, im, j)];
    s.v[Stencil::at(2, 0)] = phi[cix(G, ip, j)];
    s.v[Stencil::at(0, -2)] = phi[cix(G, i, jm)];
    s.v[Stencil::at(0, 2)] = phi[cix(G, i, jp)];
    s.x[0] = G.xc[im - 1];
    s.x[4] = G.xc[ip - 1];
    s.y[0] = G.yc[jm - 1];
    s.y[4] = G.yc[jp - 1];
    return s;
}

__device__ __forceinline__ double qual(double vx, double vy) { return fabs(1.0 - sqrt(vx * vx + vy * vy)); }

// The 8 candidate directions of Coupled_LS_VOF (:746-753) as the reference
// leaves them: Vset(1,2) is overwritten with +1 and Vset(2,2) never set, so
// direction 2 is (0,0) and drops out (its cosine is 0/0).
__device__ __forceinline__ void vset(int k, double& a, double& b) {
    const double A[8] = {0.0, 0.0, -1.0, -1.0, -1.0, 1.0, 1.0, 1.0};
    const double B[8] = {1.0, 0.0, 0.0, -1.0, 1.0, 0.0, -1.0, 1.0};
    a = A[k];
    b = B[k];
}

// one-sided pair chosen by the direction most parallel to grad phi
// (Normal_Vector_Irre :1768-1827 / :1855-1905)
__device__ __forceinline__ void nv_directional(const Stencil& p, int imv0, double& nx, double& ny) {
    const double eta = 0.075, nuy = eta / 8.0;
    const double vx = (p(1, 0) - p(-1, 0)) / (p.X(1) - p.X(-1));
    const double vy = (p(0, 1) - p(0, -1)) / (p.Y(1) - p.Y(-1));
    double maxv = 0.0;
    int imv = imv0;
    for (int k = 1; k <= 8; ++k) {
        double a, b;
        vset(k - 1, a, b);
        const double cp = fabs(a * vx + b * vy) / (sqrt(a * a + b * b) * sqrt(vx * vx + vy * vy));
        if (cp >= maxv) {
            maxv = cp;
            imv = k;
        }
    }
    double v1x, v1y;
    if (imv == 0) {  // zero gradient: outside Vset in the reference
        v1x = -1.0;
        v1y = 0.0;
    } else {
        double a, b;
        vset(imv - 1, a, b);
        v1x = -b;
        v1y = a;
    }
    double vx1, vx2, vy1, vy2;
    if (v1x == -1.0) {
        vx1 = (p(0, 0) - p(-1, 0)) / (p.X(0) - p.X(-1));
        vx2 = (p(1, 0) - p(0, 0)) / (p.X(1) - p.X(0));
    } else if (v1x == 0.0) {
        vx1 = (p(1, 0) - p(-1, 0)) / (p.X(1) - p.X(-1));
        vx2 = vx1;
    } else {
        vx1 = (p(1, 0) - p(0, 0)) / (p.X(1) - p.X(0));
        vx2 = (p(0, 0) - p(-1, 0)) / (p.X(0) - p.X(-1));
    }
    if (v1y == -1.0) {
        vy1 = (p(0, 0) - p(0, -1)) / (p.Y(0) - p.Y(-1));
        vy2 = (p(0, 1) - p(0, 0)) / (p.Y(1) - p.Y(0));
    } else if (v1y == 0.0) {
        vy1 = (p(0, 1) - p(0, -1)) / (p.Y(1) - p.Y(-1));
        vy2 = vy1;
    } else {
        vy1 = (p(0, 1) - p(0, 0)) / (p.Y(1) - p.Y(0));
        vy2 = (p(0, 0) - p(0, -1)) / (p.Y(0) - p.Y(-1));
    }
    if (qual(vx1, vy1) < qual(vx2, vy2) + nuy) {
        nx = vx1;
        ny = vy1;
    } else {
        nx = vx2;
        ny = vy2;
    }
}

// Normal_Vector_Irre (:1710-1919), interior cells; vs the cell's vofS
__device__ __forceinline__ void normal_irre(const ClsGeo& G, const Stencil& p, double vs, int i, int j, double& nx,
                                            double& ny) {
    const double eta = 0.075;
    if (vs >= EPSI) {
        const double se = G.vofS[cix(G, i + 1, j)], sw = G.vofS[cix(G, i - 1, j)];
        const double sn = G.vofS[cix(G, i, j + 1)], ss = G.vofS[cix(G, i, j - 1)];
        if (se < 1.0 - EPSI && sw < 1.0 - EPSI)
            nx = (p(1, 0) - p(-1, 0)) / (p.X(1) - p.X(-1));
        else if (se >= 1.0 - EPSI)
            nx = (p(0, 0) - p(-1, 0)) / (p.X(0) - p.X(-1));
        else
            nx = (p(1, 0) - p(0, 0)) / (p.X(1) - p.X(0));
        if (sn < 1.0 - EPSI && ss < 1.0 - EPSI)
            ny = (p(0, 1) - p(0, -1)) / (p.Y(1) - p.Y(-1));
        else if (sn > 1.0 - EPSI)
            ny = (p(0, 0) - p(0, -1)) / (p.Y(0) - p.Y(-1));
        else
            ny = (p(0, 1) - p(0, 0)) / (p.Y(1) - p.Y(0));
        return;
    }
    const double cx = (p(1, 0) - p(-1, 0)) / (p.X(1) - p.X(-1));
    const double cy = (p(0, 1) - p(0, -1)) / (p.Y(1) - p.Y(-1));
    const double q0 = qual(cx, cy);
    double vx, vy;
    vx = i >= 3 ? (p(0, 0) - p(-2, 0)) / (p.X(0) - p.X(-2)) : (p(0, 0) - p(-1, 0)) / (p.X(0) - p.X(-1));
    vy = (p(-1, 1) - p(-1, -1)) / (p.Y(1) - p.Y(-1));
    const double qm = qual(vx, vy);
    vx = i <= G.ni - 2 ? (p(2, 0) - p(0, 0)) / (p.X(2) - p.X(0))
                       : (p(1, 0) - p(0, 0)) / (p.X(1) - p.X(0));
    vy = (p(1, 1) - p(1, -1)) / (p.Y(1) - p.Y(-1));
    const double qp = qual(vx, vy);
    int sx = 0, sy = 0;
    int start = -1;  // the directional rule, and the direction it starts from (one copy of its code)
    if (qm < eta && qp >= eta) sx = -1;
    else if (qm >= eta && qp < eta) sx = 1;
    else if (qm < eta && q0 < eta && qp < eta) sx = 0;
    else if (qm >= eta && q0 >= eta && qp >= eta) sx = 0;
    else start = 0;
    vy = j >= 3 ? (p(0, 0) - p(0, -2)) / (p.Y(0) - p.Y(-2)) : (p(0, 0) - p(0, -1)) / (p.Y(0) - p.Y(-1));
    vx = (p(1, -1) - p(-1, -1)) / (p.X(1) - p.X(-1));
    const double rm = qual(vx, vy);
    vx = (p(1, 1) - p(-1, 1)) / (p.X(1) - p.X(-1));
    vy = j <= G.nj - 2 ? (p(0, 2) - p(0, 0)) / (p.Y(2) - p.Y(0))
                       : (p(0, 1) - p(0, 0)) / (p.Y(1) - p.Y(0));
    const double rp = qual(vx, vy);
    if (rm < eta && rp >= eta) sy = -1;
    else if (rm >= eta && rp < eta) sy = 1;
    else if (rm < eta && q0 < eta && rp < eta) sy = 0;
    else if (rm >= eta && q0 >= eta && rp >= eta) sy = 0;
    else if (start < 0) start = 1;
    if (start >= 0) {
        nv_directional(p, start, nx, ny);
        return;
    }
    if (sx == -1) nx = (p(0, 0) - p(-1, 0)) / (p.X(0) - p.X(-1));
    else if (sx == 1) nx = (p(1, 0) - p(0, 0)) / (p.X(1) - p.X(0));
    else nx = cx;
    if (sy == -1) ny = (p(0, 0) - p(0, -1)) / (p.Y(0) - p.Y(-1));
    else if (sy == 1) ny = (p(0, 1) - p(0, 0)) / (p.Y(1) - p.Y(0));
    else ny = cy;
}

// interface class of Interface_Reconstruct (:1258-1266): 0 none, 1 two
// phases, 2 three phases
__device__ __forceinline__ int recon_class(double vf, double vs) {
    if (vf >= VOFEPS && vf < (1.0 - VOFEPS - vs)) {
        if (vs < EPSI) return 1;
        if (vs < 1.0 - EPSI) return 2;
    }
    return 0;
}

__device__ __forceinline__ void normalise(double& nx, double& ny) {
    const double t = sqrt(nx * nx + ny * ny);
    if (t < 1.0e-14) {
        nx = 0.0;
        ny = 1.0;
    } else {
        nx = nx / t;
        ny = ny / t;
    }
}

// one-sided differences the reference uses on the domain edge (:1272-1283)
__device__ __forceinline__ double edge_nx(const PhiView& p, int i, int j, int ni) {
    return i == 1 ? (p(2, j) - p(1, j)) / (p.X(2) - p.X(1)) : (p(ni, j) - p(ni - 1, j)) / (p.X(ni) - p.X(ni - 1));
}
__device__ __forceinline__ double edge_ny(const PhiView& p, int i, int j, int nj) {
    return j == 1 ? (p(i, 2) - p(i, 1)) / (p.Y(2) - p.Y(1)) : (p(i, nj) - p(i, nj - 1)) / (p.Y(nj) - p.Y(nj - 1));
}

__device__ __forceinline__ int cls_of(const ClsGeo& G, const double* vof, int i, int j) {
    const size_t c = cix(G, i, j);
    return recon_class(vof[c], G.vofS[c]);
}

// final normal of a cell on the west or east edge (i = 1 or ni).  Away from
// the corners the reference's y component is the previous cell's (i,j-1)
// final value (a stale local, :1271-1283), so a run of interface cells up the
// edge is a chain; it is walked from the cell below its start.
__device__ void final_side(const ClsGeo& G, const double* vof, const double* phi, int i, int j, double& nx,
                           double& ny) {
    const PhiView p{G, phi};
    const int nj = G.nj;
    if (!cls_of(G, vof, i, j)) {
        nx = 0.0;
        ny = 1.0;
        return;
    }
    if (j == 1 || j == nj) {
        nx = edge_nx(p, i, j, G.ni);
        ny = edge_ny(p, i, j, nj);
        normalise(nx, ny);
        return;
    }
    int js = j - 1;
    while (js > 1 && cls_of(G, vof, i, js)) --js;
    double nyp;
    if (js == 1 && cls_of(G, vof, i, 1)) {
        double a = edge_nx(p, i, 1, G.ni), b = edge_ny(p, i, 1, nj);
        normalise(a, b);
        nyp = b;
    } else {
        nyp = 1.0;
    }
    for (int k = js + 1; k <= j; ++k) {
        double a = edge_nx(p, i, k, G.ni), b = nyp;
        normalise(a, b);
        nyp = b;
        if (k == j) {
            nx = a;
            ny = b;
        }
    }
}

// The inner cell whose normal a cell that is not on the west or east edge
// starts from: its own, or on the south and north edges (1 < i < ni) that of
// the previous cell in the reference's loop order, (i,nj-1) for the north edge
// and for the south edge (i-1,nj), which takes its own from (i-1,nj-1).
__device__ __forceinline__ void normal_base(const ClsGeo& G, int i, int j, int& bi, int& bj) {
    bi = j == 1 ? i - 1 : i;
    bj = j == 1 || j == G.nj ? G.nj - 1 : j;
    // within the grid's inner cells also where the caller will not use it
    bi = min(max(bi, 2), G.ni - 1);
}

// final normal of interface cell (i,j) away from the west and east edges; p, vsb
// the stencil and vofS of its base cell
__device__ __forceinline__ void final_inner(const ClsGeo& G, const double* vof, const double* phi, const Stencil& p,
                                            double vsb, int i, int j, double& nx, double& ny) {
    const int ni = G.ni, nj = G.nj;
    int bi, bj;
    normal_base(G, i, j, bi, bj);
    const bool edge = j == 1 || j == nj;
    bool own = true;  // the base cell's normal is wanted
    if (j == nj) own = cls_of(G, vof, i, nj - 1) != 0;
    if (j == 1) own = i > 2 && cls_of(G, vof, i - 1, nj) && cls_of(G, vof, i - 1, nj - 1);
    nx = 0.0;
    ny = 1.0;
    if (own) {
        normal_irre(G, p, vsb, bi, bj, nx, ny);
        normalise(nx, ny);
    }
    if (!edge) return;
    const PhiView q{G, phi};
    if (j == 1) {
        if (i == 2) {
            double t;
            final_side(G, vof, phi, 1, nj, nx, t);
        } else if (cls_of(G, vof, i - 1, nj)) {
            double b = edge_ny(q, i - 1, nj, nj);
            normalise(nx, b);
        } else {
            nx = 0.0;
        }
    }
    ny = edge_ny(q, i, j, nj);
    normalise(nx, ny);
}

// ---- kernels ------------------------------------------------------------------

// PLIC planes of the last reconstruction.  They are stored only for interface
// cells (class 1 or 2); every other cell has n = (0,1) and its plane constant
// follows from its volume fraction (Interface_Reconstruct :1307-1314), so
// readers rebuild those on the fly instead of reading them.
struct Planes {
    double* nx;
    double* ny;
    double* dis;
};

__device__ __forceinline__ double default_dis(double vf, double vs, double hy) {
    return 1.0 - vs > VOFEPS ? (0.5 - vf / (1.0 - vs)) * hy : (0.0 - vf) * hy;
}

__device__ __forceinline__ void plane_of(const ClsGeo& G, const Planes& P, size_t c, double vf, double hy, double& nx,
                                         double& ny, double& d) {
    const double vs = G.vofS[c];
    if (recon_class(vf, vs)) {
        nx = P.nx[c];
        ny = P.ny[c];
        d = P.dis[c];
    } else {
        nx = 0.0;
        ny = 1.0;
        d = default_dis(vf, vs, hy);
    }
}
// plane_of from values already loaded (cnx, cny, cdis: the stored plane)
__device__ __forceinline__ void plane_pick(double vf, double vs, double hy, double cnx, double cny, double cdis,
                                           double& nx, double& ny, double& d) {
    if (recon_class(vf, vs)) {
        nx = cnx;
        ny = cny;
        d = cdis;
    } else {
        nx = 0.0;
        ny = 1.0;
        d = default_dis(vf, vs, hy);
    }
}

// One bit per cell (a 64-bit word per 64 cells of a row) for what later kernels
// ask of every cell, written by whoever has the cell's vof in a register (a
// sweep, or a scanning reconstruction) so that nobody reads vof and vofS again
// only to find the interface.
enum { BIT_LIST = 0, BIT_SRC, BIT_GAS, BIT_LIQ, NBITS };
struct Bits {
    unsigned long long* w[NBITS];
    int mw;  // words per row
};
// BIT_LIST: an interface cell, or one whose face fluxes need the PLIC geometry
// (vof_flux's branch); BIT_SRC: a source of re-distancing; BIT_GAS, BIT_LIQ:
// empty or full cells, which take the band value away from the interface
__device__ __forceinline__ bool bit_list(double f, double vs) {
    return recon_class(f, vs) != 0 || !(f >= (1.0 - VOFEPS) || f <= VOFEPS);
}
__device__ __forceinline__ bool bit_src(double f, double vs) { return (0.0 + VOFEPS) < f && f < (1.0 - VOFEPS - vs); }
__device__ __forceinline__ bool bit_gas(double f) { return f <= VOFEPS; }
__device__ __forceinline__ bool bit_liq(double f, double vs) { return f >= (1.0 - VOFEPS - vs); }

// Boundary_Condition (:961-973) on two arrays: every ring cell takes its
// value from an interior cell, so the copy is race-free in place.
__global__ void k_bc(int ni, int nj, double* __restrict__ a, double* __restrict__ b) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int i, j, si, sj;
    if (t < ni) {
        i = t + 1; j = 1;
    } else if (t < 2 * ni) {
        i = t - ni + 1; j = nj;
    } else if (t < 2 * ni + (nj - 2)) {
        i = 1; j = t - 2 * ni + 2;
    } else if (t < 2 * ni + 2 * (nj - 2)) {
        i = ni; j = t - 2 * ni - (nj - 2) + 2;
    } else {
        return;
    }
    si = i == 1 ? 2 : (i == ni ? ni - 1 : i);
    sj = j == 1 ? 2 : (j == nj ? nj - 1 : j);
    const size_t d = (size_t)(i - 1) + (size_t)(j - 1) * ni, s = (size_t)(si - 1) + (size_t)(sj - 1) * ni;
    a[d] = a[s];
    b[d] = b[s];
}

// ---- sweeps -------------------------------------------------------------------
// A sweep along x (X=true) walks i in row b=j; along y it walks j in column
// b=i.  Index a is the position along the sweep, na its extent.
template <bool X>
struct Line {
    const ClsGeo& G;
    int b;
    __device__ int na() const { return X ? G.ni : G.nj; }
    __device__ size_t c(int a) const { return X ? cix(G, a, b) : cix(G, b, a); }
    // masked face velocity ue(a,j) / ve(i,a) (Coupled_LS_VOF :778-797)
    // (both loads are issued before the flag selects: no dependent round trip)
    __device__ double vel(int a) const {
        const int af = a > 0 ? a : 1;
        if (X) {
            const double w = G.u[gix(G, a, b)];
            const bool on = G.uflag[cix(G, af, b)];
            return a == 0 || on ? w : 0.0;
        }
        const double w = G.v[gix(G, b, a)];
        const bool on = G.vflag[cix(G, b, af)];
        return a == 0 || on ? w : 0.0;
    }
    // the same through a face that is not masked
    __device__ double raw(int a) const { return X ? G.u[gix(G, a, b)] : G.v[gix(G, b, a)]; }
    __device__ double ap(int a) const { return X ? G.aE[gix(G, a, b)] : G.aN[gix(G, b, a)]; }
    __device__ double am(int a) const { return X ? G.aW[gix(G, a, b)] : G.aS[gix(G, b, a)]; }
    __device__ double h(int a) const { return X ? G.dx[a - 1] : G.dy[a - 1]; }
    __device__ double hc() const { return X ? G.dy[b - 1] : G.dx[b - 1]; }
    __device__ double pos(int a) const { return X ? G.xc[a - 1] : G.yc[a - 1]; }
};

// rightflux/leftflux/topflux/bottomflux (:1416-1522): liquid volume swept
// through the far (side=+1) or near (side=-1) face over a width w
template <bool X>
__device__ double plic_face_flux(int side, double nxx, double nyy, double diss, double volf, double nxs, double nys,
                                 double phis, double vols, double hx, double hy, double w) {
    if (w == 0.0) return 0.0;
    const double nl = X ? nxx : nyy, ns = X ? nxs : nys, len = X ? hx : hy;
    const double sh = 0.5 * (w - len);
    const double dl = side > 0 ? diss - sh * nl : diss + sh * nl;
    double flux;
    if (vols < EPSI) {
        flux = X ? plic_frac(nxx, nyy, dl, w, hy) : plic_frac(nxx, nyy, dl, hx, w);
    } else if (vols >= 1.0 - EPSI) {
        return volf;
    } else {
        const double ps = side > 0 ? phis - sh * ns : phis + sh * ns;
        double volss;
        if (X)
            cell_geo(nxs, nys, ps, nxx, nyy, dl, w, hy, volss, flux);
        else
            cell_geo(nxs, nys, ps, nxx, nyy, dl, hx, w, volss, flux);
        if (volf / (1.0 - vols) >= 1.0 - VOFEPS) flux = 1.0 - volss;
        flux = flux / (1.0 - volss + TOLDENO);
        if (volf + vols > 1.0 - 1.0e-14) flux = 1.0;
    }
    return flux * w;
}

struct SweepIn {
    const double* vof;
    const double* phi;
    // PLIC fluxes prepared by the reconstruction: the sweep itself holds none
    // of the plane geometry, which keeps it free of scratch and light on registers
    const double* fr;
    const double* fl;
};

// vof_flux (X_Sweep :1014-1051) once the upwind cell of the face is known:
// f, vsU its vof and vofS, apU its aperture of the face, plic the PLIC flux
// precomputed for that side (read only for an interface cell, where
// VOFEPS < f < 1-VOFEPS)
__device__ __forceinline__ double upwind_flux(double w, double f, double vsU, double apU, const double* plic,
                                              size_t cU, double dtv) {
    double flux;
    if (f >= (1.0 - VOFEPS) || f <= VOFEPS) {
        flux = f * w * dtv;
        if (f >= 1.0) flux = w * dtv;
        if (f < 0.0) flux = 0.0;
    } else {
        flux = plic[cU];
    }
    if (apU > 1.0 - VOFEPS && vsU > 1.0 - VOFEPS) flux = 1.0 * w * dtv;
    return flux;
}

// level-set flux through interior face a (:1073-1096) from the level set
// at a-1, a, a+1, a+2 (pa1 = phi(a+1), pa2 = phi(a+2), ...)
__device__ __forceinline__ double ls_face(double w, int a, int n, double pm1, double p0, double p1, double p2,
                                          double dtv) {
    double l;
    if (w >= 0.0)
        l = (p1 + pm1) / 2.0;
    else if (a <= n - 2)
        l = (p2 + p0) / 2.0;
    else
        l = (p1 + pm1) / 2.0;
    return w * l * dtv;
}

// level-set flux through face 1 (:1098-1108 / :1218-1227)
template <bool X>
__device__ double ls_flux_first(const Line<X>& L, const double* phi, double dtv) {
    const double w = L.vel(1);
    const double p1 = phi[L.c(1)], p2 = phi[L.c(2)], p3 = phi[L.c(3)];
    double l;
    if (w >= 0.0)
        l = p1 + L.h(1) / 2.0 * (1.0 - w * dtv / L.h(1)) * (p2 - p1) / (L.pos(2) - L.pos(1));
    else
        l = p2 - L.h(2) / 2.0 * (1.0 + w * dtv / L.h(2)) * (p3 - p1) / (X ? 2.0 * L.h(2) : L.pos(3) - L.pos(1));
    return l * w * dtv;
}

__device__ __forceinline__ unsigned long long lane_word(unsigned long long v, int lane) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), lane);
    return (unsigned long long)hi << 32 | lo;
}

// ---- reconstruction ---------------------------------------------------------

// the sweep whose PLIC face fluxes a reconstruction prepares
enum FluxDir { FLUX_NONE = 0, FLUX_X, FLUX_Y };

struct ReconOut {
    Planes P;
    double* fr;
    double* fl;
};

// what the PLIC face fluxes of a cell need besides its plane
struct FluxIn {
    double nxs, nys, phis, w, w0;
};

// the PLIC face fluxes of cell c (VOFEPS < vof < 1-VOFEPS) with its plane: the
// far-face flux where the cell is upwind of its far face, the near-face flux
// where it is upwind of its near face -- exactly the values vof_flux would
// compute for them in the sweep (a loop over the two keeps one copy of the code)
template <bool X>
__device__ __forceinline__ void cell_fluxes(const FluxIn& F, int c, double f, double vs, double nx, double ny, double d,
                                            double hx, double hy, double dtv, double* __restrict__ fr,
                                            double* __restrict__ fl) {
    if (f >= (1.0 - VOFEPS) || f <= VOFEPS) return;  // not vof_flux's PLIC branch
#pragma unroll 1
    for (int side = 1; side >= -1; side -= 2) {
        const double w = side > 0 ? F.w : F.w0;
        if ((X ? (w >= 0.0) : (w > 0.0)) != (side > 0)) continue;
        const double flux = plic_face_flux<X>(side, nx, ny, d, f, F.nxs, F.nys, F.phis, vs, hx, hy,
                                              side > 0 ? w * dtv : -w * dtv);
        if (side > 0)
            fr[c] = flux;
        else
            fl[c] = -flux;
    }
}

// Interface_Reconstruct of cell c of the lanes with `in`: its normal and plane
// constant where it is an interface cell, then its fluxes.  A three-phase cell
// whose Ridders search leaves the plane constant unassigned takes the one of the
// nearest earlier cell in the reference's loop order (i outer, j inner) that
// assigns it (the reference keeps the previous cell's).  Those cells are worked
// out again from the same fields, which costs the wavefronts that hold such a
// cell another chain or two and every other reconstruction nothing: two steps
// back each lane on its own, then, as a run of such cells can be as long as a
// wall, 64 cells at a time for one lane, and for those whose run it is part of.
// (As a kernel over a list of such cells it took 3.6 us of each reconstruction
// at 333 x 171, empty or not; with each lane alone, a run of 1024 cells on 256 x
// 1024 took 3.3 ms of each against 77 us.)
constexpr int STALE_ALONE = 2;
template <int DIR>
__device__ __forceinline__ void recon_cell(const ClsGeo& G, const double* __restrict__ vof,
                                           const double* __restrict__ phi, const ReconOut& O, double dtv, bool in,
                                           int c, bool full) {
    const int lane = __lane_id();
    const int ci = c % G.ni + 1, cj = c / G.ni + 1;
    double vf = 0.0, vsc = 0.0, hxc = 0.0, hyc = 0.0;
    FluxIn F{};
    double nx = 0.0, ny = 1.0, d = 0.0;
    bool itf = false;
    int at = (ci - 1) * G.nj + cj - 1;  // the cell to ask next, in the loop's order
    bool open = in;                     // no plane constant yet
    for (int round = 0;; ++round) {
        const unsigned long long left = __ballot(open);
        if (!left) break;
        const bool own = round == 0, joint = round > STALE_ALONE;
        const int top = joint ? __builtin_amdgcn_readlane(at, 63 - __clzll((long long)left)) : 0;
        const int pos = joint ? top - lane : at;
        bool set = false;
        double dp = 0.0;  // before the first cell: the reference's uninitialised local
        if (joint ? pos >= 0 : open) {
            const int i = own ? ci : pos / G.nj + 1, j = own ? cj : pos % G.nj + 1;
            // everything a two-phase cell may need in one trip to memory
            const size_t p = cix(G, i, j);
            int bi, bj;
            normal_base(G, i, j, bi, bj);
            const double v = vof[p], vs = G.vofS[p], vsb = G.vofS[cix(G, bi, bj)];
            const double hx = G.dx[i - 1], hy = G.dy[j - 1];
            const Stencil S = stencil(G, phi, bi, bj);
            if (own) {
                vf = v;
                vsc = vs;
                hxc = hx;
                hyc = hy;
                if (DIR != FLUX_NONE) {
                    const Line<DIR == FLUX_X> L{G, DIR == FLUX_X ? j : i};
                    const int a = DIR == FLUX_X ? i : j;
                    F = FluxIn{G.nxS[p], G.nyS[p], G.phiS[p], L.vel(a), L.vel(a - 1)};
                }
            }
            const int cl = recon_class(v, vs);
            set = true;
            if (cl) {
                double mx, my;
                if (i == 1 || i == G.ni)
                    final_side(G, vof, phi, i, j, mx, my);
                else
                    final_inner(G, vof, phi, S, vsb, i, j, mx, my);
                if (cl == 1)
                    dp = plic_distance(v, mx, my, hx, hy);
                else
                    set = distance_fluid(G.nxS[p], G.nyS[p], G.phiS[p], mx, my, v, hx, hy, dp);
                if (own) {
                    nx = mx;
                    ny = my;
                    itf = true;
                }
            } else {
                dp = default_dis(v, vs, hy);
            }
        }
        if (!joint) {
            if (open && (set || at == 0)) {
                d = set ? dp : 0.0;
                open = false;
            }
            --at;
        } else {
            const unsigned long long hit = __ballot(pos < 0 || set);
            const int last = hit ? __ffsll((long long)hit) - 1 : 64;  // cells top .. top - last + 1 assign none
            const double found = __shfl(dp, last & 63, 64);
            if (open && at <= top && at >= top - last) {
                if (hit) {
                    d = found;
                    open = false;
                } else {
                    at = top - 64;
                }
            }
        }
    }
    if (!in) return;
    if (itf || full) {
        O.P.nx[c] = nx;
        O.P.ny[c] = ny;
    }
    if (itf) O.P.dis[c] = d;
    if (DIR != FLUX_NONE)
        cell_fluxes<DIR == FLUX_X>(F, c, vf, vsc, nx, ny, d, hxc, hyc, dtv, O.fr, O.fl);
}

// Interface_Reconstruct over the grid: a workgroup lists the cells of its 64 by
// `rows` that BIT_LIST names in LDS and works on them packed one per lane -- the
// geometry costs the same per cell wherever a cell lies, and packing keeps the
// wavefronts of bulk liquid and gas out of it.  SCAN: the bits are not there
// yet (a call's first reconstruction, or vofS has moved since the sweep), so
// they come from vof and vofS here and are written for the kernels after.
// full: also n = (0,1) for the other cells (the PCell%nx/ny output).  With
// srcs the sources of re-distancing are appended to it, one atomic a workgroup.
//
// Bound by the latency of one cell's chain of divisions and square roots, with
// SCAN also by 16 bytes a cell.  As a scan, a kernel over the listed cells, one
// over those with a stale plane constant and one for the fluxes it took 19.6 us
// at 333 x 171 and 37.3 us at 2048^2; now 8.5 and 15.1 us (8.1 and 19.2 us listing
// the sources, scanning 9.9 and 31.2).
//
// Few rows a workgroup keep a thread's share of a dense interface short, one
// cell of 64 x 4; many keep the wavefronts full where it is sparse.  A call of six
// sub-steps, us, by 4 / 8 / 16 / 32 rows (64 rows in front):
//   bubbles on a lattice of 8 cells, 256^2             1465: 620 / 700 / 777 / 990
//   the same at 512^2                                  2337: 1650 / 1665 / 1740 / 1910
//   the same at 1024^2                                 5940: 5800 / 5715 / 5725 / 5757
//   swarm 256^2                                         468: 334 / 357 / 356 / 400
//   swarm 512^2                                         515: 434 / 428 / 441 / 438
//   swarm 1024^2                                        795: - / 760 / 750 / 765
//   swarm 1448^2                                       1120: - / 1190 / 1125 / 1115
//   swarm 2048^2                                       1835: - / 2024 / 1893 / 1850
constexpr int RECON_NT = 256;
constexpr int RECON_H = 32;  // most rows of a workgroup (one a lane when the words are listed: 64 at most)
int recon_rows(size_t cells) { return cells < (1ull << 18) ? 4 : cells < (1ull << 21) ? 16 : RECON_H; }
template <int DIR, bool SCAN>
__global__ void __launch_bounds__(RECON_NT) k_recon(ClsGeo G, const double* __restrict__ vof,
                                                    const double* __restrict__ phi, ReconOut O, Bits B, double dtv,
                                                    int rows, int full, int* __restrict__ srcs,
                                                    unsigned* __restrict__ nsrc) {
    constexpr int NW = RECON_NT / 64, R = RECON_H / NW;
    __shared__ unsigned long long words[2][SCAN ? RECON_H : 1];
    __shared__ unsigned short list[64 * RECON_H];
    __shared__ unsigned gbase;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i0 = blockIdx.x * 64, jb = blockIdx.y * rows;
    if (SCAN) {
        const int i = i0 + lane + 1;
        // every row's operands loaded before any test
        double vf[R], vs[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = r * NW + w, j = jb + row + 1;
            const bool in = row < rows && i <= G.ni && j <= G.nj;
            const size_t c = in ? cix(G, i, j) : 0;
            vf[r] = in ? vof[c] : 0.0;
            vs[r] = in ? G.vofS[c] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int row = r * NW + w, j = jb + row + 1;
            const bool row_in = row < rows && j <= G.nj, in = row_in && i <= G.ni;
            unsigned long long b[NBITS];
            b[BIT_LIST] = __ballot(in && bit_list(vf[r], vs[r]));
            b[BIT_SRC] = __ballot(in && bit_src(vf[r], vs[r]));
            b[BIT_GAS] = __ballot(in && bit_gas(vf[r]));
            b[BIT_LIQ] = __ballot(in && bit_liq(vf[r], vs[r]));
            if (lane == 0) {
                words[0][row] = b[BIT_LIST];
                words[1][row] = b[BIT_SRC];
            }
            if (lane < NBITS && row_in) {
                const unsigned long long v = lane == 0 ? b[0] : lane == 1 ? b[1] : lane == 2 ? b[2] : b[3];
                B.w[lane][(size_t)(j - 1) * B.mw + blockIdx.x] = v;
            }
        }
        __syncthreads();
    }
    // one row's word a lane, in every wavefront
    unsigned long long wl = 0ull, ws = 0ull;
    if (lane < rows && jb + lane < G.nj) {
        const size_t at = (size_t)(jb + lane) * B.mw + blockIdx.x;
        wl = SCAN ? words[0][lane] : B.w[BIT_LIST][at];
        if (srcs) ws = SCAN ? words[1][lane] : B.w[BIT_SRC][at];
    }
    // the cells on the west and east edges, whose normals take a walk along a run
    // of them, come first in the list, a lane each: no thread has two walks to do
    // (256^2, an interface cell everywhere: 141 us against 2940 with up to sixteen)
    const int ei = G.ni - 1 - i0;
    const unsigned long long west = i0 == 0 ? 1ull : 0ull, east = ei < 64 ? 1ull << ei : 0ull;
    const unsigned long long wrows = __ballot((wl & west) != 0ull), erows = __ballot((wl & east) != 0ull);
    const unsigned nw = (unsigned)__popcll(wrows), nside = nw + (unsigned)__popcll(erows);
    // where each row's other cells and its sources start in the two lists: an
    // inclusive scan of the packed counts (low and high 16 bits) over the rows
    const unsigned own = (unsigned)__popcll(wl & ~(west | east)) | ((unsigned)__popcll(ws) << 16);
    unsigned incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    const unsigned all = (unsigned)__builtin_amdgcn_readlane((int)incl, 63);
    const unsigned n = nside + (all & 0xFFFFu), first = incl - own;
    if (!n && !(all >> 16) && !full) return;  // the workgroup as a whole
    if (all >> 16 && threadIdx.x == 0) gbase = atomicAdd(nsrc, all >> 16);
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int row = w; row < rows; row += NW) {
        const unsigned long long rl = lane_word(wl, row), before = (1ull << row) - 1ull;
        const bool on = rl >> lane & 1ull;
        unsigned at = (unsigned)__builtin_amdgcn_readlane((int)first, row) & 0xFFFFu;
        if (west >> lane & 1ull)
            at = (unsigned)__popcll(wrows & before);
        else if (east >> lane & 1ull)
            at = nw + (unsigned)__popcll(erows & before);
        else
            at += nside + (unsigned)__popcll(rl & ~(west | east) & below);
        if (on) list[at] = (unsigned short)(row * 64 + lane);
        if (full && !on && i0 + lane < G.ni && jb + row < G.nj) {
            const size_t c = cix(G, i0 + lane + 1, jb + row + 1);
            O.P.nx[c] = 0.0;
            O.P.ny[c] = 1.0;
        }
    }
    __syncthreads();
    if (all >> 16)
        for (int row = w; row < rows; row += NW) {
            const unsigned long long rs = lane_word(ws, row);
            const unsigned at = (unsigned)__builtin_amdgcn_readlane((int)first, row) >> 16;
            if (rs >> lane & 1ull)
                srcs[gbase + at + (unsigned)__popcll(rs & below)] = (int)cix(G, i0 + lane + 1, jb + row + 1);
        }
    for (unsigned t0 = w * 64u; t0 < n; t0 += RECON_NT) {
        const bool in = t0 + lane < n;
        const unsigned e = in ? list[t0 + lane] : 0u;
        const int c = (int)cix(G, i0 + (int)(e & 63u) + 1, jb + (int)(e >> 6) + 1);
        recon_cell<DIR>(G, vof, phi, O, dtv, in, c, full != 0);
    }
}

// The sweep's update of inner cell (i,j): t the new volume fraction (IMPL: the
// unclipped temvf), q the new level set.  Every operand a cell may need is
// loaded up front, with neighbour indices clamped to the line, before any of
// them decides which one is used: the upwind choice then costs no second round
// trip to memory.  OPEN: the cell and its neighbours along the sweep are free
// of solid, with open faces (k_open), so the aperture, solid fraction and face
// flag arrays are not read: their values are those written here.
//
// The first and last cells of a line lie on the domain's ring, whose results
// Boundary_Condition overwrites; so the reference's fluxes through the domain's
// own faces (the inflow among them) reach no cell and are not worked out.
template <bool X, bool IMPL, bool OPEN>
__device__ __forceinline__ void sweep_cell(const ClsGeo& G, const SweepIn& s, double dtv,
                                           const double* __restrict__ tv_in, int i, int j, double& t, double& q) {
    const Line<X> L{G, X ? j : i};
    const int a = X ? i : j;
    const int n = L.na();
    const int am2 = a > 2 ? a - 2 : a - 1;
    const int ap2 = a + 1 < n ? a + 2 : a + 1;
    const size_t c = L.c(a), cm = L.c(a - 1), cp = L.c(a + 1);
    const double vs = OPEN ? 0.0 : G.vofS[c], vsm = OPEN ? 0.0 : G.vofS[cm], vsp = OPEN ? 0.0 : G.vofS[cp];
    const double f0 = s.vof[c], fm = s.vof[cm], fp = s.vof[cp];
    const double wm = OPEN ? L.raw(a - 1) : L.vel(a - 1), w0 = OPEN ? L.raw(a) : L.vel(a);
    const double am0 = OPEN ? 1.0 : L.am(a), ap0 = OPEN ? 1.0 : L.ap(a);
    const double apm = OPEN ? 1.0 : L.ap(a - 1), amp = OPEN ? 1.0 : L.am(a + 1);
    const double ph0 = s.phi[c], phm1 = s.phi[cm], php1 = s.phi[cp];
    const double phm2 = s.phi[L.c(am2)], php2 = s.phi[L.c(ap2)];
    const double h = L.h(a);
    const double tvi = IMPL ? 0.0 : tv_in[c];
    // volume of fluid: temvf(a) after the sweep's in-place updates
    t = f0;
    if (vs < 1.0 - VOFEPS) t = t / (1.0 - vs);
    {
        // face a-1: upwind cell a-1 or a
        const double fx = (X ? (wm >= 0.0) : (wm > 0.0)) ? upwind_flux(wm, fm, vsm, apm, s.fr, cm, dtv)
                                                         : upwind_flux(wm, f0, vs, am0, s.fl, c, dtv);
        t = t * (1.0 - vs) + fx * am0 / h;
    }
    {
        // face a: upwind cell a or a+1
        const double fx = (X ? (w0 >= 0.0) : (w0 > 0.0)) ? upwind_flux(w0, f0, vs, ap0, s.fr, c, dtv)
                                                         : upwind_flux(w0, fp, vsp, amp, s.fl, cp, dtv);
        t = t - fx * ap0 / h;
    }
    // level set: temls(a)
    q = ph0;
    if (OPEN || a >= 3) q = q * (1.0 - vs) + ls_face(wm, a - 1, n, phm2, phm1, ph0, php1, dtv) * am0 / h;
    q = q - ls_face(w0, a, n, phm1, ph0, php1, php2, dtv) * ap0 / h;
    if (!OPEN && a == 2) q = q + ls_flux_first<X>(L, s.phi, dtv) * L.ap(1) / L.h(2);
    const double dvel = w0 * ap0 - wm * am0;
    if (IMPL) {
        const double den = (1.0 - vs + TOLDENO) - dtv / h * dvel;
        t = t / den;
        q = q / den;
    } else {
        // ph0 is the first sweep's temls: only the ring's was overwritten
        t = t + dtv / h * tvi * dvel;
        q = q + dtv / h * ph0 * dvel;
        q = vs < 1.0 - EPSI ? q / (1.0 - vs) : ph0;
    }
}

// One sweep with its boundary copy (Boundary_Condition :961-973): every thread
// works out an inner cell, a thread of the domain's ring the one its cell
// copies.  IMPL: first sweep of the sub-step (implicit divergence, clip);
// otherwise second sweep (explicit divergence with the first sweep's temvf).
// The results' class bits go out with them: a wavefront covers 32 cells of two
// rows, half a word each.
//
// Bound by bytes: 48 a cell in an open tile (vof, phi, a velocity, and three
// written, or temvf and two written), 76 otherwise.  At 2048^2 an x sweep takes
// 54 us (3.7 TB/s on the 48), a y sweep, whose halo rows are read again, 60 to
// 69 us; with a temls array of its own, the arrays above read everywhere and
// the boundary copy in a launch of its own, 74 to 80 us and 4.9 for the copy.
constexpr int SWEEP_W = 32, SWEEP_H = 8;  // cells per workgroup (a word half: SWEEP_W = 32)
template <bool X, bool IMPL>
__global__ void __launch_bounds__(SWEEP_W * SWEEP_H) k_sweep(ClsGeo G, SweepIn s, Bits B, double dtv,
                                                             const unsigned char* __restrict__ open,
                                                             const double* __restrict__ tv_in,
                                                             double* __restrict__ tv_out,
                                                             double* __restrict__ vof_out,
                                                             double* __restrict__ phi_out) {
    // x sweeps: XCD-aware tiles, so the tiles either side of a tile (whose
    // cells its stencil reads) share its L2; y sweeps: launch order, which
    // keeps vertically adjacent tiles on one XCD already
    int tx = blockIdx.x, ty = blockIdx.y;
    if (X) xcd_tile(tx, ty);
    const int i = tx * SWEEP_W + threadIdx.x + 1;
    const int j = ty * SWEEP_H + threadIdx.y + 1;
    const bool in = i <= G.ni && j <= G.nj;
    const bool free = open && (open[(size_t)ty * gridDim.x + tx] >> (X ? 0 : 1) & 1);
    double f = 0.0, q = 0.0, vs = 0.0;
    if (in) {
        // the inner cell whose result this cell takes
        const int si = min(max(i, 2), G.ni - 1), sj = min(max(j, 2), G.nj - 1);
        const size_t c = cix(G, i, j);
        double t;
        if (free) {
            sweep_cell<X, IMPL, true>(G, s, dtv, tv_in, si, sj, t, q);
        } else {
            vs = G.vofS[c];
            sweep_cell<X, IMPL, false>(G, s, dtv, tv_in, si, sj, t, q);
        }
        f = t;
        if (IMPL) {
            tv_out[c] = t;
            const double vss = free ? 0.0 : G.vofS[cix(G, si, sj)];
            f = t * (1.0 - vss);
            if (f >= 1.0 - VOFEPS - vss) f = 1.0 - vss;
            if (f < VOFEPS) f = 0.0;
        }
        vof_out[c] = f;
        phi_out[c] = q;
    }
    unsigned long long b[NBITS];
    b[BIT_LIST] = __ballot(in && bit_list(f, vs));
    if (!IMPL) {
        b[BIT_SRC] = __ballot(in && bit_src(f, vs));
        b[BIT_GAS] = __ballot(in && bit_gas(f));
        b[BIT_LIQ] = __ballot(in && bit_liq(f, vs));
    }
    if (threadIdx.x < (IMPL ? 1 : NBITS) && j <= G.nj) {
        const int k = threadIdx.x;
        const unsigned long long v =
            IMPL || k == 0 ? b[BIT_LIST] : k == 1 ? b[BIT_SRC] : k == 2 ? b[BIT_GAS] : b[BIT_LIQ];
        ((unsigned*)B.w[k])[(size_t)(j - 1) * (2 * B.mw) + tx] = (unsigned)(v >> (threadIdx.y % 2 * 32));
    }
}

// The sweep tiles free of solid: bit 0 (1) when no cell of the tile or beside it
// along x (y) holds solid or has a face along x (y) that is masked or not fully
// open, and the tile does not touch the domain's ring.  Once per call, since
// every sweep of a call sees the same geometry unless the solid moves.
// Bound by its 48 bytes a cell: a workgroup takes OPEN_TILES tiles of a column
// of them with every load issued before the first test (57.8 us at 2048^2, 71.6
// with one tile a workgroup).
constexpr int OPEN_TILES = 4;
__global__ void __launch_bounds__(SWEEP_W * SWEEP_H) k_open(ClsGeo G, unsigned char* __restrict__ open, int nty) {
    __shared__ unsigned closed[OPEN_TILES];
    const int x = threadIdx.x, y = threadIdx.y;
    const int i0 = blockIdx.x * SWEEP_W, t0 = blockIdx.y * OPEN_TILES;
    if (y == 0 && x < OPEN_TILES) closed[x] = 0u;
    __syncthreads();
    unsigned bad[OPEN_TILES];
#pragma unroll
    for (int k = 0; k < OPEN_TILES; ++k) {
        const int j0 = (t0 + k) * SWEEP_H;
        bad[k] = 0u;
        if (i0 == 0 || j0 == 0 || i0 + SWEEP_W >= G.ni || j0 + SWEEP_H >= G.nj) {
            bad[k] = 3u;
            continue;
        }
        auto check = [&](int i, int j, unsigned dirs) {
            const size_t c = cix(G, i, j), g = gix(G, i, j);
            const bool e = G.vofS[c] == 0.0;
            unsigned b = 0u;
            if (dirs & 1u) b |= !(e & (G.aE[g] == 1.0) & (G.aW[g] == 1.0) & (G.uflag[c] != 0)) ? 1u : 0u;
            if (dirs & 2u) b |= !(e & (G.aN[g] == 1.0) & (G.aS[g] == 1.0) & (G.vflag[c] != 0)) ? 2u : 0u;
            return b;
        };
        bad[k] = check(i0 + x + 1, j0 + y + 1, 3u);
        if (x < 2) bad[k] |= check(x ? i0 + SWEEP_W + 1 : i0, j0 + y + 1, 1u);
        if (y < 2) bad[k] |= check(i0 + x + 1, y ? j0 + SWEEP_H + 1 : j0, 2u);
    }
#pragma unroll
    for (int k = 0; k < OPEN_TILES; ++k)
        if (bad[k]) atomicOr(&closed[k], bad[k]);
    __syncthreads();
    if (y == 0 && x < OPEN_TILES && t0 + x < nty)
        open[(size_t)(t0 + x) * gridDim.x + blockIdx.x] = (unsigned char)(~closed[x] & 3u);
}

// ---- redistance -----------------------------------------------------------------

// isinsiderect (:1921-1955)
__device__ bool inside_rect(double xp, double yp, double dx, double dy) {
    const double x1 = -0.5 * dx, y1 = 0.5 * dy, x2 = 0.5 * dx, y2 = 0.5 * dy;
    const double x3 = 0.5 * dx, y3 = -0.5 * dy, x4 = -0.5 * dx, y4 = -0.5 * dy;
    const double b1 = sqrt((x1 - xp) * (x1 - xp) + (y1 - yp) * (y1 - yp));
    const double b2 = sqrt((x2 - xp) * (x2 - xp) + (y2 - yp) * (y2 - yp));
    const double b3 = sqrt((x3 - xp) * (x3 - xp) + (y3 - yp) * (y3 - yp));
    const double b4 = sqrt((x4 - xp) * (x4 - xp) + (y4 - yp) * (y4 - yp));
    const double u1 = 0.5 * (dx + b1 + b2), u2 = 0.5 * (dy + b2 + b3);
    const double u3 = 0.5 * (dx + b3 + b4), u4 = 0.5 * (dy + b4 + b1);
    const double a1 = sqrt(u1 * (u1 - dx) * (u1 - b1) * (u1 - b2));
    const double a2 = sqrt(u2 * (u2 - dy) * (u2 - b2) * (u2 - b3));
    const double a3 = sqrt(u3 * (u3 - dx) * (u3 - b3) * (u3 - b4));
    const double a4 = sqrt(u4 * (u4 - dy) * (u4 - b4) * (u4 - b1));
    return fabs(a1 + a2 + a3 + a4 - dx * dy) < 1.0e-10;
}

struct Target {
    double v, s, phi, x, y;  // vof, vofS, phi, centre of the target cell
};

// What one visit of a target by an interface source does (:1550-1686):
//   R2  two-phase target:   pa = sign(0.5-vof) * min(d, |pa|)
//   R3  three-phase target: if d < |pa|: pa = -d (liquid-full) or +d (empty)
//   RS  full-solid target:  if d < |pa|: pa = sign(dij) * d
// R2 and R3 reduce to a minimum over the visits in any order; RS depends on
// which source comes first among equal distances.
enum { V_NONE = 0, V_R2, V_R3, V_RS };
struct Visit {
    int kind;
    double d;
    double sg;  // RS sign
};

// the source cell's data a visit reads (its size, centre and solid line)
struct SrcCell {
    double dxs, dys, xc, yc, sxn, syn, sph, vs;
};
__device__ __forceinline__ SrcCell src_cell(const ClsGeo& G, int i, int j) {
    const size_t c = cix(G, i, j);
    return SrcCell{G.dx[i - 1], G.dy[j - 1], G.xc[i - 1], G.yc[j - 1], G.nxS[c], G.nyS[c], G.phiS[c], G.vofS[c]};
}

__device__ Visit propose(const SrcCell& S, int ii, int jj, double n1, double n2, double d1, const Target& T) {
    const double dxs = S.dxs, dys = S.dys;
    const double sxn = S.sxn, syn = S.syn, sph = S.sph;
    const int l = ii < -1 ? -1 : (ii > 1 ? 1 : ii);
    const int m = jj < -1 ? -1 : (jj > 1 ? 1 : jj);
    // point of the source cell's edge facing the target, moved off the solid
    double xv = dxs * (double)l / 2.0;
    double yv = dys * (double)m / 2.0;
    double dvs = sxn * xv + syn * yv + sph;
    if (dvs < 0.0) {
        if (fabs(yv) < VOFEPS) {
            yv = dys / 2.0;
            dvs = sxn * xv + syn * yv + sph;
            if (dvs < 0.0) {
                yv = -dys / 2.0;
                dvs = sxn * xv + syn * yv + sph;
                if (dvs < 0.0) {
                    xv = dxs * (0.0 - (double)l) / 2.0;
                    dvs = sxn * xv + syn * yv + sph;
                    if (dvs < 0.0) yv = dys / 2.0;
                }
            }
        } else if (fabs(xv) < VOFEPS) {
            xv = dxs / 2.0;
            dvs = sxn * xv + syn * yv + sph;
            if (dvs < 0.0) {
                xv = -dxs / 2.0;
                dvs = sxn * xv + syn * yv + sph;
                if (dvs < 0.0) {
                    yv = dys * (0.0 - (double)m) / 2.0;
                    dvs = sxn * xv + syn * yv + sph;
                    if (dvs < 0.0) xv = dxs / 2.0;
                }
            }
        } else {
            yv = dys * (0.0 - (double)m) / 2.0;
            dvs = sxn * xv + syn * yv + sph;
            if (dvs < 0.0) {
                xv = dxs * (0.0 - (double)l) / 2.0;
                yv = dys * (double)m / 2.0;
                dvs = sxn * xv + syn * yv + sph;
                if (dvs < 0.0) yv = dys * (0.0 - (double)m) / 2.0;
            }
        }
    }
    const double ddx = T.x - S.xc, ddy = T.y - S.yc;
    const int rule = T.s < EPSI ? V_R2 : V_R3;
    const double dv = n1 * xv + n2 * yv + d1;
    if (dv * fsign(1.0, T.phi) <= 0.0) {
        const double ax = ddx - xv, ay = ddy - yv;
        return {rule, sqrt(ax * ax + ay * ay), 0.0};
    }
    // projection of the target centre onto the source's PLIC line
    const double dij = n1 * ddx + n2 * ddy + d1;
    const double xp = ddx - dij * n1, yp = ddy - dij * n2;
    const bool inside = inside_rect(xp, yp, dxs, dys);
    if (inside && T.s < 1.0 - EPSI) {
        const double ax = ddx - xp, ay = ddy - yp;
        return {rule, sqrt(ax * ax + ay * ay), 0.0};
    }
    if (T.s >= 1.0 - EPSI) {
        if (S.vs < EPSI) {
            const double ax = ddx - xp, ay = ddy - yp;
            return {V_RS, sqrt(ax * ax + ay * ay), fsign(1.0, dij)};
        }
        return {V_NONE, 0.0, 0.0};
    }
    // nearest end of the segment
    const double tol = 1.0e-24;
    const double xoff = fmax(fabs(xp) - 0.5 * dxs, 0.0);
    const double yoff = fmax(fabs(yp) - 0.5 * dys, 0.0);
    const double xfc = fsign(1.0, xp) * 0.5 * dxs;
    const double yfc = fsign(1.0, yp) * 0.5 * dys;
    double xs, ys;
    if (xoff * fabs(n1 + tol) >= yoff * fabs(n2 + tol)) {
        xs = xfc;
        ys = (d1 + n1 * xs) / (-n2 + tol);
    } else {
        ys = yfc;
        xs = (d1 + n2 * ys) / (-n1 + tol);
    }
    const double ax = ddx - xs, ay = ddy - ys;
    const double deuc = sqrt(ax * ax + ay * ay);
    if (sxn * xs + syn * ys + sph >= 0.0) return {rule, deuc, 0.0};
    return {V_NONE, 0.0, 0.0};
}

__device__ __forceinline__ void apply(const Visit& w, const Target& T, double& pa) {
    if (w.kind == V_R2) {
        pa = fsign(1.0, 0.5 - T.v) * fmin(w.d, fabs(pa));
    } else if (w.kind == V_R3) {
        if (fabs(w.d) < fabs(pa) && T.v >= 1.0 - VOFEPS - T.s) pa = -fabs(w.d);
        if (fabs(w.d) < fabs(pa) && T.v < VOFEPS) pa = fabs(w.d);
    } else if (w.kind == V_RS) {
        if (fabs(w.d) < fabs(pa)) pa = w.sg * w.d;
    }
}

constexpr unsigned long long BEST_NONE = 0x7FF0000000000000ull;  // +inf: no proposal yet

__device__ __forceinline__ bool rd_source(double v, double s) { return (0.0 + VOFEPS) < v && v < (1.0 - VOFEPS - s); }
__device__ __forceinline__ bool rd_target(double v, double s) { return v < 0.0 + VOFEPS || v >= 1.0 - VOFEPS - s; }

// (source, offset) pairs of the listed interface cells; pair p is source
// p/81 and window offset o = p%81: column offset o%9 - BAND, row offset
// o/9 - BAND (consecutive lanes walk along a row of the window)
struct PairView {
    const int* srcs;
    const unsigned* cnt;
};

// Each pair proposes a distance to its target; two- and three-phase
// targets keep the minimum (the bit pattern of a non-negative double orders
// like the value).  Full-solid targets are left to the ordered gather of
// k_redistance.  `best` and `hit` hold +inf and 0 on entry: every cell
// a pair can reach lies in the band, and k_redistance puts them back
// after reading them.
__global__ void __launch_bounds__(256) k_rd_scatter(ClsGeo G, const double* __restrict__ vof,
                                                    const double* __restrict__ phi, Planes P, PairView pv,
                                                    unsigned long long* __restrict__ best,
                                                    unsigned char* __restrict__ hit) {
    const unsigned long long np = (unsigned long long)pv.cnt[0] * 81ull;
    for (unsigned long long p = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; p < np;
         p += (unsigned long long)gridDim.x * blockDim.x) {
        const int c0 = pv.srcs[p / 81];
        const int o = (int)(p % 81);
        const int si = c0 % G.ni + 1, sj = c0 / G.ni + 1;
        const int ii = o % 9 - BAND, jj = o / 9 - BAND;
        const int ti = si + ii, tj = sj + jj;
        if (ti < 1 || ti > G.ni || tj < 1 || tj > G.nj) continue;
        const size_t t = cix(G, ti, tj);
        // the target's and the source's data, loaded before the tests that
        // decide whether they are used
        Target T;
        T.v = vof[t];
        T.s = G.vofS[t];
        T.phi = phi[t];
        T.x = G.xc[ti - 1];
        T.y = G.yc[tj - 1];
        const SrcCell S = src_cell(G, si, sj);
        const double sv = vof[c0], snx = P.nx[c0], sny = P.ny[c0], sdis = P.dis[c0];
        if (!rd_target(T.v, T.s) || T.s >= 1.0 - EPSI) continue;
        double n1, n2, d1;
        plane_pick(sv, S.vs, S.dys, snx, sny, sdis, n1, n2, d1);
        const Visit w = propose(S, ii, jj, n1, n2, d1, T);
        if (w.kind == V_NONE) continue;
        if (w.kind == V_R2) hit[t] = 1;
        if (!(w.d != w.d)) atomicMin(best + t, (unsigned long long)__double_as_longlong(w.d));
    }
}

// bits lane-BAND .. lane+BAND of a row's words l, m, r (bit k <-> column
// offset k - BAND from the lane's cell)
__device__ __forceinline__ unsigned window_bits(unsigned long long l, unsigned long long m, unsigned long long r,
                                                int lane) {
    const int lo = lane - BAND;
    unsigned long long b = lo >= 0 ? m >> lo : (m << -lo) | (l >> (64 + lo));
    if (lo > 64 - (2 * BAND + 1)) b |= r << (64 - lo);
    return (unsigned)b & ((1u << (2 * BAND + 1)) - 1u);
}

// Redistance over the grid, one wavefront per 64-cell word of the source mask:
// interface cells take their plane constant, cells reached from an interface
// cell the nearest distance, the rest the band value.
//
// A word is in the band when an interface cell lies in rows j-BAND..j+BAND of
// mask words w-1..w+1, a superset of the windows of its 64 cells (BAND < 64).
// The wavefront reads those 27 words once, one per lane; or-ed over the rows
// they say of every lane whether its window holds a source.  In the band each
// cell's minimum and hit flag go back to +inf and 0 once read, ready for the
// next k_rd_scatter: the band holds every cell a pair can reach.  Full-solid
// targets replay their visits in the reference's source order (i ascending,
// then j ascending).
//
// Bound by its bytes, 8 a cell outside the band and 33 to 50 inside, and on a
// small grid by two trips to memory.  One kernel, because as three (test and
// list the words, cells outside, cells inside) it took 13.8 us at 333 x 171 and
// 69 us at 2048^2, against 4.2 and 31.2 us.
__global__ void __launch_bounds__(256) k_redistance(ClsGeo G, const double* __restrict__ vof, Planes P, Bits B,
                                                    unsigned long long* __restrict__ best,
                                                    unsigned char* __restrict__ hit, double* __restrict__ phi) {
    constexpr int ROWS = 2 * BAND + 1;
    const unsigned long long* mask = B.w[BIT_SRC];
    const int mw = B.mw;
    const int lane = threadIdx.x & 63;
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= mw * G.nj) return;  // the wavefront as a whole
    const int w = k % mw, tj = k / mw + 1, ti = w * 64 + lane + 1;
    const bool in = ti <= G.ni;
    const size_t c = cix(G, in ? ti : G.ni, tj);
    unsigned long long bits = 0ull;
    {
        const int r = tj - 1 + (lane & 15) - BAND, x = w + (lane >> 4) - 1;
        if ((lane & 15) < ROWS && lane < 48 && r >= 0 && r < G.nj && x >= 0 && x < mw)
            bits = mask[(size_t)r * mw + x];
    }
    const unsigned long long gas = B.w[BIT_GAS][k], liq = B.w[BIT_LIQ][k];
    const double hx = G.dx[(in ? ti : G.ni) - 1], hy = G.dy[tj - 1];
    unsigned long long any = bits;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) any |= __shfl_xor(any, o, 64);
    const unsigned long long l = lane_word(any, 0), m = lane_word(any, 16), r = lane_word(any, 32);
    if (l | m | r) {
        Target T;
        T.v = vof[c];
        T.s = G.vofS[c];
        const unsigned long long bc = best[c];
        const bool hc = hit[c] != 0;
        const bool source = rd_source(T.v, T.s);
        const bool visited = in && !source && rd_target(T.v, T.s) && window_bits(l, m, r, lane);
        double pa = 1.0e4;
        if (in && bc != BEST_NONE) best[c] = BEST_NONE;
        if (in && hc) hit[c] = 0;
        if (in && source) {
            double n1, n2, d1;
            plane_of(G, P, c, T.v, hy, n1, n2, d1);
            phi[c] = d1;  // an interface cell keeps its own plane constant
        }
        const bool solid = T.s >= 1.0 - EPSI;
        if (visited && !solid) {
            const double b = __longlong_as_double((long long)bc);
            if (T.s < EPSI) {
                if (hc) pa = fsign(1.0, 0.5 - T.v) * fmin(b, 1.0e4);
            } else if (b < 1.0e4) {
                pa = T.v >= 1.0 - VOFEPS - T.s ? -b : b;
            }
        }
        if (__ballot(visited && solid)) {
            // the sources of the window, column by column: bit ROWS * column + row
            unsigned long long set[2] = {0ull, 0ull};
#pragma unroll
            for (int row = 0; row < ROWS; ++row) {
                const unsigned win = window_bits(lane_word(bits, row), lane_word(bits, 16 + row),
                                                 lane_word(bits, 32 + row), lane);
#pragma unroll
                for (int col = 0; col < ROWS; ++col) {
                    const int at = ROWS * col + row;
                    set[at >> 6] |= (unsigned long long)(win >> col & 1u) << (at & 63);
                }
            }
            if (visited && solid) {
                T.phi = phi[c];
                T.x = G.xc[ti - 1];
                T.y = G.yc[tj - 1];
                while (set[0] | set[1]) {
                    int at;
                    if (set[0]) {
                        at = __ffsll((long long)set[0]) - 1;
                        set[0] &= set[0] - 1ull;
                    } else {
                        at = 64 + __ffsll((long long)set[1]) - 1;
                        set[1] &= set[1] - 1ull;
                    }
                    const int ii = at / ROWS - BAND, jj = at % ROWS - BAND;  // source - target
                    const int si = ti + ii, sj = tj + jj;
                    const size_t sc = cix(G, si, sj);
                    double n1, n2, d1;
                    plane_of(G, P, sc, vof[sc], G.dy[sj - 1], n1, n2, d1);
                    apply(propose(src_cell(G, si, sj), -ii, -jj, n1, n2, d1, T), T, pa);
                }
            }
        }
        if (!in || source) return;
        if (visited && !(pa > 9.999e3)) {
            phi[c] = pa;
            return;
        }
    }
    if (gas >> lane & 1ull)  // (no bit beyond the grid)
        phi[c] = (double)(BAND + 1) * sqrt(hx * hx + hy * hy);
    else if (liq >> lane & 1ull)
        phi[c] = -(double)(BAND + 1) * sqrt(hx * hx + hy * hy);
}

__global__ void k_fill_u64(unsigned long long* __restrict__ a, size_t n, unsigned long long v) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) a[t] = v;
}

__global__ void k_zero(unsigned* __restrict__ a, int n) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) a[t] = 0u;
}

// ---- interface on the U / V cells (Initial_ClsVofUV :402-710) ----------------

// LagrangePoly (:712-726) at PosTar = 0
__device__ double lagrange4(const double (&posi)[4], const double (&valu)[4]) {
    double val = 0.0;
    for (int i = 0; i < 4; ++i) {
        double mult = valu[i];
        for (int j = 0; j < 4; ++j)
            if (j != i) mult = mult * (0.0 - posi[j]) / (posi[i] - posi[j]);
        val = val + mult;
    }
    return val;
}

struct UVIn {
    const double *vof, *phi, *nx, *ny;   // P cells
    const double *vofST, *phiST;         // staggered solid fraction / level set
};

// liquid fraction of the half of P cell (i,j) facing the staggered cell
// (right: the half of the next cell); false when no branch of :448-536 /
// :591-672 assigns it
template <int W>
__device__ bool half_volf(const ClsGeo& G, const UVIn& in, bool right, int i, int j, double phisT, double& out) {
    const size_t c = cix(G, i, j);
    const double vf = in.vof[c], vs = G.vofS[c];
    const double dx = G.dx[i - 1], dy = G.dy[j - 1];
    double ph;
    if (W == 0)
        ph = right ? in.phi[c] - dx / 4.0 * in.nx[c] : in.phi[c] + dx / 4.0 * in.nx[c];
    else
        ph = right ? in.phi[c] - dy / 4.0 * in.ny[c] : in.phi[c] + dy / 4.0 * in.ny[c];
    const double hx = W == 0 ? dx / 2.0 : dx, hy = W == 0 ? dy : dy / 2.0;
    bool set = false;
    double v = 0.0;
    if (vf >= 1.0 - VOFEPS && vs < EPSI) { v = 1.0; set = true; }
    if (vf < 1.0 - VOFEPS && vf >= VOFEPS && vs < EPSI) { v = plic_frac(in.nx[c], in.ny[c], ph, hx, hy); set = true; }
    if (vf < VOFEPS && vs < EPSI) { v = 0.0; set = true; }
    if (vf < VOFEPS && vs >= 1.0 - EPSI) { v = 0.0; set = true; }
    if (vf < VOFEPS && vs < (W == 0 ? 1.0 - VOFEPS : 1.0 - EPSI) && vs >= EPSI) { v = 0.0; set = true; }
    if (vf >= VOFEPS && vf < 1.0 - VOFEPS && vs >= EPSI && vs < 1.0 - EPSI) {
        double vols;
        cell_geo(G.nxS[c], G.nyS[c], phisT, in.nx[c], in.ny[c], ph, hx, hy, vols, v);
        set = true;
    }
    if (set) out = v;
    return set;
}

// previous staggered cell in the reference's loop order (U: j outer, i
// inner over i < ni; V: i outer, j inner over j < nj); false before the first
template <int W>
__device__ __forceinline__ bool prev_cell(const ClsGeo& G, int& i, int& j) {
    if (W == 0) {
        if (i > 1) { --i; return true; }
        if (j > 1) { --j; i = G.ni - 1; return true; }
        return false;
    }
    if (j > 1) { --j; return true; }
    if (i > 1) { --i; j = G.nj - 1; return true; }
    return false;
}

// volfl / volfr of staggered cell (i,j), walking back to the last cell that
// assigned it when this one does not (stale locals of the reference)
template <int W>
__device__ double half_stale(const ClsGeo& G, const UVIn& in, bool right, int i, int j) {
    double v = 0.0;
    for (;;) {
        const int ip = W == 0 ? i + 1 : i, jp = W == 0 ? j : j + 1;
        const double phisT = in.phiST[cix(G, i, j)];
        if (right ? half_volf<W>(G, in, true, ip, jp, phisT, v) : half_volf<W>(G, in, false, i, j, phisT, v)) return v;
        if (!prev_cell<W>(G, i, j)) return 0.0;
    }
}

template <int W>
__device__ void uv_cell(const ClsGeo& G, const UVIn& in, int i, int j, double& tv, double& tp, double& tx, double& ty) {
    const int ip = W == 0 ? i + 1 : i, jp = W == 0 ? j : j + 1;
    const bool lagr = W == 0 ? (i >= 3 && i <= G.ni - 2) : (j >= 3 && j <= G.nj - 2);
    double p, a, b;
    if (lagr) {
        double posi[4], v1[4], v2[4], v3[4];
        for (int m = 0; m < 4; ++m) {
            const int ii = W == 0 ? i - 1 + m : i, jj = W == 0 ? j : j - 1 + m;
            posi[m] = W == 0 ? (G.xc[i - 1] + 0.5 * G.dx[i - 1]) - G.xc[ii - 1]
                             : (G.yc[j - 1] + 0.5 * G.dy[j - 1]) - G.yc[jj - 1];
            const size_t c = cix(G, ii, jj);
            v1[m] = in.phi[c];
            v2[m] = in.nx[c];
            v3[m] = in.ny[c];
        }
        p = lagrange4(posi, v1);
        a = lagrange4(posi, v2);
        b = lagrange4(posi, v3);
    } else {
        const size_t c0 = cix(G, i, j), c1 = cix(G, ip, jp);
        p = 0.5 * (in.phi[c1] + in.phi[c0]);
        a = 0.5 * (in.nx[c1] + in.nx[c0]);
        b = 0.5 * (in.ny[c1] + in.ny[c0]);
    }
    const double temn = W == 0 ? sqrt(a * a + b * b) + 1.0e-14 : sqrt(a * a + b * b + 1.0e-30);
    tp = p;
    tx = a / temn;
    ty = b / temn;
    const double vl = half_stale<W>(G, in, false, i, j);
    const double vr = half_stale<W>(G, in, true, i, j);
    double t = 0.5 * (vl + vr);
    const double vsT = in.vofST[cix(G, i, j)];
    if (t < VOFEPS) t = 0.0;
    if (t > 1.0 - VOFEPS - vsT) t = 1.0 - vsT;
    const int im = W == 0 ? i - 1 : i, jm = W == 0 ? j : j - 1;
    if ((W == 0 ? i > 1 : j > 1) && in.vof[cix(G, im, jm)] >= 1.0 - VOFEPS - G.vofS[cix(G, im, jm)] &&
        in.vof[cix(G, ip, jp)] >= 1.0 - VOFEPS - G.vofS[cix(G, ip, jp)])
        t = 1.0 - vsT;
    tv = t;
}

// one thread per staggered cell; the last column (U) / row (V) copies its
// neighbour (:555-558 / :700-703)
template <int W>
__global__ void __launch_bounds__(256) k_to_uv(ClsGeo G, UVIn in, double* __restrict__ tvof,
                                               double* __restrict__ tphi, double* __restrict__ tnx,
                                               double* __restrict__ tny) {
    // U: XCD-aware tiles (the stencil reaches along x); V: launch order
    int bx = blockIdx.x, by = blockIdx.y;
    if (W == 0) xcd_tile(bx, by);
    const int i = bx * blockDim.x + threadIdx.x + 1;
    const int j = by * blockDim.y + threadIdx.y + 1;
    if (i > G.ni || j > G.nj) return;
    const bool last = W == 0 ? i == G.ni : j == G.nj;
    const int si = last && W == 0 ? i - 1 : i, sj = last && W == 1 ? j - 1 : j;
    double tv, tp, tx, ty;
    uv_cell<W>(G, in, si, sj, tv, tp, tx, ty);
    const size_t c = cix(G, i, j);
    tvof[c] = tv;
    tphi[c] = tp;
    tnx[c] = tx;
    tny[c] = ty;
}

ClsGeo make_geo(Ctx* c) {
    ClsGeo G;
    G.ni = c->ni;
    G.nj = c->nj;
    G.dx = c->dx;
    G.dy = c->dy;
    G.xc = c->cls.xc;
    G.yc = c->cls.yc;
    G.vofS = (const double*)c->field[SG_F_VOFS];
    G.nxS = (const double*)c->field[SG_F_NXS];
    G.nyS = (const double*)c->field[SG_F_NYS];
    G.phiS = (const double*)c->field[SG_F_PHIS];
    G.aE = (const double*)c->field[SG_F_AE];
    G.aW = (const double*)c->field[SG_F_AW];
    G.aN = (const double*)c->field[SG_F_AN];
    G.aS = (const double*)c->field[SG_F_AS];
    G.uflag = (const int*)c->field[SG_F_UFLAG];
    G.vflag = (const int*)c->field[SG_F_VFLAG];
    G.u = (const double*)c->field[SG_F_U];
    G.v = (const double*)c->field[SG_F_V];
    return G;
}

}  // namespace

int clsvof_allocate(Ctx* c) {
    const size_t n = (size_t)c->ni * c->nj;
    ClsBuffers& B = c->cls;
    B.mw = (c->ni + 63) / 64;
    B.xc = (double*)dev_alloc(c, c->ni * sizeof(double));
    B.yc = (double*)dev_alloc(c, c->nj * sizeof(double));
    B.dis = (double*)dev_alloc(c, n * sizeof(double));
    B.vt = (double*)dev_alloc(c, n * sizeof(double));
    B.pt = (double*)dev_alloc(c, n * sizeof(double));
    B.tv = (double*)dev_alloc(c, n * sizeof(double));
    B.hit = (unsigned char*)dev_alloc(c, n);
    B.best = (unsigned long long*)dev_alloc(c, n * sizeof(unsigned long long));
    if (B.best) {
        hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, B.best, n,
                           BEST_NONE);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess) return SG_ERR_ALLOC;
    }
    B.srcs = (int*)dev_alloc(c, n * sizeof(int));
    B.fr = (double*)dev_alloc(c, n * sizeof(double));
    B.fl = (double*)dev_alloc(c, n * sizeof(double));
    B.cnt = (unsigned*)dev_alloc(c, ClsBuffers::MAX_NSUB * sizeof(unsigned));
    B.bits = (unsigned long long*)dev_alloc(c, NBITS * (size_t)B.mw * c->nj * sizeof(unsigned long long));
    B.open = (unsigned char*)dev_alloc(c, (size_t)((c->ni + SWEEP_W - 1) / SWEEP_W) * ((c->nj + SWEEP_H - 1) / SWEEP_H));
    if (!B.xc || !B.yc || !B.dis || !B.vt || !B.pt || !B.tv || !B.hit || !B.best || !B.srcs || !B.fr || !B.fl ||
        !B.cnt || !B.bits || !B.open)
        return SG_ERR_ALLOC;
    return SG_OK;
}

// the recorded sweep launches' durations into the totals (waits for them)
int sweep_timing_drain(Ctx* c) {
    auto& T = c->sweep_timing;
    for (int k = 0; k < T.used; ++k) {
        SG_HIP(hipEventSynchronize(T.ev[2 * k + 1]));
        float ms = 0.f;
        SG_HIP(hipEventElapsedTime(&ms, T.ev[2 * k], T.ev[2 * k + 1]));
        T.ms += ms;
        T.launches += 1;
    }
    T.used = 0;
    return SG_OK;
}

// From how many cells a call works out which of its sweep tiles are free of
// solid.  A call of 6 sub-steps (12 sweeps) and the U/V interface with and without,
// us, a swarm of bubbles: 724^2 642 / 641, 1024^2 798 / 792, 1200^2 906 / 924, 1448^2
// 1063 / 1134, 1600^2 1200 / 1311, 1800^2 1440 / 1606, 2048^2 1835 / 1960; waves with a
// solid 4096 x 2048 3150 / 3318; the sweeps alone at 512^2 508 / 491.  The flags pay
// for themselves from about 1.2 million cells, where a sweep's arrays, 104 bytes a
// cell with the geometry, are half the last-level cache's 256 MB and other kernels'
// take the rest; the line stands where they gain 6%, not where they break even.
constexpr size_t OPEN_MIN_CELLS = 1ull << 21;

// Coupled_LS_VOF on the device fields VOF, PHI (in/out), NX, NY (out),
// U, V (in).
int clsvof_advect(Ctx* c, double dt, int nsub) {
    const ClsGeo G = make_geo(c);
    ClsBuffers& B = c->cls;
    double* vof = (double*)c->field[SG_F_VOF];
    double* phi = (double*)c->field[SG_F_PHI];
    const Planes P{(double*)c->field[SG_F_NX], (double*)c->field[SG_F_NY], B.dis};
    const int ring = 2 * c->ni + 2 * (c->nj - 2);
    const dim3 rblk(256), rgrd((ring + 255) / 256);
    const dim3 pblk(256), pgrd(1024);  // a grid-stride loop over the listed pairs
    const int rrows = recon_rows((size_t)c->ni * c->nj);
    const dim3 rcgrd((c->ni + 63) / 64, (c->nj + rrows - 1) / rrows);
    // sweeps: 32x8 tiles (3% faster per transport call than 64x4, 256x1 or
    // 128x2 at 2048^2: the y stencil's rows stay within fewer tiles)
    const dim3 sblk(SWEEP_W, SWEEP_H), sgrd((c->ni + SWEEP_W - 1) / SWEEP_W, (c->nj + SWEEP_H - 1) / SWEEP_H);
    const double dtv = dt / (double)nsub;
    hipStream_t st = c->stream;
    // the number of sources listed, one per sub-step
    hipLaunchKernelGGL(k_zero, dim3((nsub + 255) / 256), dim3(256), 0, st, B.cnt, nsub);
    Bits bits;
    bits.mw = B.mw;
    for (int k = 0; k < NBITS; ++k) bits.w[k] = B.bits + (size_t)k * B.mw * c->nj;
    const bool moves = c->moving.shape.kind != SG_SOLID_NONE;
    const unsigned char* open = nullptr;
    if (!moves && (size_t)c->ni * c->nj >= OPEN_MIN_CELLS) {
        hipLaunchKernelGGL(k_open, dim3(sgrd.x, (sgrd.y + OPEN_TILES - 1) / OPEN_TILES), sblk, 0, st, G, B.open,
                           (int)sgrd.y);
        open = B.open;
    }
    // One reconstruction and, with `dir`, the face fluxes of the sweep after it.
    // scan: the class bits are not those of v yet; full: also n = (0,1) on the
    // other cells -- only the transport's very last one, since within the
    // transport a stored plane is read only where the cell is an interface cell
    // of the current vof (plane_of, plane_pick), and every such plane is
    // rewritten by the reconstruction
    auto recon = [&](auto dir, const double* v, const double* p, bool scan, bool full, int* srcs, unsigned* nsrc) {
        constexpr int DIR = decltype(dir)::value;
        const ReconOut O{P, B.fr, B.fl};
        if (scan)
            hipLaunchKernelGGL((k_recon<DIR, true>), rcgrd, dim3(RECON_NT), 0, st, G, v, p, O, bits, dtv, rrows,
                               full ? 1 : 0, srcs, nsrc);
        else
            hipLaunchKernelGGL((k_recon<DIR, false>), rcgrd, dim3(RECON_NT), 0, st, G, v, p, O, bits, dtv, rrows,
                               full ? 1 : 0, srcs, nsrc);
    };
    using std::integral_constant;
    const integral_constant<int, FLUX_NONE> no_flux{};
    const integral_constant<int, FLUX_X> flux_x{};
    const integral_constant<int, FLUX_Y> flux_y{};
    // sg_sweep_timing: an event before (end = 0) and after (end = 1) each sweep
    // (waiting for those before it when the pool is used up, wherever that is in a call)
    auto& TM = c->sweep_timing;
    auto sweep_mark = [&](int end) -> int {
        if (!TM.on) return SG_OK;
        if (!end && TM.used == Ctx::SweepTiming::POOL) {
            const int rc = sweep_timing_drain(c);
            if (rc) return rc;
        }
        SG_HIP(hipEventRecord(TM.ev[2 * TM.used + end], st));
        if (end) ++TM.used;
        return SG_OK;
    };
    int rc = SG_OK;
    for (int k = 1; k <= nsub; ++k) {
        // first sweep: (vof, phi) -> (vt, pt), implicit divergence; after the
        // first sub-step the bits are those of the last reconstruction, and
        // re-distancing has changed phi only
        if (k % 2 == 1)
            recon(flux_x, vof, phi, k == 1, false, nullptr, nullptr);
        else
            recon(flux_y, vof, phi, k == 1, false, nullptr, nullptr);
        const SweepIn s1{vof, phi, B.fr, B.fl};
        if ((rc = sweep_mark(0))) return rc;
        if (k % 2 == 1)
            hipLaunchKernelGGL((k_sweep<true, true>), sgrd, sblk, 0, st, G, s1, bits, dtv, open, nullptr, B.tv, B.vt,
                               B.pt);
        else
            hipLaunchKernelGGL((k_sweep<false, true>), sgrd, sblk, 0, st, G, s1, bits, dtv, open, nullptr, B.tv, B.vt,
                               B.pt);
        if ((rc = sweep_mark(1))) return rc;
        // second sweep: (vt, pt) -> (vof, phi), explicit divergence
        if (k % 2 == 1)
            recon(flux_y, B.vt, B.pt, false, false, nullptr, nullptr);
        else
            recon(flux_x, B.vt, B.pt, false, false, nullptr, nullptr);
        const SweepIn s2{B.vt, B.pt, B.fr, B.fl};
        if ((rc = sweep_mark(0))) return rc;
        if (k % 2 == 1)
            hipLaunchKernelGGL((k_sweep<false, false>), sgrd, sblk, 0, st, G, s2, bits, dtv, open, B.tv, nullptr, vof,
                               phi);
        else
            hipLaunchKernelGGL((k_sweep<true, false>), sgrd, sblk, 0, st, G, s2, bits, dtv, open, B.tv, nullptr, vof,
                               phi);
        if ((rc = sweep_mark(1))) return rc;
        if (moves) {
            // ObjectMovement (Clsvof_Mod.f90:2384-2398) over the sub-step,
            // then SolidVolumeFraction on the P cells (:920-921)
            auto& m = c->moving;
            m.shape.cy = m.shape.cy + 0.5 * m.asy * (dtv * dtv) + m.vs * dtv;
            m.shape.cx = m.shape.cx + 0.5 * m.asx * (dtv * dtv) + m.us * dtv;
            m.us = m.us + m.asx * dtv;
            m.vs = m.vs + m.asy * dtv;
            if ((rc = solid_fraction_step(c, &m.shape))) return rc;
            // the solid has changed vof too
            hipLaunchKernelGGL(k_bc, rgrd, rblk, 0, st, c->ni, c->nj, vof, phi);
        }
        // reconstruction (full normals out) and re-distancing
        unsigned* cnt = B.cnt + (k - 1);
        recon(no_flux, vof, phi, moves, k == nsub, B.srcs, cnt);
        const PairView pv{B.srcs, cnt};
        hipLaunchKernelGGL(k_rd_scatter, pgrd, pblk, 0, st, G, vof, phi, P, pv, B.best, B.hit);
        hipLaunchKernelGGL(k_redistance, dim3((unsigned)((B.mw * c->nj + 3) / 4)), dim3(256), 0, st, G, vof, P,
                           bits, B.best, B.hit, phi);
    }
    SG_HIP(hipGetLastError());
    return SG_OK;
}

}  // namespace sg

namespace sg {

// Initial_ClsVofUV for both staggered grids: device fields VOF, PHI, NX, NY
// (+ the solid geometry) -> UVOF/UPHI/UNX/UNY and VVOF/VPHI/VNX/VNY.
int interface_to_uv(Ctx* c) {
    const ClsGeo G = make_geo(c);
    const dim3 blk(64, 4), grd((c->ni + 63) / 64, (c->nj + 3) / 4);
    auto f = [&](int k) { return (double*)c->field[k]; };
    UVIn in{f(SG_F_VOF), f(SG_F_PHI), f(SG_F_NX), f(SG_F_NY), c->stag[0].a[STG_VOFS], c->stag[0].a[STG_PHIS]};
    hipLaunchKernelGGL(k_to_uv<0>, grd, blk, 0, c->stream, G, in, f(SG_F_UVOF), f(SG_F_UPHI), f(SG_F_UNX),
                       f(SG_F_UNY));
    in.vofST = c->stag[1].a[STG_VOFS];
    in.phiST = c->stag[1].a[STG_PHIS];
    hipLaunchKernelGGL(k_to_uv<1>, grd, blk, 0, c->stream, G, in, f(SG_F_VVOF), f(SG_F_VPHI), f(SG_F_VNX),
                       f(SG_F_VNY));
    SG_HIP(hipGetLastError());
    return SG_OK;
}

}  // namespace sg
