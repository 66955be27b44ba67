// Lagrangian particles on gfx950: TrackingParticles (Particles.f90:71-205)
// with Drag (:206-223) and ParticlePosition (:228-249), one thread per
// particle, FP64, in the reference's expression order with FP contraction
// off (exp and pow are the device library's, so results agree with a CPU
// restatement to rounding, not bit for bit).
//
// Kept from the reference: the fluid velocity at a particle is taken in its
// P-cell at the position of the start of the time step for all itp = 10
// sub-steps (the sub-steps advance the new position, not the one used for the
// lookup); u is interpolated linearly in x only and v in y only; a particle
// outside the grid is left alone; one past the last cell centre, or in a cell
// that is neither fluid nor full solid, is parked at (1e3, 1e3) with its
// velocity unchanged; one in a full-solid cell moves with the solid.
// ParticlePosition scans the columns and rows for the first closed interval
// [x_i - dx_i/2, x_i + dx_i/2] holding the point; here a binary search finds
// the first column whose upper edge is not below the point and the scan goes
// on from there, which picks the same column.
#include <algorithm>

#include "sg_internal.hpp"
#include "sg_divisor.hpp"

namespace sg {

namespace {

constexpr int ITP = 10;          // itp, Particles.f90:8
constexpr double TOLP = 1.0e-20; // tol, Particles.f90:9
constexpr double CAP = 0.5;      // Ca, Particles.f90:9

struct PGeo {
    int ni, nj;
    const double *xc, *yc, *dx, *dy;
    const double *vof, *vofS;  // cell arrays
    const double *u, *v;       // ghosted TVar%u, TVar%v
};

__device__ double drag(double re) {
    if (re < 1.0) return 24.0 / (re + TOLP);
    if (re <= 1000.0) return 24.0 / (re + TOLP) * (1.0 + 0.15 * pow(re, 0.687));
    return 0.44;
}

// 1-based index of the first interval [c_k - h_k/2, c_k + h_k/2] holding t, -1 if none
__device__ int locate(const double* __restrict__ c, const double* __restrict__ h, int n, double t) {
    // the first column whose upper edge is not below t: where an even spacing
    // puts it, if it and the one before say so (two trips to memory), else by
    // a binary search (one for every factor of two)
    const double a0 = c[0] - h[0] / 2.0, a1 = c[n - 1] + h[n - 1] / 2.0;
    int lo = (int)fmin(fmax((t - a0) / (a1 - a0) * (double)n, 0.0), (double)(n - 1));
    const int before = lo > 0 ? lo - 1 : 0;
    const bool here = c[lo] + h[lo] / 2.0 >= t, above = lo == 0 || !(c[before] + h[before] / 2.0 >= t);
    if (!(here && above)) {
        int hi = n;
        lo = 0;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (c[mid] + h[mid] / 2.0 >= t)
                hi = mid;
            else
                lo = mid + 1;
        }
    }
    for (int k = lo; k < n; ++k) {
        const double a = c[k] - h[k] / 2.0;
        if (t >= a && t <= c[k] + h[k] / 2.0) return k + 1;
        if (a > t) break;
    }
    return -1;
}

// One sub-step's chain -- square root, quotients, pow, exp -- is the kernel's
// time: with 1e5 particles there are one or two wavefronts a SIMD, and each
// waits for its own operations.  So the quotients by what does not change over
// the sub-steps take five operations instead of a division's dozen, and the
// look-up two trips to memory instead of nine (30.4 -> 27.0 us at 512^2).
__global__ void __launch_bounds__(256) k_particles(PGeo G, int n, double* __restrict__ px, double* __restrict__ py,
                                                   double* __restrict__ pu, double* __restrict__ pv,
                                                   const double* __restrict__ pd, sg_particle_params P, double dt,
                                                   unsigned* flagged) {
    const int p0 = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = p0 < n;
    const int p = in ? p0 : n - 1;
    const int ni = G.ni, nj = G.nj;
    const double x0 = px[p], y0 = py[p], dpp = pd[p];
    const double dtp = dt * (P.lref / P.uref) / (double)ITP;
    // the lookup uses the start-of-step position in every sub-step
    const int ii = locate(G.xc, G.dx, ni, x0 / P.lref);
    const int jj = locate(G.yc, G.dy, nj, y0 / P.lref);
    double xx = x0, yy = y0, upo = pu[p], vpo = pv[p];
    bool bad = false;
    if (ii != -1 && jj != -1) {
        const size_t c = (size_t)(ii - 1) + (size_t)(jj - 1) * ni;
        const size_t g = (size_t)ii + (size_t)jj * (ni + 2);
        const double f = G.vof[c], s = G.vofS[c];
        const bool fluid = x0 / P.lref < G.xc[ni - 1] && y0 / P.lref < G.yc[nj - 1] && s < 1.0 - EPSI;
        // the fluid velocity at the particle is the same in every sub-step
        double ug = 0.0, vg = 0.0, gama = 0.0, nupp = 0.0;
        if (fluid) {
            const double ropp = P.rho_l * f / (1.0 - s + TOLP) + P.rho_g * (1.0 - f - s) / (1.0 - s + TOLP);
            gama = P.rho_p / ropp;
            nupp = P.nu_l * f / (1.0 - s + TOLP) + P.nu_g * (1.0 - f - s) / (1.0 - s + TOLP);
            const double dudx = (G.u[g] - G.u[g - 1]) / G.dx[ii - 1];
            const double dvdy = (G.v[g] - G.v[g - (ni + 2)]) / G.dy[jj - 1];
            const double ug0 = 0.5 * (G.u[g] + G.u[g - 1]);
            const double vg0 = 0.5 * (G.v[g] + G.v[g - (ni + 2)]);
            ug = (ug0 + dudx * (x0 / P.lref - G.xc[ii - 1])) * P.uref;
            vg = (vg0 + dvdy * (y0 / P.lref - G.yc[jj - 1])) * P.uref;
        }
        const double half = dpp / 2.0, mass = gama + CAP;
        const Divisor by_nu(nupp), by_half(half), by_mass(mass);
        // with these within 2^+-60 and vrel >= 1e-7, re, cd (24 / 1e-20 at most) and
        // the quotients of 3 cd / 8 stay within 2^+-200; a re that overflows on the
        // way has a drag of 0.44 as it is or as a NaN
        const bool quick = Divisor::safe(dpp) && Divisor::safe(nupp) && Divisor::safe(mass);
        const double sigx = (1.0 - gama) / mass * P.gx, sigy = (1.0 - gama) / mass * P.gy;
        for (int itep = 1; itep <= ITP; ++itep) {
            if (fluid) {
                double vrel = sqrt((upo - ug) * (upo - ug) + (vpo - vg) * (vpo - vg));
                if (vrel < 1.0e-7) vrel = 1.0e-7;
                const double reyp = quick ? by_nu(dpp * vrel) : dpp * vrel / nupp;
                const double cd = drag(reyp);
                const double c0 = 3.0 * cd / 8.0;
                const double ck = quick ? by_mass(by_half(c0)) : c0 / half / mass;
                const double mag = sqrt((upo - ug) * (upo - ug) + (vpo - vg) * (vpo - vg));
                const double axp = sigx - ck * (upo - ug) * mag;
                const double beta = ck * mag;
                const double e = exp(-beta * dtp);
                const double upn = upo * e + ug * (1.0 - e) + sigx / beta * (1.0 - e);
                xx = xx + 0.5 * (upn + upo) * dtp;
                const double vpn = vpo * e + vg * (1.0 - e) + sigy / beta * (1.0 - e);
                yy = yy + 0.5 * (vpn + vpo) * dtp;
                if (isnan(upo) || fabs(xx) > 1.0e10 || fabs(axp) > 1.0e10 || isnan(upn) || isnan(vpn)) bad = true;
                upo = upn;
                vpo = vpn;
            } else if (s > 1.0 - EPSI) {
                const double upn = P.us, vpn = P.vs;
                xx = xx + 0.5 * (upn + upo) * dtp;
                yy = yy + 0.5 * (vpn + vpo) * dtp;
                upo = upn;
                vpo = vpn;
            } else {
                xx = 1.0e3;
                yy = 1.0e3;
            }
        }
    }
    if (in) {
        px[p] = xx;
        py[p] = yy;
        pu[p] = upo;
        pv[p] = vpo;
    }
    // a workgroup's count goes straight to the host's array, which it zeroes
    // before the launch: usually there is none, and nothing to write or copy
    const int nbad = __syncthreads_count(in && bad);
    if (nbad && threadIdx.x == 0) flagged[blockIdx.x] = (unsigned)nbad;
}

constexpr int PART_NT = 256;
int part_blocks(int n) { return (n + PART_NT - 1) / PART_NT; }

}  // namespace

int particles_reserve(Ctx* c, int n) {
    ParticleState& S = c->part;
    if (n <= S.cap) return SG_OK;
    // grows only; earlier buffers are released with the context
    const size_t b = (size_t)n * sizeof(double);
    double* a[5];
    bool ok = true;
    for (double*& p : a) ok = (p = (double*)dev_alloc(c, b)) != nullptr && ok;
    unsigned* flagged = nullptr;
    ok = ok && hipHostMalloc((void**)&flagged, (size_t)part_blocks(n) * sizeof(unsigned), hipHostMallocDefault) ==
                   hipSuccess;
    if (!ok) {
        set_error("particle buffers: device allocation failed");
        return SG_ERR_ALLOC;
    }
    if (S.flagged) {
        // a launch may still write the old counts
        const hipError_t e = hipStreamSynchronize(c->stream);
        (void)hipHostFree(S.flagged);
        S.flagged = nullptr;
        if (e != hipSuccess) (void)hipHostFree(flagged);
        SG_HIP(e);
    }
    S.x = a[0];
    S.y = a[1];
    S.u = a[2];
    S.v = a[3];
    S.d = a[4];
    S.flagged = flagged;
    S.cap = n;
    return SG_OK;
}

int particles_launch(Ctx* c, double dt, const sg_particle_params* prm) {
    ParticleState& S = c->part;
    if (S.n == 0) return SG_OK;
    const PGeo G{c->ni,
                 c->nj,
                 c->cls.xc,
                 c->cls.yc,
                 c->dx,
                 c->dy,
                 (const double*)c->field[SG_F_VOF],
                 (const double*)c->field[SG_F_VOFS],
                 (const double*)c->field[SG_F_U],
                 (const double*)c->field[SG_F_V]};
    hipStream_t s = c->stream;
    hipLaunchKernelGGL(k_particles, dim3((unsigned)part_blocks(S.n)), dim3(PART_NT), 0, s, G, S.n, S.x, S.y, S.u, S.v,
                       (const double*)S.d, *prm, dt, S.flagged);
    SG_HIP(hipGetLastError());
    S.last = *prm;
    S.last_dt = dt;
    S.tracked = true;
    return SG_OK;
}

int particles_track(Ctx* c, double dt, const sg_particle_params* prm, int* flagged) {
    ParticleState& S = c->part;
    if (flagged) *flagged = 0;
    if (S.n == 0) return SG_OK;
    // (nothing on the stream writes the counts: every tracking call waits for its own)
    const int nb = part_blocks(S.n);
    std::fill(S.flagged, S.flagged + nb, 0u);
    const int rc = particles_launch(c, dt, prm);
    if (rc) return rc;
    SG_HIP(hipStreamSynchronize(c->stream));
    unsigned h = 0;
    for (int b = 0; b < nb; ++b) h += S.flagged[b];
    if (flagged) *flagged = (int)h;
    return SG_OK;
}

}  // namespace sg
