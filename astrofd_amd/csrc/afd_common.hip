// afd_common.hip -- stage update / rhs kernels and the RMHD face dispatcher.
#include "afd_launch.hpp"

namespace afd {

// ------------------------------------------------------------------ non-template kernels
// Which right-face variants the reference subtracts per direction, in the order WENO5 (bit 0), PPM
// (bit 1), MUSCL (bit 2), and which variant's left flux survives; no variant: the direction has no term.
enum { PASS_RMHD_MUSCL, PASS_SRHD_MUSCL, PASS_SRHD_PPM };
template <int MODE> constexpr int pass_right(int dir) {
    return MODE == PASS_RMHD_MUSCL ? 7 : (MODE == PASS_SRHD_MUSCL ? (dir == 0 ? 7 : (dir == 1 ? 0 : 4))
                                                                  : (dir == 0 ? 0 : (dir == 1 ? 7 : 3)));
}
template <int MODE> constexpr int pass_left(int dir) { return MODE == PASS_SRHD_PPM && dir == 2 ? 1 : 2; }

template <int MODE, int DIR>
AFD_D void passive_dir(const PassiveArgs &a, const double *__restrict__ b, long c, const int *ijk, double &r) {
#pragma clang fp contract(off)
    constexpr int right = pass_right<MODE>(DIR);
    if constexpr (right != 0) {
        const Grid &g = a.g;
        constexpr bool wide = (right & 3) != 0;  // WENO5 and PPM reach one cell further than MUSCL
        const long s = dstride<DIR>(g);
        const int n = DIR == 0 ? g.nx : (DIR == 1 ? g.ny : g.nz);
        double q[7];
#pragma unroll
        for (int o = -3; o <= 3; ++o)
            q[o + 3] = wide || (o >= -2 && o <= 2) ? b[c + pwrap(ijk[DIR], o, n) * s] : 0.0;
        const double *ax = a.aux[DIR];
        const long cp = c + s;
        const double sLa = ax[c], sRa = ax[g.ncell + c], vLa = ax[2 * g.ncell + c], vRa = ax[3 * g.ncell + c];
        const double vLb = ax[2 * g.ncell + cp], vRb = ax[3 * g.ncell + cp];
        double sLb = sLa, sRb = sRa;
        if (MODE != PASS_RMHD_MUSCL) {  // RMHD: right faces keep the left face's speeds (core/rmhd_core.py:915)
            sLb = ax[cp];
            sRb = ax[g.ncell + cp];
        }
        const Div<double> by(a.d[DIR]);
        const double FL = passive_flux<pass_left<MODE>(DIR)>(a.lim, q, vLa, vRa, sLa, sRa);
        if (right & 1) r -= by(passive_flux<0>(a.lim, q + 1, vLb, vRb, sLb, sRb) - FL);
        if (right & 2) r -= by(passive_flux<1>(a.lim, q + 1, vLb, vRb, sLb, sRb) - FL);
        if (right & 4) r -= by(passive_flux<2>(a.lim, q + 1, vLb, vRb, sLb, sRb) - FL);
    }
}

template <int MODE> __global__ __launch_bounds__(BLOCK) void k_passives(PassiveArgs a) {
#pragma clang fp contract(off)
    const Grid &g = a.g;
    const long c = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= g.ncell) return;
    const int t = blockIdx.y;
    int ijk[3];
    cell_ijk(g, c, ijk[0], ijk[1], ijk[2]);
    double r = 0.0;
    if (in_range(g, c)) {
        const double *b = a.P + (a.po + t) * g.ncell;
        passive_dir<MODE, 0>(a, b, c, ijk, r);
        passive_dir<MODE, 1>(a, b, c, ijk, r);
        passive_dir<MODE, 2>(a, b, c, ijk, r);
    }
    const long o = t * g.ncell + c;
    if (a.nst == 0) {
        a.out[o] = r;
    } else {
        const double dr = a.dt * r;
        a.out[o] = ssprk_combine(a.stage, a.nst, a.P0[o], a.Pin[o], dr);
    }
}

// physics and recon: a context with passive fluxes (RMHD MUSCL, SRHD MUSCL or PPM)
hipError_t launch_passives(const PassiveArgs &a, bool rmhd, int recon, hipStream_t s) {
    const dim3 grid(grid1d(a.g.ncell).x, (unsigned)a.np);
    if (rmhd) hipLaunchKernelGGL(k_passives<PASS_RMHD_MUSCL>, grid, dim3(BLOCK), 0, s, a);
    else if (recon == 0) hipLaunchKernelGGL(k_passives<PASS_SRHD_MUSCL>, grid, dim3(BLOCK), 0, s, a);
    else hipLaunchKernelGGL(k_passives<PASS_SRHD_PPM>, grid, dim3(BLOCK), 0, s, a);
    return hipGetLastError();
}

// RMHD: bound by FP64 instructions of waves with few live lanes.  A tenth of a batch of wide-ranging states
// goes all the way (50 Newton steps from each start, then the bisection: 300 evaluations of f, against about
// 11 for the rest), and where it lies keeps nearly every wave running.  So a state that PACK_AFTER steps
// (twice the mean of those that end) have not brought home goes through LDS to the workgroup's first free
// thread, and one wave of four takes the rest of the way.  The operations of a state do not depend on the
// thread.  150001 states: 405 -> 210 us.
constexpr int PACK_AFTER = 12;

__global__ __launch_bounds__(BLOCK) void k_c2p_batch(BatchArgs a) {
    const long m = (long)blockIdx.x * BLOCK + threadIdx.x;
    C2PStats st = {0, 0, 0};
    const bool count = a.iters || a.stats;
    if (a.physics == 1) {
        __shared__ double Zs[BLOCK];
        __shared__ RmhdRoot roots[BLOCK];
        __shared__ int steps[BLOCK], flags[BLOCK], packed;
        if (threadIdx.x == 0) packed = 0;
        __syncthreads();
        const RmhdC2PParams cp = {a.gamma, a.gfac, a.p_max, a.v_max};
        double q0[5], Z = 0.0;
        RmhdRoot r;
        int slot = -1;
        if (m < a.n) {
            double U[9];
            for (int v = 0; v < 9; ++v) U[v] = a.in[9 * m + v];
            Z = rmhd_c2p_start(cp, U, q0, r, st, count);
            int it = 0;
            if (!rmhd_newton_steps(cp, Z, r.D, r.tau, r.B2, r.SB, r.S2, r.tol(), it, PACK_AFTER, RMHD_NEWTON_STEPS, st)) {
                slot = atomicAdd(&packed, 1);
                Zs[slot] = Z;
                roots[slot] = r;
                steps[slot] = it;
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < packed) {
            const RmhdRoot w = roots[threadIdx.x];
            C2PStats sw = {0, 0, 0};
            double Zw = Zs[threadIdx.x];
            int it = steps[threadIdx.x];
            if (!rmhd_newton_steps(cp, Zw, w.D, w.tau, w.B2, w.SB, w.S2, w.tol(), it, RMHD_NEWTON_STEPS,
                                   RMHD_NEWTON_STEPS, sw))
                Zw = rmhd_c2p_second(cp, w, sw);
            Zs[threadIdx.x] = Zw;
            steps[threadIdx.x] = sw.newton_iters;
            flags[threadIdx.x] = sw.flags;
        }
        __syncthreads();
        if (slot >= 0) {
            Z = Zs[slot];
            st.newton_iters += steps[slot];
            st.flags |= flags[slot];
        }
        if (m < a.n) {
            double U[9], q[9];
            for (int v = 0; v < 9; ++v) U[v] = a.in[9 * m + v];
            rmhd_recover(cp, Z, U, r.B2, r.SB, q0, q, st);
            for (int v = 0; v < 9; ++v) a.out[9 * m + v] = q[v];
        }
    } else if (m < a.n) {
        double U[5], q[5];
        for (int v = 0; v < 5; ++v) U[v] = a.in[5 * m + v];
        hydro_c2p(a.gamma, a.gfac, a.p_max, a.v_max, U, q, st, count);
        for (int v = 0; v < 5; ++v) a.out[5 * m + v] = q[v];
    }
    if (a.iters && m < a.n) a.iters[m] = st.hydro_iters + st.newton_iters;
    if (a.stats) wave_add_stats(a.stats, st);  // reached by every lane
}

__global__ __launch_bounds__(BLOCK) void k_p2c_batch(BatchArgs a) {
    long m = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (m >= a.n) return;
    if (a.physics == 1) {
        double q[9], U[9];
        for (int v = 0; v < 9; ++v) q[v] = a.in[9 * m + v];
        rmhd_p2c_cell(a.gfac, a.p_max, a.v_max, q, U);
        for (int v = 0; v < 9; ++v) a.out[9 * m + v] = U[v];
    } else {
        double q[5], U[5];
        for (int v = 0; v < 5; ++v) q[v] = a.in[5 * m + v];
        srhd_p2c_cell(a.gfac, q, U);
        for (int v = 0; v < 5; ++v) a.out[5 * m + v] = U[v];
    }
}

__global__ __launch_bounds__(BLOCK) void k_fill_y(BcArgs a) {
#pragma clang fp contract(off)
    const Grid &g = a.g;
    long t = (long)blockIdx.x * BLOCK + threadIdx.x;
    long tot = (long)g.nv * g.nx * 2 * a.ng * g.nz;
    if (t >= tot) return;
    int k = (int)(t % g.nz);
    long r = t / g.nz;
    int gg = (int)(r % (2 * a.ng));
    r /= 2 * a.ng;
    int i = (int)(r % g.nx);
    int v = (int)(r / g.nx);
    int jd, js;
    if (gg < a.ng) {
        jd = gg;
        js = a.bc ? a.ng : g.ny - 2 * a.ng + gg;
    } else {
        jd = g.ny - a.ng + (gg - a.ng);
        js = a.bc ? g.ny - a.ng - 1 : a.ng + (gg - a.ng);
    }
    double *b = a.P + (long)v * g.ncell;
    b[cidx(g, i, jd, k)] = b[cidx(g, i, js, k)];
}

__global__ __launch_bounds__(BLOCK) void k_fill_z(BcArgs a) {
    const Grid &g = a.g;
    long t = (long)blockIdx.x * BLOCK + threadIdx.x;
    long tot = (long)g.nv * g.nx * g.ny * 2 * a.ng;
    if (t >= tot) return;
    int gg = (int)(t % (2 * a.ng));
    long r = t / (2 * a.ng);
    int j = (int)(r % g.ny);
    r /= g.ny;
    int i = (int)(r % g.nx);
    int v = (int)(r / g.nx);
    int kd, ks;
    if (gg < a.ng) {
        kd = gg;
        ks = a.bc ? a.ng : g.nz - 2 * a.ng + gg;
    } else {
        kd = g.nz - a.ng + (gg - a.ng);
        ks = a.bc ? g.nz - a.ng - 1 : a.ng + (gg - a.ng);
    }
    double *b = a.P + (long)v * g.ncell;
    b[cidx(g, i, j, kd)] = b[cidx(g, i, j, ks)];
}

__global__ __launch_bounds__(BLOCK) void k_outflow_x(BcArgs a) {
    const Grid &g = a.g;
    long t = (long)blockIdx.x * BLOCK + threadIdx.x;
    long plane = (long)g.ny * g.nz;
    long tot = (long)g.nv * a.ng * plane;
    if (t >= tot) return;
    long jk = t % plane;
    long r = t / plane;
    int gi = (int)(r % a.ng);
    int v = (int)(r / a.ng);
    double *b = a.P + (long)v * g.ncell;
    b[(long)(g.nx - a.ng + gi) * plane + jk] = b[(long)(g.nx - a.ng - 1) * plane + jk];
}

// The nozzle's value of variable v in cell c, ghost plane gi and interior (j, k) number jk
AFD_D void nozzle_value(const NozzleArgs &a, int v, long c, int gi, unsigned jk, unsigned plane) {
#pragma clang fp contract(off)
    if (v >= 32 || !((a.mask >> v) & 1u)) return;
    double val = a.tmpl[(long)v * plane + jk];
    int rank = a.idx[jk];
    if (a.perturb && rank >= 0 && v >= 2 && v <= 4) {
        const double *d = a.draws + 3 * ((long)gi * a.nact + rank);
        if (v == 2) val = val + a.vamp * (2.0 * d[0] - 1.0);
        else if (v == 3) val = val + a.vamp * (2.0 * d[1] - 1.0);
        else val = val * (1.0 + a.pamp * (2.0 * d[2] - 1.0));
    }
    a.P[(long)v * a.g.ncell + c] = val;
}

__global__ __launch_bounds__(BLOCK) void k_nozzle(NozzleArgs a) {
    const Grid &g = a.g;
    const unsigned t = blockIdx.x * BLOCK + threadIdx.x, plane = (unsigned)a.ny_int * a.nz_int;
    if (t >= (unsigned)a.ng * plane) return;
    const unsigned gi = t / plane, jk = t - gi * plane, jj = jk / a.nz_int;
    const long c = cidx(g, (int)gi, a.ng + (int)jj, a.ng + (int)(jk - jj * a.nz_int));
    for (int v = 0; v < g.nv && v < 32; ++v) nozzle_value(a, v, c, (int)gi, jk, plane);
}

// Source index of the y or z fill at position j of an axis of n cells (interior positions: j)
AFD_D int fill_source(int j, int n, int ng, int bc) {
    if (j < ng) return bc ? ng : n - 2 * ng + j;
    if (j >= n - ng) return bc ? n - ng - 1 : ng + (j - (n - ng));
    return j;
}
AFD_D int ghost_pos(int a, int n, int ng) { return a < ng ? a : n - 2 * ng + a; }  // ghost a of 2 ng

// The ghost positions filled from interior position j: [lo0, lo1) and [hi0, hi1)
struct Images {
    int lo0, lo1, hi0, hi1;
};
AFD_D Images fill_images(int j, int n, int ng, int bc) {
    const int m = n - 2 * ng;  // interior cells
    if (bc) return Images{0, j == ng ? ng : 0, n - ng, j == n - ng - 1 ? n : n - ng};
    return Images{j - m, j - m + (j >= m ? 1 : 0), j + m, j + m + (j < 2 * ng ? 1 : 0)};
}

__global__ __launch_bounds__(BLOCK) void k_fill_ghosts(FillArgs a) {
    const Grid &g = a.n.g;
    const int ng = a.n.ng;
    double *P = a.n.P;
    if (blockIdx.x < a.bA) {
        const unsigned t = blockIdx.x * BLOCK + threadIdx.x;
        if (t >= a.nA) return;
        const unsigned q = udiv(a.ring, t), rows = 2u * ng * g.nz;
        unsigned r = t - q * (rows + 2u * ng * a.n.ny_int);
        const int first = a.nozzle ? ng : 0, ni = g.nx - ng - first;
        const unsigned v = udiv(a.ni, q);
        const int i = first + (int)(q - v * ni);
        int j, k;
        if (r < rows) {
            const unsigned gj = udiv(g.dnz, r);
            k = (int)(r - gj * g.nz);
            j = ghost_pos((int)gj, g.ny, ng);
        } else {
            r -= rows;
            const unsigned jj = udiv(a.ng2, r);
            k = ghost_pos((int)(r - jj * 2u * ng), g.nz, ng);
            j = ng + (int)jj;
        }
        double *b = P + (long)v * g.ncell;
        b[cidx(g, i, j, k)] = b[cidx(g, i, fill_source(j, g.ny, ng, a.bc_y), fill_source(k, g.nz, ng, a.bc_z))];
    } else if (blockIdx.x < a.bA + a.bB) {
        const unsigned t = (blockIdx.x - a.bA) * BLOCK + threadIdx.x;
        if (t >= a.nB) return;
        const unsigned q = udiv(a.plane, t), jk = t - q * (unsigned)g.sx, v = udiv(a.ng, q), ju = udiv(g.dnz, jk);
        const int i = g.nx - ng + (int)(q - v * ng), j = (int)ju, k = (int)(jk - ju * g.nz);
        double *b = P + (long)v * g.ncell;
        b[cidx(g, i, j, k)] =
            b[cidx(g, g.nx - ng - 1, fill_source(j, g.ny, ng, a.bc_y), fill_source(k, g.nz, ng, a.bc_z))];
    } else {
        const unsigned t = (blockIdx.x - a.bA - a.bB) * BLOCK + threadIdx.x;
        if (t >= a.nC) return;
        const unsigned plane = (unsigned)a.n.ny_int * a.n.nz_int, q = udiv(a.plane_int, t), jk = t - q * plane;
        const unsigned v = udiv(a.ng, q), jj = udiv(a.nz_int, jk);
        const int i = (int)(q - v * ng), j = ng + (int)jj, k = ng + (int)(jk - jj * a.n.nz_int);
        const long c = cidx(g, i, j, k);
        if (j < 2 * ng || j >= g.ny - 2 * ng || k < 2 * ng || k >= g.nz - 2 * ng) {
            double *b = P + (long)v * g.ncell;
            const double old = b[c];
            const Images y = fill_images(j, g.ny, ng, a.bc_y), z = fill_images(k, g.nz, ng, a.bc_z);
            auto row = [&](int jd, bool own) {
                for (int kd = z.lo0; kd < z.lo1; ++kd) b[cidx(g, i, jd, kd)] = old;
                for (int kd = z.hi0; kd < z.hi1; ++kd) b[cidx(g, i, jd, kd)] = old;
                if (!own) b[cidx(g, i, jd, k)] = old;
            };
            row(j, true);
            for (int jd = y.lo0; jd < y.lo1; ++jd) row(jd, false);
            for (int jd = y.hi0; jd < y.hi1; ++jd) row(jd, false);
        }
        nozzle_value(a.n, (int)v, c, i, jk, plane);
    }
}

// core/chemistry.py:17-27: collisional ionization fit, T in K
__device__ static double rate_ci(double a, double e, double T) {
#pragma clang fp contract(off)
    return a * sqrt(T) * exp(-e / pymax(T, 1.0)) / (1.0 + sqrt(T / 1.0e5));
}

__device__ static double clamp01(double x, double lo, double hi) { return x < lo ? lo : (x > hi ? hi : x); }

__global__ __launch_bounds__(BLOCK) void k_sources(SourceArgs a) {
#pragma clang fp contract(off)
    const Grid &g = a.g;
    int i, j, k;
    if (!interior_cell(g, a.in, i, j, k)) return;
    const long c = cidx(g, i, j, k), n = g.ncell;
    double *P = a.P;
    const double rho = P[c];
    double p = P[4 * n + c];
    if (a.which & SRC_COOL) {  // core/source_terms.py:19-27
        double p_new = p + a.dt * (a.heat - a.cool * rho * p);
        if (p_new < 1e-12) p_new = 1e-12;
        if (p_new > a.p_cap) p_new = a.p_cap;
        p = p_new;
        P[4 * n + c] = p;
    }
    if (a.which & SRC_TWO_TEMP) {  // core/source_terms.py:45-54
        double T = p / pymax(rho, 1e-12);
        double *Te = P + (long)a.t_off * n + c, *Ti = Te + n;
        double te = *Te, ti = *Ti;
        te += a.dt * (T - te) / a.tau;
        ti += a.dt * (T - ti) / a.tau;
        *Te = te;
        *Ti = ti;
    }
    if ((a.which & SRC_CHEM) && rho > 0.0 && p > 0.0) {  // core/chemistry.py:78-137
        const double SM = 1e-20;
        double T = (p / pymax(rho, SM)) * a.tunit;
        if (T < a.tmin) T = a.tmin;
        double nH = a.X * rho, nHe = a.Y * rho / 4.0;
        double *x = P + (long)a.c_off * n + c;
        double xHII = clamp01(x[0], 0.0, 1.0), xHeII = clamp01(x[n], 0.0, 1.0), xHeIII = clamp01(x[2 * n], 0.0, 1.0);
        xHeII = pymin(xHeII, 1.0 - xHeIII);
        double xHeI = pymax(0.0, 1.0 - xHeII - xHeIII);
        double xHI = 1.0 - xHII;
        double ne = pymax(nH * xHII + nHe * (xHeII + 2.0 * xHeIII), SM);
        double C_H = a.rate_scale * rate_ci(5.85e-11, 157809.1, T);
        double C_HeI = a.rate_scale * rate_ci(2.38e-11, 285335.4, T);
        double C_HeII = a.rate_scale * rate_ci(5.68e-12, 631515.0, T);
        // case-B recombination, core/chemistry.py:30-40: (T / 1e4)^y as exp(y log(T / 1e4)), one
        // log for the three powers; |y log| <= ~20 over T in [1, 1e12] K, so the result is within
        // ~20 ulp of the correctly rounded power
        double lt4 = log(T / 1.0e4);
        double A_H = a.rate_scale * (2.59e-13 * exp(-0.7 * lt4));
        double A_HeII = a.rate_scale * (1.50e-10 * exp(-0.6353 * lt4));
        double A_HeIII = a.rate_scale * (3.36e-10 * exp(-0.5 * lt4));
        double dne = a.dt * ne;
        double xHII_new = (xHII + dne * C_H * xHI) / (1.0 + dne * A_H);
        double xHeIII_new = clamp01((xHeIII + dne * C_HeII * xHeII) / (1.0 + dne * A_HeIII), 0.0, 1.0);
        double xHeII_new = (xHeII + dne * (C_HeI * xHeI + A_HeIII * xHeIII_new)) / (1.0 + dne * (A_HeII + C_HeII));
        xHII_new = clamp01(xHII_new, 0.0, 1.0);
        xHeII_new = clamp01(xHeII_new, 0.0, 1.0 - xHeIII_new);
        double dE = a.energy_scale * (nH * 157809.1 * (xHII_new - xHII) + nHe * 285335.4 * (xHeII_new - xHeII) +
                                      nHe * 631515.0 * (xHeIII_new - xHeIII));
        double p_new = p + -(a.gamma - 1.0) * dE / pymax(a.tunit, SM);
        if (p_new < SM) p_new = SM;
        P[4 * n + c] = p_new;
        x[0] = xHII_new;
        x[n] = xHeII_new;
        x[2 * n] = xHeIII_new;
    }
}

__global__ __launch_bounds__(BLOCK) void k_diss(DissArgs a) {
#pragma clang fp contract(off)
    const Grid &g = a.g;
    int i, j, k;
    if (!interior_cell(g, a.in, i, j, k)) return;
    const long c = cidx(g, i, j, k), n = g.ncell, sx = g.sx, sy = g.sy;
    const double *P = a.P;
    double f[10];
#pragma unroll
    for (int m = 0; m < 10; ++m) f[m] = P[(5 + m) * n + c];
    const double vx = P[n + c], vy = P[2 * n + c], vz = P[3 * n + c];
    if (a.advect) {  // core/dissipation.py:60-92, first-order upwind with the cell's velocity
        const Div<double> hx(pymax(a.dx, 1e-12)), hy(pymax(a.dy, 1e-12)), hz(pymax(a.dz, 1e-12));
        const long ox = vx > 0.0 ? -sx : sx, oy = vy > 0.0 ? -sy : sy, oz = vz > 0.0 ? -1 : 1;
#pragma unroll
        for (int m = 0; m < 10; ++m) {
            const double *q = P + (5 + m) * n + c;
            const double u0 = f[m];
            double dudx = hx(vx > 0.0 ? u0 - q[ox] : q[ox] - u0);
            double dudy = hy(vy > 0.0 ? u0 - q[oy] : q[oy] - u0);
            double dudz = hz(vz > 0.0 ? u0 - q[oz] : q[oz] - u0);
            f[m] = u0 - a.dt * (vx * dudx + vy * dudy + vz * dudz);
        }
    }
    const double i2x = 0.5 / pymax(a.dx, 1e-12), i2y = 0.5 / pymax(a.dy, 1e-12), i2z = 0.5 / pymax(a.dz, 1e-12);
    const double *V1 = P + n + c, *V2 = P + 2 * n + c, *V3 = P + 3 * n + c;
    const double dvx_dx = (V1[sx] - V1[-sx]) * i2x, dvx_dy = (V1[sy] - V1[-sy]) * i2y, dvx_dz = (V1[1] - V1[-1]) * i2z;
    const double dvy_dx = (V2[sx] - V2[-sx]) * i2x, dvy_dy = (V2[sy] - V2[-sy]) * i2y, dvy_dz = (V2[1] - V2[-1]) * i2z;
    const double dvz_dx = (V3[sx] - V3[-sx]) * i2x, dvz_dy = (V3[sy] - V3[-sy]) * i2y, dvz_dz = (V3[1] - V3[-1]) * i2z;
    const double divv = dvx_dx + dvy_dy + dvz_dz;
    const double cap = a.cap;
    auto clamp = [cap](double x) { return x > cap ? cap : (x < -cap ? -cap : x); };
    if (a.zeta != 0.0) {  // bulk, :122-130
        double pi_eq = -a.zeta * divv;
        const Div<double> tau(a.tau_bulk), den(1.0 + tau(a.dt));
        f[0] = clamp(den(f[0] + tau(a.dt * pi_eq)));
    }
    if (a.eta != 0.0) {  // shear, :132-177 (pi^zz reset to -(pi^xx + pi^yy) before the caps)
        const double third = 1.0 / 3.0, m2e = -2.0 * a.eta;
        const Div<double> tau(a.tau_shear), den(1.0 + tau(a.dt));
        const double e[6] = {m2e * (dvx_dx - third * divv), m2e * (dvy_dy - third * divv),
                             m2e * (dvz_dz - third * divv), m2e * (0.5 * (dvx_dy + dvy_dx)),
                             m2e * (0.5 * (dvx_dz + dvz_dx)), m2e * (0.5 * (dvy_dz + dvz_dy))};
        double s6[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) s6[m] = den(f[1 + m] + tau(a.dt * e[m]));
        s6[2] = -(s6[0] + s6[1]);
#pragma unroll
        for (int m = 0; m < 6; ++m) f[1 + m] = clamp(s6[m]);
    }
    if (a.kappa != 0.0) {  // heat flux, :179-213, T = p / max(rho, 1e-12)
        const double *R = P + c, *Pp = P + 4 * n + c;
        const Div<double> tau(a.tau_heat), den(1.0 + tau(a.dt));
        auto T = [&](long o) { return fdiv(Pp[o], pymax(R[o], 1e-12)); };
        const double g3[3] = {(T(sx) - T(-sx)) * i2x, (T(sy) - T(-sy)) * i2y, (T(1) - T(-1)) * i2z};
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            double q_eq = -a.kappa * g3[m];
            f[7 + m] = clamp(den(f[7 + m] + tau(a.dt * q_eq)));
        }
    }
#pragma unroll
    for (int m = 0; m < 10; ++m) a.S[m * n + c] = f[m];
}

__global__ __launch_bounds__(BLOCK) void k_diss_store(DissArgs a, double *P) {
    const Grid &g = a.g;
    int i, j, k;
    if (!interior_cell(g, a.in, i, j, k)) return;
    const long c = cidx(g, i, j, k), n = g.ncell;
#pragma unroll
    for (int m = 0; m < 10; ++m) P[(5 + m) * n + c] = a.S[m * n + c];
}

__global__ __launch_bounds__(BLOCK) void k_gr_rescale(GrRescaleArgs a) {
#pragma clang fp contract(off)
    const Grid &g = a.g;
    const long c = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= g.ncell) return;
    const long n = g.ncell;
    for (int v = 0; v < g.nv; ++v) a.Q[v * n + c] = a.P[v * n + c];
    int i, j, k;
    cell_ijk(g, c, i, j, k);
    if (i < a.ng || i >= g.nx - a.ng || j < a.ng || j >= g.ny - a.ng || k < a.ng || k >= g.nz - a.ng) return;
    double X[3];
    gr_xyz(a.x0, a.ng, i, j, k, a.dx, a.dy, a.dz, X);
    const double ax = pymax(gr_ks_alpha(X[0], X[1], X[2], a.mass), 1e-12);
    for (int v = 1; v <= 3; ++v) a.Q[v * n + c] = a.P[v * n + c] / ax;
}

__global__ __launch_bounds__(BLOCK) void k_max_speed_box(const double *P, Grid g, SpeedBox b, double gamma,
                                                          double gfac, unsigned long long *amax) {
    const long ni = b.hi[0] - b.lo[0], nj = b.hi[1] - b.lo[1], nk = b.hi[2] - b.lo[2], tot = ni * nj * nk;
    double m = 0.0;
    for (long t = (long)blockIdx.x * BLOCK + threadIdx.x; t < tot; t += (long)gridDim.x * BLOCK) {
        const int k = b.lo[2] + (int)(t % nk), j = b.lo[1] + (int)((t / nk) % nj), i = b.lo[0] + (int)(t / (nj * nk));
        const long c = cidx(g, i, j, k);
        const double loc = srhd_cell_speed(gamma, gfac, P[c], P[g.ncell + c], P[2 * g.ncell + c],
                                           P[3 * g.ncell + c], P[4 * g.ncell + c]);
        if (loc > m) m = loc;
    }
    wave_max_atomic(amax, m);
}

__global__ __launch_bounds__(BLOCK) void k_max_speed_shell(const double *P, Grid g, SpeedBox b, double gamma,
                                                            double gfac, unsigned long long *amax) {
    // range [1, n-1) per axis, box [lo, hi) inside it: slabs i outside (all j, k), then i inside
    // with j outside (all k), then i, j inside with k outside
    const unsigned bi = g.nx - 2, bj = g.ny - 2, bk = g.nz - 2;
    const unsigned ni = b.hi[0] - b.lo[0], nj = b.hi[1] - b.lo[1], nk = b.hi[2] - b.lo[2];
    const unsigned oi = bi - ni, oj = bj - nj, ok = bk - nk;
    const unsigned nA = oi * bj * bk, nB = ni * oj * bk, nC = ni * nj * ok;
    unsigned t = blockIdx.x * BLOCK + threadIdx.x;
    double v = 0.0;
    if (t < nA + nB + nC) {
        auto out_pos = [&](unsigned p, int ax) {
            return (int)p < b.lo[ax] - 1 ? 1 + (int)p : b.hi[ax] + ((int)p - (b.lo[ax] - 1));
        };
        int i, j, k;
        if (t < nA) {
            const unsigned r = t / bk, q = r / bj;
            k = 1 + (int)(t - r * bk);
            j = 1 + (int)(r - q * bj);
            i = out_pos(q, 0);
        } else if (t < nA + nB) {
            t -= nA;
            const unsigned r = t / bk, q = r / oj;
            k = 1 + (int)(t - r * bk);
            j = out_pos(r - q * oj, 1);
            i = b.lo[0] + (int)q;
        } else {
            t -= nA + nB;
            const unsigned r = t / ok, q = r / nj;
            k = out_pos(t - r * ok, 2);
            j = b.lo[1] + (int)(r - q * nj);
            i = b.lo[0] + (int)q;
        }
        const long c = cidx(g, i, j, k);
        v = srhd_cell_speed(gamma, gfac, P[c], P[g.ncell + c], P[2 * g.ncell + c], P[3 * g.ncell + c],
                            P[4 * g.ncell + c]);
    }
    wave_max_atomic(amax, v);
}

__global__ __launch_bounds__(BLOCK) void k_amax_finish(unsigned long long *amax, double floor_value, double *out) {
    __shared__ double red[BLOCK / 64];
    double m = 0.0;
    for (int t = threadIdx.x; t < 2 * AMAX_SLOTS; t += BLOCK) {
        unsigned long long *slot = amax + (long)t * AMAX_STRIDE;
        m = pymax(m, __longlong_as_double((long long)*slot));
        if (t >= AMAX_SLOTS) *slot = 0ull;  // each shell slot is read and cleared by this thread only
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = pymax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLOCK / 64; ++w) m = pymax(m, red[w]);
        out[0] = m < floor_value ? floor_value : m;
    }
}

__global__ __launch_bounds__(BLOCK) void k_count_nonfinite(const double *x, long n, unsigned long long *partial) {
    __shared__ unsigned long long red[BLOCK];
    unsigned long long cnt = 0;
    for (long t = (long)blockIdx.x * BLOCK + threadIdx.x; t < n; t += (long)gridDim.x * BLOCK)
        cnt += isfinite(x[t]) ? 0ull : 1ull;
    red[threadIdx.x] = cnt;
    __syncthreads();
    for (int o = BLOCK / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(BLOCK) void k_reduce_sum_u64(const unsigned long long *partial, int n,
                                                           unsigned long long *out) {
    __shared__ unsigned long long red[BLOCK];
    unsigned long long m = 0;
    for (int t = threadIdx.x; t < n; t += BLOCK) m += partial[t];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = BLOCK / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

template <typename T>
void launch_face_rmhd_t(const FaceLaunch &l, const FaceLaunch *y, const FaceLaunch *z, hipStream_t s);

hipError_t launch_face_rmhd(const FaceLaunch &l, const FaceLaunch *y, const FaceLaunch *z, hipStream_t s) {
    if (l.mixed) launch_face_rmhd_t<float>(l, y, z, s);
    else launch_face_rmhd_t<double>(l, y, z, s);
    return hipGetLastError();
}

// One stage update: k_update (flux divergence, SSPRK, con2prim).  With a Newton start other than
// the plain one, rejected cells are queued and solved densely by k_c2p_queue afterwards.
template <typename F, bool LEARNED> static void upd_stage(const UpdArgs<F> &a, dim3 grid, hipStream_t s) {
    if (a.queue) (void)hipMemsetAsync(a.qcount, 0, sizeof(unsigned) * QUEUE_SLOTS, s);
    k_update<9, F, LEARNED><<<grid, dim3(BLOCK), 0, s>>>(a);
    if (a.queue) hipLaunchKernelGGL((k_c2p_queue<F>), dim3(16, QUEUE_SLOTS), dim3(BLOCK), 0, s, a);
}

template <typename F> static void upd(const UpdLaunch &l, bool rhs_only, hipStream_t s) {
    UpdArgs<F> a;
    static_assert(sizeof(UpdArgs<F>) == sizeof(UpdArgs<double>), "layout");
    memcpy((void *)&a, (const void *)&l.a, sizeof(a));
    dim3 grid = grid1d(l.a.g.ncell);
    if (rhs_only) hipLaunchKernelGGL((k_rhs<9, F>), grid, dim3(BLOCK), 0, s, a);
    else if (l.a.mlp) upd_stage<F, true>(a, grid, s);
    else upd_stage<F, false>(a, grid, s);
}

hipError_t launch_update(const UpdLaunch &l, bool rhs_only, hipStream_t s) {
    if (l.mixed) upd<float>(l, rhs_only, s);
    else upd<double>(l, rhs_only, s);
    return hipGetLastError();
}

}  // namespace afd

namespace afd {

__global__ __launch_bounds__(BLOCK) void k_diag(DiagArgs a) {
    const Grid &g = a.g;
    __shared__ double red[DIAG_N][BLOCK];
    const long ni = g.nx - 2 * a.ng, nj = g.ny - 2 * a.ng, nk = g.nz - 2 * a.ng, tot = ni * nj * nk;
    double v[DIAG_N] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const long n = g.ncell;
    for (long t = (long)blockIdx.x * BLOCK + threadIdx.x; t < tot; t += (long)gridDim.x * BLOCK) {
        const int k = a.ng + (int)(t % nk), j = a.ng + (int)((t / nk) % nj), i = a.ng + (int)(t / (nj * nk));
        const long c = cidx(g, i, j, k);
        double vx = a.P[n + c], vy = a.P[2 * n + c], vz = a.P[3 * n + c];
        double v2 = vx * vx + vy * vy + vz * vz;
        if (v2 >= 1.0) v2 = 1.0 - 1e-14;
        double W = 1.0 / sqrt(1.0 - v2);
        if (W > v[0]) v[0] = W;
        if (a.rmhd) {
            double dBx = (a.P[5 * n + c + g.sx] - a.P[5 * n + c - g.sx]) / (2.0 * a.dx);
            double dBy = (a.P[6 * n + c + g.sy] - a.P[6 * n + c - g.sy]) / (2.0 * a.dy);
            double dBz = (a.P[7 * n + c + 1] - a.P[7 * n + c - 1]) / (2.0 * a.dz);
            double d = dBx + dBy + dBz;
            if (fabs(d) > v[1]) v[1] = fabs(d);
            v[2] += d;
            v[3] += d * d;
        }
        if (i == a.ng) {
            double q[9], U[9];
            for (int m = 0; m < (a.rmhd ? 9 : 5); ++m) q[m] = a.P[m * n + c];
            if (a.rmhd) rmhd_p2c_cell(a.gfac53, a.p_max, a.v_max, q, U);
            else srhd_p2c_cell(a.gfac53, q, U);
            v[4] += U[1] * a.dy * a.dz;
        }
    }
    for (int m = 0; m < DIAG_N; ++m) red[m][threadIdx.x] = v[m];
    __syncthreads();
    for (int o = BLOCK / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            red[0][threadIdx.x] = pymax(red[0][threadIdx.x], red[0][threadIdx.x + o]);
            red[1][threadIdx.x] = pymax(red[1][threadIdx.x], red[1][threadIdx.x + o]);
            for (int m = 2; m < DIAG_N; ++m) red[m][threadIdx.x] += red[m][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x < DIAG_N) a.partial[threadIdx.x * gridDim.x + blockIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(BLOCK) void k_diag_reduce(const double *partial, int nblocks, double *out) {
    __shared__ double red[DIAG_N][BLOCK];
    double v[DIAG_N] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int t = threadIdx.x; t < nblocks; t += BLOCK) {
        v[0] = pymax(v[0], partial[t]);
        v[1] = pymax(v[1], partial[nblocks + t]);
        for (int m = 2; m < DIAG_N; ++m) v[m] += partial[m * nblocks + t];
    }
    for (int m = 0; m < DIAG_N; ++m) red[m][threadIdx.x] = v[m];
    __syncthreads();
    for (int o = BLOCK / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            red[0][threadIdx.x] = pymax(red[0][threadIdx.x], red[0][threadIdx.x + o]);
            red[1][threadIdx.x] = pymax(red[1][threadIdx.x], red[1][threadIdx.x + o]);
            for (int m = 2; m < DIAG_N; ++m) red[m][threadIdx.x] += red[m][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x < DIAG_N) out[threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(BLOCK) void k_centerline(const double *P, Grid g, int ng, double v_max, double *out) {
    const int nxi = g.nx - 2 * ng;
    const int t = blockIdx.x * BLOCK + threadIdx.x;
    if (t >= nxi) return;
    const int j = ng + (g.ny - 2 * ng) / 2, k = ng + (g.nz - 2 * ng) / 2;
    const long n = g.ncell, c = cidx(g, ng + t, j, k);
    double vx = P[n + c], vy = P[2 * n + c], vz = P[3 * n + c];
    double v2 = vx * vx + vy * vy + vz * vz;
    const double vmax2 = v_max * v_max;
    if (v2 >= vmax2) {
        double fac = v_max / sqrt(v2 + 1e-32);
        vx *= fac;
        v2 = vmax2 - 1e-14;
    }
    double v2c = v2 < 0.0 ? 0.0 : (v2 > 1.0 - 1e-14 ? 1.0 - 1e-14 : v2);
    out[t] = 1.0 / sqrt(1.0 - v2c);
    out[nxi + t] = P[c];
    out[2 * nxi + t] = P[4 * n + c];
    out[3 * nxi + t] = vx;
}

}  // namespace afd
