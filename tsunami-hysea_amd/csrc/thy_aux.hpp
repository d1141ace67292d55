// thy_aux.hpp -- kernels around the step: initial dt, Okada (FP64), metric init,
// output conversion, gauges, mass.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "thy_step.hpp"

namespace thy {

// ---------------------------------------------------------------------------
// Initial dt (src/GPU/Timestep.cu:11-33): per cell the sum of the four faces'
// wave speeds (src/GPU/Arista_kernel.cu:1237-1428), dt = 2*CFL*A/sum with CFL
// passed as float (src/GPU/Volumen_kernel.cu:78-94), min over cells.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_initial_dt(const StepArgs<T> a, int cur, unsigned int *out) {
    const int nx = a.nx, ny = a.ny, P = a.pitch;
    const bool per = a.periodic != 0;
    const T *e = a.e[cur], *qx = a.qx[cur], *qy = a.qy[cur];
    float m = 3.0e38f;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const int64_t o = (int64_t)j * P + i;
        const T h = e[o] + a.D[o];
        T sum = T(0);
        const RowGeo<T> rg = a.row[j];
        // x faces i (left) and i+1 (right)
        for (int s = 0; s < 2; s++) {
            const int g = i + s;               // face index
            if (per && g == nx) { /* face nx of cell nx-1 == face 0 */ }
            int il = g - 1, ir = g;
            bool lb = false, rb = false;
            if (il < 0) { if (per) il += nx; else { il = 0; lb = true; } }
            if (ir >= nx) { if (per) ir -= nx; else { ir = nx - 1; rb = true; } }
            const int64_t ol = (int64_t)j * P + il, orr = (int64_t)j * P + ir;
            T h0 = e[ol] + a.D[ol], q0 = qx[ol];
            T h1 = e[orr] + a.D[orr], q1 = qx[orr];
            T nrm = T(1);
            if (lb) { q0 *= a.bizq; nrm = T(-1); T t = h0; h0 = h1; h1 = t; t = q0; q0 = q1; q1 = t; }
            if (rb) q1 *= a.bder;
            sum += rg.ilx * init_wave(h0, q0 * nrm, h1, q1 * nrm, a.eps_h);
        }
        for (int s = 0; s < 2; s++) {
            const int g = j + s;
            int jl = g - 1, jr = g;
            bool lb = false, rb = false;
            if (jl < 0) { jl = 0; lb = true; }
            if (jr >= ny) { jr = ny - 1; rb = true; }
            const int64_t ol = (int64_t)jl * P + i, orr = (int64_t)jr * P + i;
            T h0 = e[ol] + a.D[ol], q0 = qy[ol];
            T h1 = e[orr] + a.D[orr], q1 = qy[orr];
            T nrm = T(1);
            if (lb) { q0 *= a.bsup; nrm = T(-1); T t = h0; h0 = h1; h1 = t; t = q0; q0 = q1; q1 = t; }
            if (rb) q1 *= a.binf;
            sum += a.fy[g].len * init_wave(h0, q0 * nrm, h1, q1 * nrm, a.eps_h);
        }
        (void)h;
        const T cflf = (T)(float)a.cfl;
        const T dtc = (sum < Num<T>::eps) ? Num<T>::big : Num<T>::div(T(2) * cflf * rg.A, sum);
        m = fminf(m, (float)dtc);
    }
    m = wave_min(m);
    __shared__ float red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) r = fminf(r, red[w]);
        atomicMin(out, __float_as_uint(r));
    }
}

// ---------------------------------------------------------------------------
// Okada (1992) rectangular source evaluated on the free surface (z = 0).
// At z = 0 the DC3D real-source part-A terms and the image-source part-A terms
// cancel identically (src/GPU/DC3D.cu:716-835 with d = depth for both), and the
// part-C terms enter multiplied by z, so the vertical displacement is the
// rotated part-B contribution  U_Z = sum_corners (+-) (B1 sin(dip) + B2 cos(dip)).
// Corner guards, singular cases and log branches follow DC3D (:661-714, :72-157).
// Projection: Gauss-Krueger about the fault centroid (src/GPU/prtoxy.cu:33-54).
// ---------------------------------------------------------------------------
// What bounds it is FP64 arithmetic: some eight inverse tangents, eight logarithms, thirty
// quotients and ten square roots a cell for 8 bytes written.  Sums over the corners inside the
// logarithms and tangents need fewer (204 us a fault), but round otherwise, and a cell whose
// rise comes close to the arrival threshold then arrives a step earlier or later.  So every
// sum keeps its terms and its order, and what is saved leaves each value as it is, or rounds
// a quotient or root in another way at most (none of the faults tried shows a difference):
//   * quotients and square roots without scaling and special cases, one reciprocal for all
//     quotients by the same divisor;
//   * the functions of the fault's angles and of a row's latitude come from tables;
//   * logarithms only with strike slip, tangents only with dip slip;
//   * a loop over the corners holds the registers of one.
// Per fault on 2000x2000 cells: 319 us, with 114 registers and 4 wavefronts a SIMD; 882 us in
// the general forms without tables (181 registers, 2 wavefronts).
// ---------------------------------------------------------------------------
struct OkadaFault {
    double lon_c, lat_c, depth, L, W, H, strike, dip, rake, slip;
    double lon0, dlon;
};

// functions of a fault's angles
struct OkadaPlane {
    double ss, cs;                   // sine and cosine of the strike
    double sd, cd, sdcd, cdcd;       // of the dip (cd 0 and sd +-1 within 1e-6 of vertical)
    double kcd, rcd, rH;             // 1 / cdcd, newton_rcp of cdcd and of H
    double d1, d2, c1, c2;           // slip components, and over 2 pi
};

// functions of a grid row's latitude that the projection uses
struct OkadaRow {
    double lat, sl, cl, hv2, c2;  // latitude (degrees), sin, cos, half of v2, cos of the double angle
};

__global__ void k_okada_rows(const double lat0, const double dlat, const int ny, OkadaRow *rows) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ny) return;
    OkadaRow r;
    r.lat = lat0 + j * dlat;
    const double rlat = r.lat * 0.017453292371619689;
    r.sl = sin(rlat);
    r.cl = cos(rlat);
    r.hv2 = (r.cl * 0.0067397251 * r.cl + 1.0) * 0.5;
    r.c2 = cos(rlat * 2.0);
    rows[j] = r;
}

__global__ void k_okada_plane(const OkadaFault f, OkadaPlane *out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const double RAD = 3.14159265358979323846 / 180.0, pi2 = 6.283185307179586;
    OkadaPlane o;
    o.ss = sin(RAD * f.strike);
    o.cs = cos(RAD * f.strike);
    o.sd = sin(f.dip * (pi2 / 360.0));
    o.cd = cos(f.dip * (pi2 / 360.0));
    if (fabs(o.cd) < 1e-6) {
        o.cd = 0.0;
        if (o.sd > 0.0) o.sd = 1.0;
        if (o.sd < 0.0) o.sd = -1.0;
    }
    o.sdcd = o.sd * o.cd;
    o.cdcd = o.cd * o.cd;
    o.kcd = 1.0 / o.cdcd;
    o.rcd = Num<double>::newton_rcp(o.cdcd);
    o.rH = Num<double>::newton_rcp(f.H);
    o.d1 = f.slip * cos(RAD * f.rake);
    o.d2 = f.slip * sin(RAD * f.rake);
    o.c1 = o.d1 / pi2;
    o.c2 = o.d2 / pi2;
    *out = o;
}

// x, y: position along and across the strike
__device__ __forceinline__ double okada_uz(const OkadaFault &f, const OkadaPlane &o, const double x, const double y) {
    using N = Num<double>;
    const double alpha = 2.0 / 3.0;
    const double alp3 = (1.0 - alpha) / alpha;
    const double sd = o.sd, cd = o.cd, sdcd = o.sdcd, cdcd = o.cdcd;
    double xi0 = x - -0.5 * f.L, xi1 = x - 0.5 * f.L;
    if (fabs(xi0) < 1e-6) xi0 = 0.0;
    if (fabs(xi1) < 1e-6) xi1 = 0.0;
    const double p = y * cd + f.depth * sd;
    double q = y * sd - f.depth * cd;
    double et0 = p - -0.5 * f.W, et1 = p - 0.5 * f.W;
    if (fabs(q) < 1e-6) q = 0.0;
    if (fabs(et0) < 1e-6) et0 = 0.0;
    if (fabs(et1) < 1e-6) et1 = 0.0;
    if (q == 0.0 && ((xi0 * xi1 <= 0.0 && et0 * et1 == 0.0) || (et0 * et1 <= 0.0 && xi0 * xi1 == 0.0)))
        return 0.0;  // on a fault edge
    const double q2 = q * q;
    // (x is 0 or at least 1e-12)
    auto root = [](const double x) { return x == 0.0 ? 0.0 : N::plain_sqrt(x); };
    const double r12 = root(xi0 * xi0 + et1 * et1 + q2);
    const double r21 = root(xi1 * xi1 + et0 * et0 + q2);
    const double r22 = root(xi1 * xi1 + et1 * et1 + q2);
    // corners beyond the end of the fault's edge lines, where r + xi or r + et cancels
    const bool kxi0 = xi0 < 0.0 && r21 + xi1 < 1e-6, kxi1 = xi0 < 0.0 && r22 + xi1 < 1e-6;
    const bool ket0 = et0 < 0.0 && r12 + et1 < 1e-6, ket1 = et0 < 0.0 && r22 + et1 < 1e-6;
    double uz = 0.0;
#pragma unroll 1
    for (int c = 0; c < 4; c++) {
        const bool j = (c & 1) != 0, k = (c & 2) != 0;
        const double X = j ? xi1 : xi0, E = k ? et1 : et0;
        const bool kxi = k ? kxi1 : kxi0, ket = j ? ket1 : ket0;
        const double xi2 = X * X;
        const double r = root(xi2 + E * E + q2);
        if (r == 0.0) continue;
        const double yy = E * cd + q * sd;
        const double dd = E * sd - q * cd;
        const double rd = r + dd, ird = N::newton_rcp(rd);
        double b1 = 0.0, b2 = 0.0;
        if (o.d1 != 0.0) {
            const double l = log(ket ? r - E : r + E), ale = ket ? -l : l, lrd = log(rd);
            const double y11 = ket ? 0.0 : N::plain_rcp(r * (r + E));
            double ai3;
            if (cd != 0.0) ai3 = N::plain_div(N::plain_div(yy * cd, rd, ird) - ale + sd * lrd, cdcd, o.rcd);
            else ai3 = (N::plain_div(E, rd, ird) + N::plain_div(yy * q, rd * rd) - ale) / 2.0;
            const double ai2 = lrd + ai3 * sd;
            b1 += o.c1 * (N::plain_div(-q, r) + N::plain_div(alp3 * yy, rd, ird) * sd);
            b2 += o.c1 * (q * (q * y11) - alp3 * ai2 * sd);
        }
        if (o.d2 != 0.0) {
            const double tt = (q == 0.0) ? 0.0 : atan(N::plain_div(X * E, q * r));
            const double qx = q * (kxi ? 0.0 : N::plain_rcp(r * (r + X)));
            double ai4 = 0.0;
            if (cd != 0.0) {
                if (X != 0.0) {
                    const double xx = root(xi2 + q2);
                    ai4 = o.kcd * (N::plain_div(X, rd, ird) * sdcd +
                                   2.0 * atan(N::plain_div(E * (xx + q * cd) + xx * (r + xx) * sd, X * (r + xx) * cd)));
                }
            } else {
                ai4 = N::plain_div(X * yy, rd * rd) / 2.0;
            }
            b1 += o.c2 * (-E * qx - tt - N::plain_div(alp3 * X, rd, ird) * sdcd);
            b2 += o.c2 * (q * qx + alp3 * ai4 * sdcd);
        }
        const double v = b1 * sd + b2 * cd;
        uz += j == k ? v : -v;
    }
    return uz;
}

__device__ __forceinline__ void gauss_krueger(const OkadaRow &g, const double lon, const double lat0, const double lon0,
                                              double &x, double &y) {
    using N = Num<double>;
    const double D2R = 0.017453292371619689;
    const double al = lon - lon0;
    const double ph1 = g.lat + g.hv2 * al * al * g.sl * g.cl * D2R;
    const double rph1 = ph1 * D2R;
    const double rph2 = (ph1 + lat0) * 0.5 * D2R;
    const double s1 = sin(rph1), s2 = sin(rph2);
    const double dd = N::plain_sqrt(1.0 - s2 * 0.0066946053 * s2);
    const double r = N::plain_div(6335.4607362597517, dd * (dd * dd));
    const double an = N::plain_div(6378.16, N::plain_sqrt(1.0 - s1 * 0.0066946053 * s1));
    y = N::plain_div(ph1 - lat0, N::plain_div(57.29578, r));
    x = N::plain_div(al * g.cl, N::plain_div(57.29578, an)) * (N::plain_div(al * al * g.c2, 19696.838434850401) + 1.0);
}

// U_Z / H of the cell (i, row)
__device__ __forceinline__ double okada_cell(const OkadaFault &f, const OkadaPlane &o, const OkadaRow &g, const int i) {
    double xp, yp;
    gauss_krueger(g, f.lon0 + i * f.dlon, f.lat_c, f.lon_c, xp, yp);
    return Num<double>::plain_div(okada_uz(f, o, xp * o.ss + yp * o.cs, -xp * o.cs + yp * o.ss), f.H, o.rH);
}

// add a cell's displacement (src/GPU/Deformacion.cu:22-53); eta_ini += U_Z, but a cell
// that has arrived keeps its arrival time
template <typename T>
__device__ __forceinline__ void okada_add(const double u, const int64_t o, T *e, T *D, T *arr) {
    D[o] = (T)((double)D[o] - u);
    e[o] = (T)((double)e[o] + u);
    if (arr && !Arrival<T>::arrived(arr[o])) arr[o] = (T)((double)arr[o] + u);
}

// U_Z of every cell into `def` and its largest magnitude (for the relative crop), as a
// float (src/GPU/Deformacion.cu:13-20,132-136)
__global__ void __launch_bounds__(256) k_okada(const OkadaFault f, const OkadaPlane *plane, const OkadaRow *rows, int nx, int ny, double *def,
                                               unsigned int *absmax) {
    const OkadaPlane o = *plane;
    float m = 0.f;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const double uz = okada_cell(f, o, rows[j], i);
        def[c] = uz;
        m = fmaxf(m, (float)fabs(uz));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(absmax, __float_as_uint(m));
}

// U_Z of every cell, cropped at an absolute height (thr <= 0: not cropped) and added at
// once: where the crop does not depend on the largest U_Z, the field needs no second pass
template <typename T>
__global__ void __launch_bounds__(256) k_okada_add(const OkadaFault f, const OkadaPlane *plane, const OkadaRow *rows, int nx, int ny, int P,
                                                   const double thr, T *e, T *D, T *arr) {
    const OkadaPlane o = *plane;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        double u = okada_cell(f, o, rows[j], i);
        if (fabs(u) < thr) u = 0.0;
        okada_add(u, (int64_t)j * P + i, e, D, arr);
    }
}

// crop + add: src/GPU/Deformacion.cu:22-53,132-142
template <typename T>
__global__ void __launch_bounds__(256) k_okada_apply(const double *def, int nx, int ny, int P, int crop_flag,
                                                     double crop_value, const unsigned int *absmax, T *e, T *D, T *arr) {
    double thr = -1.0;
    if (crop_flag == 1) thr = crop_value * (double)__uint_as_float(*absmax);
    else if (crop_flag == 2) thr = crop_value;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        double u = def[c];
        if (crop_flag != 0 && fabs(u) < thr) u = 0.0;
        okada_add(u, (int64_t)j * P + i, e, D, arr);
    }
}

// eta_max / eta_ini / arrival init (src/GPU/Metrics.cu:6-21,44-55 as called at
// src/GPU/ShallowWater.cu:305-309)
template <typename T>
__global__ void __launch_bounds__(256) k_init_metrics(const T *e, const T *D, int nx, int ny, int P, T eps_h,
                                                      T *emax, T *arr) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const int64_t o = (int64_t)j * P + i;
        const T h = e[o] + D[o];
        const T v = (h < eps_h) ? T(-1e30) : e[o];
        emax[o] = v;
        if (arr) arr[o] = v;  // eta_ini, by the same kernel as eta_max (src/GPU/ShallowWater.cu:305-308)
    }
}

// metric update outside the step kernel (src/GPU/Metrics.cu:23-42,57-77)
template <typename T>
__global__ void __launch_bounds__(256) k_update_metrics(const T *e, const T *D, int nx, int ny, int P, T eps_h,
                                                        T dif_at, T t, T *emax, T *arr) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const int64_t o = (int64_t)j * P + i;
        const T h = e[o] + D[o];
        if (e[o] > emax[o] && h > eps_h) emax[o] = e[o];
        if (arr && !Arrival<T>::arrived(arr[o]) && tabs(e[o] - arr[o]) > dif_at) arr[o] = Arrival<T>::enc(t);
    }
}

// output fields (src/GPU/netcdf_kernel.cu:6-126) into a dense [ny][nx] float array
template <typename T>
__global__ void __launch_bounds__(256) k_output(int which, const T *e, const T *qx, const T *qy, const T *D,
                                                const T *emax, const T *arr, int nx, int ny, int P, T eps_h,
                                                double Href, double Q, double Tscale, float *out) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const int64_t o = (int64_t)j * P + i;
        double v;
        if (which == 0) {
            const T h = e[o] + D[o];
            v = (h < eps_h) ? -9999.0 : (double)e[o] * Href;
        } else if (which == 1 || which == 2) {
            const double h = (double)e[o] + (double)D[o];
            const double eh = (double)eps_h;
            const double f = (h < eh) ? 1.4142135623730951 * h / sqrt(h * h * h * h + eh * eh * eh * eh) * (Q / Href)
                                      : Q / (h * Href);
            v = (double)(which == 1 ? qx[o] : qy[o]) * f;
        } else if (which == 3) {
            v = (double)D[o] * Href;
        } else if (which == 4) {
            v = ((double)emax[o] < -1e20) ? -9999.0 : (double)emax[o] * Href;
        } else {
            v = (arr && Arrival<T>::arrived(arr[o])) ? Arrival<T>::dec(arr[o]) * Tscale : -1.0;
        }
        out[c] = (float)v;
    }
}

// per-block FP64 partial sums of h*area for the mass check
template <typename T>
__global__ void __launch_bounds__(256) k_mass(const T *e, const T *D, const RowGeo<T> *row, const double *area,
                                              int nx, int ny, int P, double *partial) {
    double s = 0.0;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const int64_t o = (int64_t)j * P + i;
        s += ((double)e[o] + (double)D[o]) * area[j];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) r += red[w];
        partial[blockIdx.x] = r;
    }
}

}  // namespace thy
