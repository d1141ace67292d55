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
// What bounds it is FP64 arithmetic (one thread evaluates some ten square roots, inverse
// tangents and logarithms for 8 bytes written), so the work is to call fewer of them:
//   * the sums over the four corners are taken inside the functions: the logarithms of a
//     sum over corners become one logarithm of a quotient of products (8 -> 2, none
//     without strike slip), and two inverse tangents become one of a complex product,
//     atan(a1/b1) - atan(a2/b2) = arg((b1 + i a1)(b2 - i a2)) for b1, b2 > 0, exact since
//     the difference lies within (-pi, pi) (8 -> 4, and their 8 quotients go with them);
//   * square roots and quotients shared between corners are taken once;
//   * sines and cosines of the fault's angles come with it, those of a row's latitude from
//     a table of the grid.
// Either form of a sum rounds to a few units of the largest term.
// Per fault on 2000x2000 cells: 882 us before, 204 now (181 registers, 2 wavefronts a SIMD, before; 118 and 4 now).
// ---------------------------------------------------------------------------
struct OkadaFault {
    double lon_c, lat_c, depth, L, W, H;
    double ss, cs;          // sine and cosine of the strike
    double sd, cd;          // of the dip (cd 0 and sd +-1 within 1e-6 of vertical)
    double d1, d2;          // slip components
    double lon0, dlon;
};

// functions of a grid row's latitude that the projection uses
struct OkadaRow {
    double lat, cl, slcl, c2;  // latitude (degrees), cos, sin * cos, cos of the double angle
};

// a / b for b in the normal range, its reciprocal by Newton's iteration from the hardware
// estimate and the quotient corrected by its residual
__device__ __forceinline__ double okada_div(const double a, const double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// atan(a1 / b1) - atan(a2 / b2)
__device__ __forceinline__ double okada_datan(double a1, double b1, double a2, double b2) {
    if (b1 < 0.0) { a1 = -a1; b1 = -b1; }
    if (b2 < 0.0) { a2 = -a2; b2 = -b2; }
    return atan2(__builtin_fma(a1, b2, -(a2 * b1)), __builtin_fma(b1, b2, a1 * a2));
}

// x, y: position along and across the strike
__device__ __forceinline__ double okada_uz(const OkadaFault &f, const double x, const double y) {
    constexpr double alp3 = 0.5;  // (1 - alpha) / alpha with alpha = 2/3
    constexpr double pi2 = 6.283185307179586;
    const double sd = f.sd, cd = f.cd;
    const double sdcd = sd * cd, cdcd = cd * cd;
    double xi[2] = {x + 0.5 * f.L, x - 0.5 * f.L};
    const double p = y * cd + f.depth * sd;
    double q = y * sd - f.depth * cd;
    double et[2] = {p + 0.5 * f.W, p - 0.5 * f.W};
#pragma unroll
    for (int k = 0; k < 2; k++) {
        if (fabs(xi[k]) < 1e-6) xi[k] = 0.0;
        if (fabs(et[k]) < 1e-6) et[k] = 0.0;
    }
    if (fabs(q) < 1e-6) q = 0.0;
    if (q == 0.0 && ((xi[0] * xi[1] <= 0.0 && et[0] * et[1] == 0.0) || (et[0] * et[1] <= 0.0 && xi[0] * xi[1] == 0.0)))
        return 0.0;  // on a fault edge
    const double q2 = q * q;
    double r[2][2], xx[2];  // [j][k]: corner (xi[j], et[k])
#pragma unroll
    for (int j = 0; j < 2; j++) {
        xx[j] = sqrt(xi[j] * xi[j] + q2);
#pragma unroll
        for (int k = 0; k < 2; k++) r[j][k] = sqrt(xi[j] * xi[j] + et[k] * et[k] + q2);
    }
    // corners beyond the end of the fault's edge lines, where r + xi or r + et cancels
    bool kxi[2], ket[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        kxi[k] = xi[0] < 0.0 && r[1][k] + xi[1] < 1e-6;
        ket[k] = et[0] < 0.0 && r[k][1] + et[1] < 1e-6;
    }
    // sums over the corners with the sign of each: `s` of the rational terms, the numerator
    // and denominator of the logarithms' quotients, and the four tangents
    double s1 = 0.0, s2 = 0.0;
    double ln[2] = {1.0, 1.0}, le[2] = {1.0, 1.0};  // prod (r + d), prod (r + et): [0] corners with +, [1] with -
    double ta[2][2], tb[2][2], wa[2][2], wb[2][2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const double X = xi[j], E = et[k], R = r[j][k];
            const double sg = (j + k != 1) ? 1.0 : -1.0;
            const int m = j + k != 1 ? 0 : 1;
            ta[j][k] = 0.0; tb[j][k] = 1.0;
            wa[j][k] = 0.0; wb[j][k] = 1.0;
            if (R == 0.0) continue;
            const double yy = E * cd + q * sd;
            const double rd = R + (E * sd - q * cd);
            const double x11 = kxi[k] ? 0.0 : okada_div(1.0, R * (R + X));
            const double y11 = ket[j] ? 0.0 : okada_div(1.0, R * (R + E));
            const double ird = okada_div(1.0, rd);
            if (q != 0.0) { ta[j][k] = X * E; tb[j][k] = q * R; }
            double i3 = 0.0, i4 = 0.0;  // the parts of I3 sd and I4 sdcd outside logarithms and tangents
            if (cd != 0.0) {
                if (X != 0.0) {
                    i4 = X * ird * sdcd;
                    wa[j][k] = E * (xx[j] + q * cd) + xx[j] * (R + xx[j]) * sd;
                    wb[j][k] = X * (R + xx[j]) * cd;
                }
                i3 = yy * cd * ird;
            } else {
                i3 = (E + yy * q * ird) * ird;
                i4 = 0.5 * X * yy * ird * ird;
            }
            if (f.d1 != 0.0) {
                const double b1 = alp3 * yy * ird * sd - okada_div(q, R);
                // ai2 = log(rd) + ai3 sd: its rational part here, its logarithms below
                const double a2 = cd != 0.0 ? okada_div(i3, cdcd) * sd : 0.5 * i3 * sd;
                s1 += sg * (b1 * sd + (q * q * y11 - alp3 * a2 * sd) * cd);
                ln[m] *= rd;
                le[m] *= ket[j] ? okada_div(1.0, R - E) : R + E;
            }
            if (f.d2 != 0.0) {
                const double b1 = -E * q * x11 - alp3 * X * ird * sdcd;
                const double a4 = cd != 0.0 ? okada_div(i4, cdcd) : i4;
                s2 += sg * (b1 * sd + (q2 * x11 + alp3 * a4 * sdcd) * cd);
            }
        }
    }
    double uz = 0.0;
    if (f.d1 != 0.0) {
        // sum of ai2's logarithms: log(rd) + sd (sd log(rd) - ale) / cd^2, = log(rd) - sd ale / 2
        // for a vertical fault
        const double lr = log(okada_div(ln[0], ln[1])), la = log(okada_div(le[0], le[1]));
        const double a2 = cd != 0.0 ? lr + okada_div(sd * lr - la, cdcd) * sd : lr - 0.5 * la * sd;
        uz += f.d1 * okada_div(s1 - alp3 * a2 * sd * cd, pi2);
    }
    if (f.d2 != 0.0) {
        // sum of -atan(X E / (q R)) sd
        const double tt = okada_datan(ta[0][0], tb[0][0], ta[0][1], tb[0][1]) -
                          okada_datan(ta[1][0], tb[1][0], ta[1][1], tb[1][1]);
        s2 -= tt * sd;
        if (cd != 0.0) {
            const double w = okada_datan(wa[0][0], wb[0][0], wa[0][1], wb[0][1]) -
                             okada_datan(wa[1][0], wb[1][0], wa[1][1], wb[1][1]);
            s2 += alp3 * okada_div(2.0 * w, cdcd) * sdcd * cd;
        }
        uz += f.d2 * okada_div(s2, pi2);
    }
    return uz;
}

__device__ __forceinline__ void gauss_krueger(const OkadaRow &g, const double lon, const double lat0, const double lon0,
                                              double &x, double &y) {
    const double D2R = 0.017453292371619689;
    const double v2 = g.cl * 0.0067397251 * g.cl + 1.0;
    const double al = lon - lon0;
    const double ph1 = g.lat + v2 * 0.5 * al * al * g.slcl * D2R;
    const double s1 = sin(ph1 * D2R), s2 = sin((ph1 + lat0) * 0.5 * D2R);
    const double u = 1.0 - s2 * 0.0066946053 * s2, dd = sqrt(u);
    const double r = okada_div(6335.4607362597517, u * dd);
    const double an = okada_div(6378.16, sqrt(1.0 - s1 * 0.0066946053 * s1));
    y = okada_div((ph1 - lat0) * r, 57.29578);
    x = okada_div(al * g.cl * an, 57.29578) * (okada_div(al * al * g.c2, 19696.838434850401) + 1.0);
}

// U_Z / H of the cell (i, row)
__device__ __forceinline__ double okada_cell(const OkadaFault &f, const OkadaRow &g, const int i) {
    double xp, yp;
    gauss_krueger(g, f.lon0 + i * f.dlon, f.lat_c, f.lon_c, xp, yp);
    return okada_uz(f, xp * f.ss + yp * f.cs, -xp * f.cs + yp * f.ss) / f.H;
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
__global__ void __launch_bounds__(256) k_okada(const OkadaFault f, const OkadaRow *rows, int nx, int ny, double *def,
                                               unsigned int *absmax) {
    float m = 0.f;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        const double uz = okada_cell(f, rows[j], i);
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
__global__ void __launch_bounds__(256) k_okada_add(const OkadaFault f, const OkadaRow *rows, int nx, int ny, int P,
                                                   const double thr, T *e, T *D, T *arr) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < (int64_t)nx * ny;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(c / nx), i = (int)(c - (int64_t)j * nx);
        double u = okada_cell(f, rows[j], i);
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
