// thy_sweep.hpp -- row-sweep step kernel of the Tsunami-HySEA scheme for gfx950.
//
// Same step as k_step (src/GPU/Timestep.cu:70-120 plus the metric update and the gauge
// gather) in one launch, organised for the CDNA execution model instead of 2D LDS tiles.
// The grid is cut into segments of 56 columns, one lane each with a 4-column halo on either
// side of the wavefront (the reach of the 2s+WAF stencil through the two passes), and each
// segment into
//   * deep-water strips: rows far from coast, borders and sponges.  One wavefront walks a
//     strip from top to bottom; each row flows through a register pipeline, x-neighbours
//     come from adjacent lanes, y-neighbours from the rows before, so every face is
//     evaluated once, with no LDS tile, barrier or halo re-load inside the strip;
//   * general tiles: everything else.  One workgroup evaluates up to 8 rows out of LDS, the
//     deep-water faces in place and the others from a work list.
// Both evaluate a face through the same functions with the same border, first-order band
// and clamped-stencil conventions, so the cut changes no result.
#pragma once
#include "thy_step.hpp"

namespace thy {

constexpr int SW_HALO = 4;
constexpr int SW_OUT = 64 - 2 * SW_HALO;  // output columns per wavefront
constexpr int SW_WAVES = 4;               // wavefronts per workgroup (side by side in x)

// Cross-lane moves: lane l receives the value of lane l-1 / l+1 (the lane without a source
// receives 0 or keeps its own value; it lies outside every output cell's stencil).  FP32
// moves are data-parallel-primitive moves across the whole wavefront (wave_shr:1,
// wave_shl:1), which the compiler folds into the instruction that uses the value where
// there is one; FP64 values move as two words.
__device__ __forceinline__ float dpp_left(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float dpp_right(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double dpp_left(double v) {
    const int2 b = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, b.x, 0x138, 0xf, 0xf, true),
                                                __builtin_amdgcn_update_dpp(0, b.y, 0x138, 0xf, 0xf, true)));
}
__device__ __forceinline__ double dpp_right(double v) {
    const int2 b = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, b.x, 0x130, 0xf, 0xf, true),
                                                __builtin_amdgcn_update_dpp(0, b.y, 0x130, 0xf, 0xf, true)));
}

// read-only table entry at a wavefront-uniform address (scalar load)
template <typename S> __device__ __forceinline__ S uniform_load(const S *p) {
    static_assert(sizeof(S) % 4 == 0, "table entries are whole dwords");
    S out;
    __builtin_memcpy(&out, (const __attribute__((address_space(4))) S *)p, sizeof(S));
    return out;
}

// The argument block at a wavefront-uniform address, read again from here on.  The block's
// fields are scalar loads that hit the scalar cache; without this the compiler loads each
// once, at the top, and keeps it: the kernels below then hold some 120 scalars more than
// there are registers, spilled to lanes of vector registers, and every phase starts with
// dozens of lane reads (half of a tile's vector instructions).
template <typename T> using ArgsAt = const __attribute__((address_space(4))) StepArgs<T> *;
template <typename T> __device__ __forceinline__ const StepArgs<T> &again(ArgsAt<T> p) {
    asm volatile("" : "+s"(p));
    return *(const StepArgs<T> *)p;
}

// ---------------------------------------------------------------------------
// Deep-water forms of the face fluxes: the 2s branch that mass_flux / mom_flux take
// when all four stencil depths exceed hpos outside the first-order band
// (src/GPU/Arista_kernel.cu:545,653,1105,1214), written with the per-cell square
// roots and velocities computed once per cell.  Strips and tiles both evaluate a deep face
// through these, so either gives it the same value.  (k_step has its own 2s branch: in FP64
// with the general quotients and roots, so its last place may differ.)
// ---------------------------------------------------------------------------
// Mass flux of the x face between hL and the row's cell (h1), and of the y face between h0
// and h1: src/GPU/Arista_kernel.cu:79-95,118-130, 97-114,674-686 (Fx, Fy: normal discharge
// times the face's length factor).  The positivity limiter rarely acts: one test for both.
template <typename T>
__device__ __forceinline__ void limit_mass(T &Fx, T &Fy, T hL, T h0, T h1, T kA, T k0, T k1, T dt) {
    const T limx = (Fx > T(0) ? hL : h1) * kA, limy = Fy > T(0) ? h0 * k0 : h1 * k1;
    const T denx = habs(Fx) + Num<T>::eps, deny = habs(Fy) + Num<T>::eps;
    if (__any(dt * denx > limx || dt * deny > limy)) {
        Fx = limit_flux(Fx, limx, denx, dt);
        Fy = limit_flux(Fy, limy, deny, dt);
    }
}

// one cell of a deep momentum face: total depth, normal and tangential discharge, sqrt(h),
// normal velocity
template <typename T> struct DC {
    T h, qn, qt, s, un;
};

// x face, 2s momentum flux: src/GPU/Arista_kernel.cu:221-280.  deta: eta difference of the
// face (deta_of; e_b - e_a where both cells' eta clears the shallower bed)
template <typename T>
__device__ __forceinline__ MF<T> fast_mom_x(const DC<T> &a, const DC<T> &b, T deta, T il, T kd, T dt) {
    MF<T> o;
    const T hij = T(0.5) * (a.h + b.h);
    const T uij = Num<T>::plain_div(Num<T>::mad(a.s, a.un, b.s * b.un), a.s + b.s + Num<T>::eps);
    const T lmax = habs(uij) + Num<T>::plain_sqrt(hij);
    const bool up = uij < T(0);
    const T uu = up ? b.un : a.un;
    const T qnn = up ? b.qn : a.qn;
    const T qtt = up ? b.qt : a.qt;
    const T fn = uu * qnn * il;
    const T DES = kd * dt * (lmax * lmax) * (b.qn - a.qn);
    o.mn = Num<T>::mad(hij * deta, il, fn) - DES;
    o.pn = -fn + DES;
    const T ft = uu * qtt * il;
    o.mt = ft;
    o.pt = -ft;
    o.w = il * lmax;
    return o;
}

// y face, 2s momentum flux: src/GPU/Arista_kernel.cu:780-843 (G: FaceGeoY or DeepMom)
template <typename T, typename G>
__device__ __forceinline__ MF<T> fast_mom_y(const DC<T> &a, const DC<T> &b, T deta, const G &f, T dt) {
    MF<T> o;
    const T g0 = f.cos0, g1 = f.cos1, ic0 = f.ic0, ic1 = f.ic1, len = f.len;
    const T hij = T(0.5) * (a.h + b.h);
    const T uij = Num<T>::plain_div(Num<T>::mad(a.s, a.un, b.s * b.un), a.s + b.s + Num<T>::eps);
    const T lmax = habs(uij) + Num<T>::plain_sqrt(hij);
    deta = Num<T>::mad(-(uij * uij), f.gd, f.gh * deta);
    const bool up = uij < T(0);
    const T uu = up ? b.un : a.un;
    const T qnn = up ? b.qn : a.qn;
    const T qtt = up ? b.qt : a.qt;
    const T fn = uu * qnn * len;
    T mn, pn;
    if (up) { pn = -fn; mn = fn * f.g1ic0; }
    else { mn = fn; pn = -fn * g0 * ic1; }
    mn = Num<T>::mad(hij * deta * len, ic0, mn);
    const T DES = f.kdy * dt * (lmax * lmax) * Num<T>::mad(b.qn, g1, -(a.qn * g0));
    o.mn = Num<T>::mad(-DES, ic0, mn);
    o.pn = Num<T>::mad(DES, ic1, pn);
    const T ft = uu * qtt * len;
    o.mt = ft;
    o.pt = -ft;
    o.w = len * lmax;
    return o;
}

template <typename T> struct RowCell {
    T e, D, qx, qy;
};

// The row sweeps address the state arrays through one buffer resource over the state
// block that holds them all: the lane's column is the vector offset, the array's offset
// in the block plus the row's the scalar offset, all 32-bit (the block is under 2^31
// bytes; thy_create keeps larger grids off these kernels).  One resource instead of one
// per array leaves the scalar registers to the rest of the loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t whole_array(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, bytes, 0x00020000);
}

// byte offsets in the state block of the arrays one launch reads and writes; without
// arrival tracking the arrival load reads emax instead (its stores never apply)
template <typename T> struct StateOffsets {
    int e, D, qx, qy, oe, oqx, oqy, emax, arr;
    template <typename A>
    __device__ __forceinline__ StateOffsets(const A &a, const T *ie, const T *iD, const T *iqx, const T *iqy,
                                            const T *we, const T *wqx, const T *wqy)
        : e(at(a, ie)), D(at(a, iD)), qx(at(a, iqx)), qy(at(a, iqy)), oe(at(a, we)), oqx(at(a, wqx)),
          oqy(at(a, wqy)), emax(at(a, a.emax)), arr(at(a, a.track_arrival ? a.arr : a.emax)) {}
    template <typename A> static __device__ __forceinline__ int at(const A &a, const T *p) {
        return (int)((const char *)p - a.block);
    }
};

template <typename T> __device__ __forceinline__ T buf_load(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <> __device__ __forceinline__ float buf_load<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
template <> __device__ __forceinline__ double buf_load<double>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// Vector offset of a buffer store that must not happen: at or beyond the resource's
// record count, so the hardware drops it.  A store whose lanes may all be masked is
// issued this way instead of under a branch, so that every iteration of a row loop
// issues the same number of memory instructions and the compiler can wait for a row's
// loads without waiting for the stores issued after them (one counter covers both).
constexpr int kDropOffset = (int)0x80000000;

template <typename T>
__device__ __forceinline__ void buf_store(T v, __amdgpu_buffer_rsrc_t r, int voff, int soff, bool on = true);
template <>
__device__ __forceinline__ void buf_store<float>(float v, __amdgpu_buffer_rsrc_t r, int voff, int soff, bool on) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, on ? voff : kDropOffset, soff, 0);
}
template <>
__device__ __forceinline__ void buf_store<double>(double v, __amdgpu_buffer_rsrc_t r, int voff, int soff, bool on) {
    using V2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v), r, on ? voff : kDropOffset, soff, 0);
}

// a stencil cell with a given desingularisation factor f ...
template <typename T> __device__ __forceinline__ SC<T> sc_of(T e, T D, T qn, T qt, T f) {
    SC<T> c;
    c.e = e;
    c.D = D;
    c.h = e + D;
    c.qn = qn;
    c.qt = qt;
    c.f = f;
    return c;
}
// ... or with its own (the compiler drops it where no face uses it)
template <typename T> __device__ __forceinline__ SC<T> sc_of(T e, T D, T qn, T qt, const Prm<T> &p) {
    return sc_of(e, D, qn, qt, desing(e + D, p.eps_h));
}

// ---------------------------------------------------------------------------
// General tiles: one workgroup per tile of 56 output columns and up to kTileRows rows.
//
// A shallow face costs several times a deep-water one (square roots, divisions,
// exponentials, three limiters), and along a coast only one lane in four to one in twenty
// of a wavefront's row holds one, so evaluating a row's faces in place runs the long code
// mostly for idle lanes, row after row.  Here the rows of the tile and its halo lie in
// LDS, every wavefront evaluates the deep-water forms of its rows in place, and the faces
// that take any other branch are put on a work list (ballots of the depth tests combined
// with scalar mask arithmetic, so the classification costs little vector work) that the
// workgroup then evaluates with every lane busy, x and y faces together.  Once for the
// mass pass, once for the momentum pass:
//   load the rows, classify                        | barrier
//   deep mass faces in place, list the others      | barrier
//   listed mass faces                              | barrier
//   h* (as e*) of rows y0-2 .. y0+m+1, classify    | barrier
//   list the other momentum faces                  | barrier
//   listed momentum faces                          | barrier
//   deep momentum faces in place, cell updates
// Which lane evaluates a face does not change its value, and per cell the accumulation
// order is x faces, lower y face, upper y face in every tile and strip.
// A tile's time is a chain of latencies.  Everything it reads from memory (rows, row tables,
// metrics) is requested at once, and so is everything a phase reads from LDS.  The rows'
// masks are combined in one go, a row to a lane, in every wavefront alike, and a sum over the
// lanes says where each row's faces go in the list.  With an atomic counter and a mask read for
// each row a whole step of 240x200, where nothing else counts, took 14.3 us where it takes 11.8
// (tiles of 4 and of 3 rows); 2000x2000, 1563 tiles: 50.4 and 46.4.
// ---------------------------------------------------------------------------
// 8 rows: taller tiles would have less halo (4 of 12 rows in the mass pass), but at 8 the
// tile's LDS (31 KB in FP32) lets five workgroups share a CU, as their registers do.
constexpr int kTileRows = 8;
constexpr int kTileHalf = 4;  // rows whose momentum faces always fit the result table

using mask64 = unsigned long long;

template <typename T> struct alignas(16) FaceOut {
    T mn, pn, mt, w;  // (pt = -mt)
};

template <typename T> struct TileLds {
    static constexpr int G = kTileRows;
    // listed momentum faces at a time: those of kTileHalf rows, two for each thread.  Where
    // every face is listed (a shelf shallower than hpos) a tile of 8 rows takes two such rounds;
    // with three of 3, 3 and 2 rows, in twice as many passes of the workgroup, a step of
    // 2000x2000 took 261 us and takes 226 (FP64 811 and 656).
    static constexpr int kResults = kTileHalf * 57 + (kTileHalf + 1) * 56;
    static_assert(kResults <= 2 * 64 * SW_WAVES, "two faces a thread");
    T in[4][(G + 8) * 64];   // e, D, qx, qy of rows y0-4 .. y0+m+3
    T es[(G + 4) * 64];      // e* of rows y0-2 .. y0+m+1
    // a listed face: direction << 15 | row << 6 | lane
    union {
        struct {
            T F[2][(G + 5) * 64];   // mass fluxes of the x faces (row, lane) and y faces
            unsigned short mass_list[(G + 4) * 61 + (G + 5) * 60];
        };
        struct {  // (once the fluxes have been read)
            FaceOut<T> R[kResults];  // results of the listed momentum faces
            unsigned short list[kResults];
        };
    };
    RowGeo<T> row[G + 4];    // of rows y0-2 ..
    FaceGeoY<T> fy[G + 5];   // of faces y0-2 ..
    mask64 deep[G + 8], dry[G + 8];    // lanes deeper than hpos / dry (h <= eps), by row
    mask64 sdeep[G + 4], sdry[G + 4];  // the same of h*
    int still[SW_WAVES];               // the wavefront's rows are land
};

// Lane l holds the masks of row l: the lanes whose x face, and whose lower y face, take the
// deep form (dx, dy) or go on the work list (wx, wy: x faces first), and where in the list
// the row's faces begin.
struct RowFaces {
    mask64 dx, dy, wx, wy;
    int base;
};
__device__ __forceinline__ mask64 of_row(const mask64 m, const int l) {
    return ((mask64)(unsigned)__builtin_amdgcn_readlane((int)(m >> 32), l) << 32) |
           (unsigned)__builtin_amdgcn_readlane((int)(unsigned)m, l);
}
// fills `base` for up to 16 rows and returns the length of the list
__device__ __forceinline__ int place_faces(RowFaces &f) {
    const int c = __popcll(f.wx) + __popcll(f.wy);
    int n = c;  // inclusive sum over the lanes of a row of 16 (row_shr:1, 2, 4, 8)
    n += __builtin_amdgcn_update_dpp(0, n, 0x111, 0xf, 0xf, true);
    n += __builtin_amdgcn_update_dpp(0, n, 0x112, 0xf, 0xf, true);
    n += __builtin_amdgcn_update_dpp(0, n, 0x114, 0xf, 0xf, true);
    n += __builtin_amdgcn_update_dpp(0, n, 0x118, 0xf, 0xf, true);
    f.base = n - c;
    return __builtin_amdgcn_readlane(n, 15);
}

__device__ __forceinline__ bool lane_of(const mask64 m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
__device__ __forceinline__ int rank_of(const mask64 m) {  // set bits below this lane
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
// x faces (lane = the face's high cell) whose four cells / two cells are all in m
__device__ __forceinline__ mask64 all4(const mask64 m) { return m & (m << 1) & (m << 2) & (m >> 1); }
__device__ __forceinline__ mask64 both(const mask64 m) { return m & (m << 1); }

// Columns x0 .. x0+55, rows y0 .. y0+m-1 (m <= kTileRows), with bc filled by begin_step for
// this launch; every thread of the workgroup calls it.  Returns this lane's minimum of the
// per-cell dt of the next step (3e38 when it updated no cell).
template <typename T>
__device__ __forceinline__ float general_tile(const ArgsAt<T> args, const BlockCtl<T> &bc, const int x0, const int y0,
                                              const int m, TileLds<T> &s) {
    constexpr int G = kTileRows, W = SW_WAVES;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // what follows from it is not kept across a loop over tiles
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T dt = (T)bc.dt;
    int nx, ny;
    bool per;
    float dtmin = 3.0e38f;
    bool bad = false;

    const int gx = x0 - SW_HALO + lane;
    int cx;  // column loaded by this lane: wrapped (periodic) or clamped onto the grid
    // ---- rows y0-4 .. y0+m+3, the row tables and the metrics of this wavefront's output
    // rows ra .. rb-1 ----
    constexpr int KR = (G + W - 1) / W, KL = (G + 8 + W - 1) / W;
    const int kr = (m + W - 1) / W, ra = wv * kr, rb = min(ra + kr, m);
    T pm[KR], pt[KR];
    bool still;
    {
        const StepArgs<T> &a = again<T>(args);
        nx = a.nx;
        ny = a.ny;
        per = a.periodic != 0;
        const T hpos = a.hpos;
        cx = gx < 0 ? 0 : (gx >= nx ? nx - 1 : gx);
        const int vgx = cx * (int)sizeof(T);
        if (per) cx = ((gx % nx) + nx) % nx;
        const int P = a.pitch;
        const bool c1b = __builtin_amdgcn_readfirstlane(bc.cur) != 0;
        const __amdgpu_buffer_rsrc_t rs = whole_array(a.block, a.block_bytes);
        const StateOffsets<T> o(a, c1b ? a.e[1] : a.e[0], a.D, c1b ? a.qx[1] : a.qx[0], c1b ? a.qy[1] : a.qy[0], a.e[0],
                                a.qx[0], a.qy[0]);
        const int vcx = cx * (int)sizeof(T);
        T v[KL][4];
#pragma unroll
        for (int t = 0; t < KL; t++) {
            const int y = y0 - 4 + min(wv + t * W, m + 7), r = y < 0 ? 0 : (y >= ny ? ny - 1 : y);
            const int so = r * P * (int)sizeof(T);
            v[t][0] = buf_load<T>(rs, vcx + o.e, so);
            v[t][1] = buf_load<T>(rs, vcx + o.D, so);
            v[t][2] = buf_load<T>(rs, vcx + o.qx, so);
            v[t][3] = buf_load<T>(rs, vcx + o.qy, so);
        }
        constexpr int NR = sizeof(RowGeo<T>) / sizeof(T), NF = sizeof(FaceGeoY<T>) / sizeof(T);
        static_assert(NR * (G + 4) <= 64 * W && NF * (G + 5) <= 64 * W, "one table word per thread");
        T tr = T(0), tf = T(0);
        if (tid < NR * (G + 4)) {
            const int y = y0 - 2 + tid / NR;
            tr = ((const T *)a.row)[(y < 0 ? 0 : (y >= ny ? ny - 1 : y)) * NR + tid % NR];
        }
        if (tid < NF * (G + 5)) {
            const int y = y0 - 2 + tid / NF;
            tf = ((const T *)a.fy)[(y < 0 ? 0 : (y > ny ? ny : y)) * NF + tid % NF];
        }
#pragma unroll
        for (int t = 0; t < KR; t++) {
            const int so = (y0 + min(ra + t, m - 1)) * P * (int)sizeof(T);
            pm[t] = buf_load<T>(rs, vgx + o.emax, so);
            pt[t] = buf_load<T>(rs, vgx + o.arr, so);
        }
        // (rows beyond the tile's were loaded as its last one: no guard for `still`)
        still = true;
#pragma unroll
        for (int t = 0; t < KL; t++) {
            const int i = wv + t * W;
            const T h = v[t][0] + v[t][1];
            still = still && h <= Num<T>::eps && v[t][2] == T(0) && v[t][3] == T(0);  // (no NaN)
            if (i < m + 8) {
                const int p = i * 64 + lane;
                s.in[0][p] = v[t][0];
                s.in[1][p] = v[t][1];
                s.in[2][p] = v[t][2];
                s.in[3][p] = v[t][3];
                const mask64 dp = __ballot(h > hpos), dr = __ballot(!(h > Num<T>::eps));
                if (lane == 0) {
                    s.deep[i] = dp;
                    s.dry[i] = dr;
                }
            }
        }
        if (tid < NR * (G + 4)) ((T *)s.row)[tid] = tr;
        if (tid < NF * (G + 5)) ((T *)s.fy)[tid] = tf;
        const bool all_still = __all(still);
        if (lane == 0) s.still[wv] = all_still;
    }
    // lanes outside the grid take the e* of the clamped column (clamped stencils)
    const bool xedge = !per && (x0 - SW_HALO < 0 || x0 + SW_OUT + SW_HALO > nx);
    // this lane's x face is the left face of its cell: g = gx
    const bool low_border = !per && gx == 0;
    const bool out_col = lane >= SW_HALO && lane < SW_HALO + SW_OUT && gx < nx;
    // lanes whose x face / cell lies on the grid, and x faces of the first-order band
    const mask64 on_face = __ballot(per || (gx >= 0 && gx <= nx)), on_cell = __ballot(per || (gx >= 0 && gx < nx));
    const int gw = per ? cx : gx;
    const mask64 first = __ballot(gw < 2 || gw > nx - 2);
    const T *const e_ = s.in[0], *const D_ = s.in[1], *const qx_ = s.in[2], *const qy_ = s.in[3];
    // Land: every cell of the tile and its halo dry and without discharge (a depth that is not
    // a number takes the other way, where the health check finds it), clear of the sponges.  Every face is then zero and the update leaves e (its depth stays 0) and
    // zero discharges; the arrival rule may still record the start (a dry cell's eta_ini
    // is a marker).
    __syncthreads();
    bool land = true;
    for (int w = 0; w < W; w++) land = land && s.still[w];
    if (__builtin_amdgcn_readfirstlane(land)) {
        const StepArgs<T> &a = again<T>(args);
        if (a.eps_h >= Num<T>::eps && x0 - SW_HALO >= a.sp_izq && x0 + SW_OUT + SW_HALO <= nx - a.sp_der && y0 - 2 >= a.sp_sup &&
            y0 + m + 2 <= ny - a.sp_inf) {
            const T tnow = (T)bc.t;
            const int P = a.pitch;
            const bool c1b = __builtin_amdgcn_readfirstlane(bc.cur) != 0;
            const __amdgpu_buffer_rsrc_t rs = whole_array(a.block, a.block_bytes);
            const StateOffsets<T> o(a, a.e[0], a.D, a.qx[0], a.qy[0], c1b ? a.e[0] : a.e[1], c1b ? a.qx[0] : a.qx[1],
                                    c1b ? a.qy[0] : a.qy[1]);
            const int voff = out_col ? gx * (int)sizeof(T) : kDropOffset;
            for (int f = ra; f < rb; f++) {
                const int p = (f + 4) * 64 + lane, soff = (y0 + f) * P * (int)sizeof(T);
                const T eo = e_[p], D = D_[p];
                T carr = pt[0];
#pragma unroll
                for (int t = 1; t < KR; t++) carr = f - ra == t ? pt[t] : carr;
                const bool arr_on = out_col && a.track_arrival && !Arrival<T>::arrived(carr) && tabs(eo - carr) > a.dif_at;
                buf_store<T>(Arrival<T>::enc(tnow), rs, voff, o.arr + soff, arr_on);
                buf_store<T>(eo + D > T(0) ? eo : -D, rs, voff, o.oe + soff, out_col);
                buf_store<T>(T(0), rs, voff, o.oqx + soff, out_col);
                buf_store<T>(T(0), rs, voff, o.oqy + soff, out_col);
            }
            return out_col ? (float)Num<T>::big : 3.0e38f;
        }
    }
    // ---- mass pass: x faces of rows y0-2+j, y faces g = y0-2+j ----
    int nm;
    {
        RowFaces rf;
        {
            const int i = min(lane, m + 4), y = y0 - 2 + i;
            const mask64 d2 = s.deep[i + 2], r2 = s.dry[i + 2], dy = s.deep[i] & s.deep[i + 1] & d2 & s.deep[i + 3],
                         r1 = s.dry[i + 1];
            const bool in_x = lane < m + 4 && y >= 0 && y < ny, in_y = lane < m + 5 && y >= 0 && y <= ny;
            rf.dx = in_x ? all4(d2) & ~first : 0ull;
            rf.dy = in_y && !(y < 2 || y > ny - 2) ? dy : 0ull;
            rf.wx = in_x ? ~rf.dx & ~both(r2) & on_face & 0x7ffffffffffffffcull : 0ull;   // lanes 2 .. 62
            rf.wy = in_y ? ~rf.dy & ~(r1 & r2) & on_cell & 0x3ffffffffffffffcull : 0ull;  // lanes 2 .. 61
        }
        nm = place_faces(rf);
        // this wavefront's faces j = ja + t: rows ja+1 .. of the tile in registers
        constexpr int K = (G + 5 + W - 1) / W;
        const int kj = (m + 5 + W - 1) / W, ja = wv * kj;
        T h[K + 1], qy[K], qx[K];
#pragma unroll
        for (int t = 0; t <= K; t++) {
            const int p = min(ja + 1 + t, m + 7) * 64 + lane;
            h[t] = e_[p] + D_[p];
            if (t < K) qy[t] = qy_[p];
            if (t > 0) qx[t - 1] = qx_[p];
        }
#pragma unroll
        for (int t = 0; t < K; t++) {
            const int j = ja + t;
            if (t >= kj || j >= m + 5) break;
            const mask64 dx = of_row(rf.dx, j), dy = of_row(rf.dy, j), wx = of_row(rf.wx, j), wy = of_row(rf.wy, j);
            T Fx = T(0), Fy = T(0);
            if (dx | dy) {
                const RowGeo<T> &rg = s.row[min(j, m + 3)];
                const FaceGeoY<T> &fg = s.fy[j];
                Fx = dpp_left(qx[t]) * rg.ilx;
                Fy = qy[t] * fg.lc0;
                limit_mass(Fx, Fy, dpp_left(h[t + 1]), h[t], h[t + 1], rg.kA, fg.k0, fg.k1, dt);
                Fx = lane_of(dx) ? Fx : T(0);
                Fy = lane_of(dy) ? Fy : T(0);
            }
            s.F[0][j * 64 + lane] = Fx;
            s.F[1][j * 64 + lane] = Fy;
            if (wx | wy) {
                const int b = __builtin_amdgcn_readlane(rf.base, j);
                if (lane_of(wx)) s.mass_list[b + rank_of(wx)] = (unsigned short)(j << 6 | lane);
                if (lane_of(wy)) s.mass_list[b + __popcll(wx) + rank_of(wy)] = (unsigned short)(0x8000 | j << 6 | lane);
            }
        }
    }
    __syncthreads();
    // the constants of a listed face
    struct Listed {
        Prm<T> p;
        T L, g0, g1, k0, k1, val, ic0, ic1;
        int border;
        bool yf, band;
    };
    auto listed = [&](const StepArgs<T> &a, const int code, const int j) {  // j: row of the tables
        Listed f;
        f.yf = (code & 0x8000) != 0;
        const int l = code & 63;
        const int g = f.yf ? y0 - 2 + j : x0 - SW_HALO + l, ng = f.yf ? ny : nx;
        int gp = g;
        if (per && !f.yf) gp = ((g % nx) + nx) % nx;
        f.border = (per && !f.yf) ? 0 : (g == 0 ? 1 : (g == ng ? 2 : 0));
        f.band = gp < 2 || gp > ng - 2;
        f.p.eps_h = a.eps_h;
        f.p.hpos = a.hpos;
        f.p.cvis = a.cvis;
        f.p.bl = f.yf ? a.bsup : a.bizq;
        f.p.bh = f.yf ? a.binf : a.bder;
        if (f.yf) {
            const FaceGeoY<T> &q = s.fy[j];
            f.L = q.len; f.g0 = q.cos0; f.g1 = q.cos1; f.k0 = q.k0; f.k1 = q.k1; f.val = q.valy; f.ic0 = q.ic0; f.ic1 = q.ic1;
        } else {
            const RowGeo<T> &q = s.row[j];
            f.L = q.ilx; f.k0 = f.k1 = q.kA; f.val = q.valx;
            f.g0 = f.g1 = f.ic0 = f.ic1 = T(1);
        }
        return f;
    };
    // ---- listed mass faces ----
    if (nm) {
        const StepArgs<T> &a = again<T>(args);
        for (int k = tid; k < nm; k += 64 * W) {
            const int code = s.mass_list[k], l = code & 63, j = (code >> 6) & 31;
            const Listed f = listed(a, code, j);
            const int p = (j + 2) * 64 + l, st = f.yf ? 64 : 1;
            const T *const qn = f.yf ? qy_ : qx_;
            const SC<T> M = sc_of(e_[p - 2 * st], D_[p - 2 * st], T(0), T(0), T(0));
            const SC<T> A = sc_of(e_[p - st], D_[p - st], qn[p - st], T(0), f.p), B = sc_of(e_[p], D_[p], qn[p], T(0), f.p);
            const SC<T> Q = sc_of(e_[p + st], D_[p + st], T(0), T(0), T(0));
            s.F[f.yf ? 1 : 0][j * 64 + l] = mass_waf<T>(f.yf, M, A, B, Q, f.border, f.band, f.L, f.g0, f.g1, f.k0, f.k1,
                                                        f.val, dt, f.p);
        }
        __syncthreads();
    }
    // ---- h* (as e*) of rows y0-2 .. y0+m+1, with the sponge ----
    const StepArgs<T> &ah = again<T>(args);
    {
        constexpr int K = (G + 4 + W - 1) / W;
        const int kj = (m + 4 + W - 1) / W, ja = wv * kj;
        T FL[K], FB[K + 1], ei[K], Di[K];
#pragma unroll
        for (int t = 0; t <= K; t++) {
            const int q = min(ja + t, m + 4) * 64 + lane;
            FB[t] = s.F[1][q];
            if (t < K) {
                FL[t] = s.F[0][q];
                ei[t] = e_[q + 128];
                Di[t] = D_[q + 128];
            }
        }
#pragma unroll
        for (int t = 0; t < K; t++) {
            const int j = ja + t, y = y0 - 2 + j;
            if (t >= kj || j >= m + 4) break;
            const T D = Di[t];
            T acc = (low_border ? -FL[t] : FL[t]) - dpp_right(FL[t]);
            acc = Num<T>::mad(y == 0 ? -FB[t] : FB[t], s.fy[j].ic1, acc);
            acc = Num<T>::mad(-FB[t + 1], s.fy[j + 1].ic0, acc);
            T es = Num<T>::mad(dt * s.row[j].invA, acc, ei[t]);
            if (!(es + D > T(0))) es = -D;
            if (x0 - SW_HALO < ah.sp_izq || x0 + SW_OUT + SW_HALO > nx - ah.sp_der || y < ah.sp_sup || y >= ny - ah.sp_inf)
                es = sponge_eta(ah, es, D, per ? cx : gx, y, s.row[j].dxs, s.row[j].dys);
            if (xedge) es = __shfl(es, cx - (x0 - SW_HALO), 64);
            const T h = es + D;
            const mask64 dp = __ballot(h > ah.hpos), dr = __ballot(!(h > Num<T>::eps));
            if (y >= 0 && y < ny) {  // (rows outside the grid are not read)
                s.es[j * 64 + lane] = es;
                if (lane == 0) {
                    s.sdeep[j] = dp;
                    s.sdry[j] = dr;
                }
            }
        }
    }
    __syncthreads();
    // rows outside the grid stand for the edge row (clamped stencils)
    const int jlo = max(0, 2 - y0), jhi = min(m + 3, ny + 1 - y0);
    auto row_j = [&](const int j) { return min(max(j, jlo), jhi); };
    // with an hpos below 0 dry cells count as deep: faces between two of them are zero there too
    const mask64 below = ah.hpos < T(0) ? ~0ull : 0ull;
    // ---- momentum pass, rows y0+r0 .. y0+r1-1 at a time: the whole tile, or kTileHalf rows
    // when its listed faces do not fit the result table ----
    for (int r0 = 0, r1 = m; r0 < m;) {
        // list the faces that do not take the deep form: x faces of rows y0+f, y faces g = y0+f
        RowFaces rf;
        const auto classify = [&] {
            const int i = min(lane, m), g = y0 + i;
            const mask64 d2 = s.sdeep[i + 2], dy = s.sdeep[i] & s.sdeep[i + 1] & d2 & s.sdeep[i + 3];
            const bool in_x = lane >= r0 && lane < r1, in_y = lane >= r0 && lane <= r1;
            const mask64 bx = both(s.sdry[i + 2]), by = s.sdry[row_j(i + 1)] & s.sdry[row_j(i + 2)];
            rf.dx = in_x ? all4(d2) & ~first & ~(bx & below) : 0ull;
            rf.dy = in_y && !(g < 2 || g > ny - 2) ? dy & ~(by & below) : 0ull;
            rf.wx = in_x ? ~rf.dx & ~bx & on_face & 0x1ffffffffffffff0ull : 0ull;  // lanes 4 .. 60
            rf.wy = in_y ? ~rf.dy & ~by & on_cell & 0x0ffffffffffffff0ull : 0ull;  // lanes 4 .. 59
            return place_faces(rf);
        };
        int nq = classify();
        if (nq > TileLds<T>::kResults) {
            r1 = r0 + kTileHalf;
            nq = classify();
        }
        for (int f = r0 + wv; f <= r1; f += W) {
            const mask64 wx = of_row(rf.wx, f), wy = of_row(rf.wy, f);
            if (wx | wy) {
                const int b = __builtin_amdgcn_readlane(rf.base, f);
                if (lane_of(wx)) s.list[b + rank_of(wx)] = (unsigned short)(f << 6 | lane);
                if (lane_of(wy)) s.list[b + __popcll(wx) + rank_of(wy)] = (unsigned short)(0x8000 | f << 6 | lane);
            }
        }
        __syncthreads();  // (and no wavefront still reads the results of the round before)
        if (nq) {
            const StepArgs<T> &a = again<T>(args);
            for (int k = tid; k < nq; k += 64 * W) {
                const int code = s.list[k], l = code & 63, fr = (code >> 6) & 31;
                const Listed f = listed(a, code, fr + 2);
                const T *const qn = f.yf ? qy_ : qx_, *const qt = f.yf ? qx_ : qy_;
                // the four cells: rows fr .. fr+3 of a y face, lanes l-2 .. l+1 of an x face
                auto cell = [&](const int d) {
                    const int p = f.yf ? row_j(fr + 2 + d) * 64 + l : (fr + 2) * 64 + l + d;
                    return sc_of(s.es[p], D_[p + 128], qn[p + 128], qt[p + 128], f.p);
                };
                const MF<T> r = mom_waf<T>(f.yf, cell(-2), cell(-1), cell(0), cell(1), f.border, f.band, f.L, f.g0, f.g1,
                                           f.ic0, f.ic1, f.val, dt, f.p);
                s.R[k] = FaceOut<T>{r.mn, r.pn, r.mt, r.w};
            }
            __syncthreads();
        }
        // ---- deep momentum faces and the update of this wavefront's rows ----
        const int fa = max(ra, r0), fb = min(rb, r1);
        if (fa < fb) {
            const StepArgs<T> &a = again<T>(args);
            const T hpos = a.hpos;
            const T tnow = (T)bc.t;
            const int P = a.pitch;
            const bool c1b = __builtin_amdgcn_readfirstlane(bc.cur) != 0;
            const bool spx = x0 - SW_HALO < a.sp_izq || x0 + SW_OUT + SW_HALO > nx - a.sp_der;
            const __amdgpu_buffer_rsrc_t rs = whole_array(a.block, a.block_bytes);
            const StateOffsets<T> o(a, a.e[0], a.D, a.qx[0], a.qy[0], c1b ? a.e[0] : a.e[1], c1b ? a.qx[0] : a.qx[1],
                                    c1b ? a.qy[0] : a.qy[1]);
            // rows fa-1 .. fb of h*, all read at once
            constexpr int K = KR + 2;
            T re[K], rD[K], rqx[K], rqy[K];
#pragma unroll
            for (int t = 0; t < K; t++) {
                const int q = row_j(min(fa + 1 + t, fb + 2)) * 64 + lane;
                re[t] = s.es[q];
                rD[t] = D_[q + 128];
                rqx[t] = qx_[q + 128];
                rqy[t] = qy_[q + 128];
            }
            // e*, D, sqrt(h*), qy/h*, qx, qy of row g-1 for the y faces
            T s2 = re[0], D2 = rD[0], qx2 = rqx[0], qy2 = rqy[0];
            T sq2 = Num<T>::plain_sqrt(s2 + D2), v2 = qy2 * Num<T>::plain_rcp(s2 + D2);
            T X2 = T(0), Y2 = T(0), W2 = T(0);  // accumulators of row g-1
#pragma unroll
            for (int t = 0; t <= KR; t++) {
                const int f = fa + t;
                if (f > fb) break;
                const int g = y0 + f;
                const T s1 = re[t + 1], D1 = rD[t + 1], qx1 = rqx[t + 1], qy1 = rqy[t + 1];
                const T h1 = s1 + D1;
                const T sq1 = Num<T>::plain_sqrt(h1), ih = Num<T>::plain_rcp(h1);
                const T u1 = qx1 * ih, v1 = qy1 * ih;
                // x faces of row g and the y face between rows g-1 and g
                const bool xs = f < fb;
                const mask64 dx = xs ? of_row(rf.dx, f) : 0ull, dy = of_row(rf.dy, f);
                const mask64 wf = of_row(rf.wx, f), wx = xs ? wf : 0ull, wy = of_row(rf.wy, f);
                MF<T> rx{T(0), T(0), T(0), T(0), T(0)}, ry = rx;
                if (dx | dy) {
                    const FaceGeoY<T> &fg = s.fy[f + 2];
                    const RowGeo<T> &rg = s.row[min(f + 2, m + 3)];
                    const T eL = dpp_left(s1), DL = dpp_left(D1);
                    const DC<T> L{eL + DL, dpp_left(qx1), dpp_left(qy1), dpp_left(sq1), dpp_left(u1)}, X{h1, qx1, qy1, sq1, u1};
                    const DC<T> B{s2 + D2, qy2, qx2, sq2, v2}, Y{h1, qy1, qx1, sq1, v1};
                    const MF<T> tx = fast_mom_x(L, X, deta_of(eL, s1, DL, D1), rg.ilx, rg.kdx, dt);
                    const MF<T> ty = fast_mom_y(B, Y, deta_of(s2, s1, D2, D1), fg, dt);
                    if (lane_of(dx)) rx = tx;
                    if (lane_of(dy)) ry = ty;
                }
                if (wx | wy) {
                    const int b = __builtin_amdgcn_readlane(rf.base, f);
                    if (lane_of(wx)) {
                        const FaceOut<T> o = s.R[b + rank_of(wx)];
                        rx = MF<T>{o.mn, o.mt, o.pn, -o.mt, o.w};
                    }
                    if (lane_of(wy)) {
                        const FaceOut<T> o = s.R[b + __popcll(wf) + rank_of(wy)];
                        ry = MF<T>{o.mn, o.mt, o.pn, -o.mt, o.w};
                    }
                }
                T X1 = -(low_border ? rx.mn : rx.pn) - dpp_right(rx.mn);
                T Y1 = -(low_border ? rx.mt : rx.pt) - dpp_right(rx.mt);
                T W1 = rx.w + dpp_right(rx.w);
                Y2 -= ry.mn;
                X2 -= ry.mt;
                W2 += ry.w;
                if (g == 0) { Y1 -= ry.mn; X1 -= ry.mt; }
                else { Y1 -= ry.pn; X1 -= ry.pt; }
                W1 += ry.w;
                // cell update of row g-1 (src/GPU/Volumen_kernel.cu:160-221)
                if (t > 0) {
                    const int ju = g - 1;
                    const RowGeo<T> &rg = s.row[f + 1];
                    const int soff = ju * P * (int)sizeof(T);
                    const int voff = out_col ? gx * (int)sizeof(T) : kDropOffset;
                    const T eo = e_[(f + 3) * 64 + lane];
                    T cmax = pm[0], carr = pt[0];
#pragma unroll
                    for (int k = 1; k < KR; k++)
                        if (f - 1 - ra == k) { cmax = pm[k]; carr = pt[k]; }
                    // metrics from the state before the step (src/GPU/Metrics.cu:23-42,57-77)
                    const bool max_on = out_col && eo > cmax && eo + D2 > a.eps_h;
                    const bool arr_on = out_col && a.track_arrival && !Arrival<T>::arrived(carr) && tabs(eo - carr) > a.dif_at;
                    const T dtc = (W2 < Num<T>::eps) ? Num<T>::big : Num<T>::plain_div(T(2) * a.cfl * rg.A, W2);
                    dtmin = fminf(dtmin, (float)dtc);  // halo lanes are dropped at the end
                    const T val = dt * rg.invA;
                    T qx = Num<T>::mad(val, X2, qx2), qy = Num<T>::mad(val, Y2, qy2);
                    if (spx || ju < a.sp_sup || ju >= ny - a.sp_inf) sponge_q(a, gx, ju, qx, qy);
                    const T hs = s2 + D2;
                    if (hs <= hpos) near_dry(hs, qx2, qy2, qx, qy, dt, a.mf0, a.vmax, a.eps_h);
                    bad = bad || (out_col && bad_cell(s2, qx, qy));
                    buf_store<T>(eo, rs, voff, o.emax + soff, max_on);
                    buf_store<T>(Arrival<T>::enc(tnow), rs, voff, o.arr + soff, arr_on);
                    buf_store<T>(s2, rs, voff, o.oe + soff, out_col);
                    buf_store<T>(qx, rs, voff, o.oqx + soff, out_col);
                    buf_store<T>(qy, rs, voff, o.oqy + soff, out_col);
                }
                X2 = X1; Y2 = Y1; W2 = W1;
                s2 = s1; D2 = D1; sq2 = sq1; v2 = v1; qx2 = qx1; qy2 = qy1;
            }
        }
        r0 = r1;
        r1 = min(r0 + kTileHalf, m);
    }
    raise_health(again<T>(args), bad);
    return out_col ? dtmin : 3.0e38f;
}

// workgroup minimum of the lanes' dt, folded into partial `part` of the launch's dt slot
template <typename T>
__device__ __forceinline__ void block_dt_min(const StepArgs<T> &a, const int slot, float dtmin, float *s_red,
                                             const int part) {
    const int tid = threadIdx.x;
    dtmin = wave_min(dtmin);
    if ((tid & 63) == 0) s_red[tid >> 6] = dtmin;
    __syncthreads();
    if (tid == 0) {
        float m = s_red[0];
#pragma unroll
        for (int w = 1; w < SW_WAVES; w++) m = fminf(m, s_red[w]);
        atomicMin(&a.dtmin[dt_at(slot, part)], __float_as_uint(m));
    }
}

// ---------------------------------------------------------------------------
// Deep-water strips.  Strips that with their halos lie clear of the borders, the
// first-order bands and the sponges, and whose still-water depth exceeds 3 hpos, take only
// the 2s faces: no sponge and no near-dry update, no clamped columns or rows.  Every
// wavefront checks at run time the conditions under which the general faces take the 2s
// branch (every loaded row deeper than hpos; every h* row that a face's stencil reaches
// deeper than hpos).  A strip whose check fails commits no dt and is redone as general
// tiles by its workgroup in the same launch (tile_or_strips); both evaluate the deep faces
// with the same functions, so the split changes no result.
// ---------------------------------------------------------------------------

// the value, computed where it is written (a cross-lane move folds into an instruction of
// its own basic block only)
__device__ __forceinline__ float here(float v) { asm("" : "+v"(v)); return v; }
__device__ __forceinline__ double here(double v) { return v; }

// a constant of a loop: FP64 ones in vector registers (the loop's row tables take most of the
// scalar registers)
__device__ __forceinline__ float held(float v) { return v; }
__device__ __forceinline__ double held(double v) { asm("" : "+v"(v)); return v; }

// One wavefront's strip on the deep-water path.  The 2s faces reach one row and one column,
// so the pipeline lags two rows: iteration r loads row r + 1, evaluates the mass faces of
// row r and the y face between rows r-1 and r, h* of row r-1, the momentum faces of row
// r-1 and the y face between rows r-2 and r-1, and updates row r-2.  Per cell the
// accumulation order is that of the general tiles (x faces, lower y face, upper y face), so
// the values are the same.
//
// The conditions under which the general faces take the 2s branch and its eta difference is
// e1 - e0 (every row y0-4 .. y1+3 and every h* deeper than hpos on every lane, both eta of a
// face above the shallower bed, no h* clipped at the bed) follow from one: the lowest eta
// plus the smallest depth exceeds hpos.  (A rounded sum is monotonic in its terms.)  It is
// taken over two columns and some eight rows at a time, with three running minima a row and a
// few instructions at the end of a window: over more, a trough would meet the bed of a
// shallow far from it.  (With the minima of a whole strip, a 2000x2000 step with 4.5 m troughs
// ten rows off ridges 5 m deep and hpos 1 m took 243 us instead of the 40 of a level sea.)
// Returns whether it held; if not, the caller redoes the strip (its writes are then rewritten
// and its dt is dropped).
//
// On a large grid vector issue and the traffic beyond the L2 bound it together (4000x3000, all
// deep: 102 us a step, 4.2 TB/s of the nine arrays, and no less with two rows of cells in
// flight), on a small one the latency of a row.  A steady row takes 132 vector instructions:
// no vote or comparison for each condition, neighbours' values by lane moves, one test for
// both limiters, and two rows of the loop written out, which spares the copies from row to row
// (four rows are no faster).  With those it took 175, and 2000x2000 54.9 us a step where it
// took 49.7 without, 1000x800 20.8 and 18.6, FP64 2000x2000 143.5 and 134.3.
template <typename T>
__device__ __forceinline__ bool deep_strip(const StepArgs<T> &a, const BlockCtl<T> &bc, const int x0, const int y0,
                                           const int rows, float &dtmin_out) {
    const int lane = threadIdx.x & 63;
    const bool c1 = __builtin_amdgcn_readfirstlane(bc.cur) != 0;
    const T dt = held((T)bc.dt);
    const T tnow = held(Arrival<T>::enc((T)bc.t));
    const int P = a.pitch * (int)sizeof(T);  // bytes per row
    const int y1 = y0 + rows;
    // the strip's columns x0-4 .. x0+59 and rows y0-4 .. y1+3 lie inside the grid: no
    // clamping.  Buffer accesses: the column and the array in the vector offset, the row in
    // the scalar offset.
    const __amdgpu_buffer_rsrc_t rs = whole_array(a.block, a.block_bytes);
    const StateOffsets<T> o(a, c1 ? a.e[1] : a.e[0], a.D, c1 ? a.qx[1] : a.qx[0], c1 ? a.qy[1] : a.qy[0],
                            c1 ? a.e[0] : a.e[1], c1 ? a.qx[0] : a.qx[1], c1 ? a.qy[0] : a.qy[1]);
    const int vx = (x0 - SW_HALO + lane) * (int)sizeof(T);
    const bool out_col = lane >= SW_HALO && lane < SW_HALO + SW_OUT;
    const int ve = vx + o.e, vD = vx + o.D, vqx = vx + o.qx, vqy = vx + o.qy, vm = vx + o.emax, va = vx + o.arr;
    const int vout = out_col ? vx : kDropOffset;
    const int we = vout + o.oe, wqx = vout + o.oqx, wqy = vout + o.oqy;
    auto load_row = [&](const int so) {
        RowCell<T> c;
        c.e = buf_load<T>(rs, ve, so);
        c.D = buf_load<T>(rs, vD, so);
        c.qx = buf_load<T>(rs, vqx, so);
        c.qy = buf_load<T>(rs, vqy, so);
        return c;
    };
    const T eps_h = held(a.eps_h), dif_at = held(a.dif_at), cfl2 = held(T(2) * a.cfl);
    const bool track = a.track_arrival != 0;
    const DeepRow<T> *const geo = a.deep_row;
    float dtmin = 3.0e38f;
    T nan_acc = T(0);  // turns NaN when a stored value is not finite
    // least eta of the inputs, eta of h* and depth since the last window, and the least sum of
    // the windows before; row y0-4 is an input only.  (A lane stands for its left neighbour too.)
    T emin = Num<T>::big, smin = Num<T>::big, Dmin = Num<T>::big;
    const T h_first = buf_load<T>(rs, ve, (y0 - 4) * P) + buf_load<T>(rs, vD, (y0 - 4) * P);
    T floor_h = Num<T>::min(h_first, dpp_left(h_first));
    // pipeline registers: rows r-2 and r-1 with their depths, h* of row r-2 with sqrt(h*)
    // and qy/h*, mass accumulator of row r-1, momentum accumulators of row r-2
    RowCell<T> i2 = RowCell<T>{T(0), T(0), T(0), T(0)}, i1 = i2;
    T h2 = T(0), h1 = T(0), s2 = T(0), hs2 = T(0), sq2 = T(0), v2 = T(0), m1 = T(0);
    T X2 = T(0), Y2 = T(0), W2 = T(0);
    RowCell<T> buf = load_row((y0 - 3) * P);
    T pm = buf_load<T>(rs, vm, y0 * P), pt = buf_load<T>(rs, va, y0 * P);
    // One row of the pipeline.  In the steady state (rows y0+2 .. y1) every stage applies,
    // so the stage conditions drop out at compile time; the other rows keep them.  Both
    // forms evaluate the same expressions.
    auto row = [&](const int r, auto steady_tag) {
        constexpr bool kS = decltype(steady_tag)::value;
        const RowCell<T> i0 = buf;
        const DeepRow<T> g = uniform_load(geo + r);
        const T cmax = pm, carr = pt;
        {
            buf = load_row((r + 1) * P);  // (the last one, y1+3, is an input only)
            const int jn = kS ? r - 1 : min(max(r - 1, y0), y1 - 1);
            pm = buf_load<T>(rs, vm, jn * P);
            pt = buf_load<T>(rs, va, jn * P);
        }
        const int ju = r - 2, j1 = r - 1;  // the row updated in this iteration, the row of h*
        const T h0 = i0.e + i0.D;
        emin = Num<T>::min(emin, i0.e);
        Dmin = Num<T>::min(Dmin, i0.D);
        // mass x faces of row r (h* rows y0-2 .. y1+1), y face r between rows r-1 and r
        // (faces y0-2 .. y1+2).  The limiter rarely acts: one test for both faces.
        T m0 = T(0);
        if (kS || r >= y0 - 2) {
            T Fx = dpp_left(i0.qx) * g.ilx, Fy = i1.qy * g.lc0;
            limit_mass(Fx, Fy, dpp_left(h0), h1, h0, g.kA, g.k0, g.k1, dt);
            m0 = here(Fx - dpp_right(Fx));
            m1 = Num<T>::mad(-Fy, g.ic0, m1);
            m0 = Num<T>::mad(Fy, g.ic1, m0);
        }
        // h* of row r-1 (rows y0-2 .. y1+1)
        T s1 = T(0), hs1 = T(0), sq1 = T(0), u1 = T(0), v1 = T(0);
        if (kS || (j1 >= y0 - 2 && j1 <= y1 + 1)) {
            s1 = Num<T>::mad(dt * g.p.invA, m1, i1.e);
            smin = Num<T>::min(smin, s1);
            hs1 = s1 + i1.D;
            sq1 = Num<T>::plain_sqrt(hs1);
            const T ih = Num<T>::plain_rcp(hs1);
            u1 = i1.qx * ih;
            v1 = i1.qy * ih;
        }
        // momentum x faces of row r-1 (rows y0 .. y1-1)
        T X1 = T(0), Y1 = T(0), W1 = T(0);
        if (kS || (j1 >= y0 && j1 < y1)) {
            const DC<T> A{dpp_left(hs1), dpp_left(i1.qx), dpp_left(i1.qy), dpp_left(sq1), dpp_left(u1)};
            const DC<T> B{hs1, i1.qx, i1.qy, sq1, u1};
            const MF<T> f = fast_mom_x(A, B, s1 - dpp_left(s1), g.p.ilx, g.p.kdx, dt);
            X1 = here(-f.pn - dpp_right(f.mn));
            Y1 = here(-f.pt - dpp_right(f.mt));
            W1 = here(f.w + dpp_right(f.w));
        }
        // momentum y face r-1 between rows r-2 and r-1 (faces y0 .. y1)
        if (kS || (j1 >= y0 && j1 <= y1)) {
            const DC<T> A{hs2, i2.qy, i2.qx, sq2, v2}, B{hs1, i1.qy, i1.qx, sq1, v1};
            const MF<T> f = fast_mom_y(A, B, s1 - s2, g.p, dt);
            Y2 -= f.mn;
            X2 -= f.mt;
            W2 += f.w;
            Y1 -= f.pn;
            X1 -= f.pt;
            W1 += f.w;
        }
        // cell update of row r-2 (src/GPU/Volumen_kernel.cu:160-221; h* > hpos here).  Every
        // iteration issues the five stores; those of halo rows and halo lanes, and metric
        // stores that do not apply, are dropped.
        {
            const bool on = kS || (ju >= y0 && ju < y1);
            const int so = (kS || on ? ju : y0) * P;
            const T eo = i2.e;
            const bool max_on = on && eo > cmax && h2 > eps_h;
            const bool arr_on = on && track && !Arrival<T>::arrived(carr) && habs(eo - carr) > dif_at;
            buf_store<T>(eo, rs, (max_on ? vout : kDropOffset) + o.emax, so);
            buf_store<T>(tnow, rs, (arr_on ? vout : kDropOffset) + o.arr, so);
            const T dtc = W2 < Num<T>::eps ? Num<T>::big : Num<T>::plain_div(cfl2 * g.q.A, W2);
            if (on) dtmin = Num<float>::min(dtmin, (float)dtc);  // halo lanes: dropped below
            const T val = dt * g.q.invA;
            const T qx = Num<T>::mad(val, X2, i2.qx), qy = Num<T>::mad(val, Y2, i2.qy);
            if (on) nan_acc = Num<T>::mad(s2, T(0), Num<T>::mad(qx, T(0), Num<T>::mad(qy, T(0), nan_acc)));
            buf_store<T>(s2, rs, kS || on ? we : kDropOffset, so);
            buf_store<T>(qx, rs, kS || on ? wqx : kDropOffset, so);
            buf_store<T>(qy, rs, kS || on ? wqy : kDropOffset, so);
        }
        i2 = i1; i1 = i0;
        h2 = h1; h1 = h0;
        s2 = s1; hs2 = hs1; sq2 = sq1; v2 = v1;
        m1 = m0;
        X2 = X1; Y2 = Y1; W2 = W1;
        // rows are not mixed: that would hold the registers of several at once
        __builtin_amdgcn_sched_barrier(0);
    };
    using Edge = std::integral_constant<bool, false>;
    using Steady = std::integral_constant<bool, true>;
    // Enter the loops with no memory instruction outstanding: the wait before a row then
    // only has the previous rows to account for (their stores may stay in flight while the
    // next row loads), instead of a full wait every row.
    __builtin_amdgcn_s_waitcnt(0);
    // the end of a window; the next one begins with the faces between rows r-2 and r-1
    auto window = [&] {
        int lane = threadIdx.x & 63;
        asm("" : "+v"(lane));  // (no masks held for it)
        const T e = lane == 0 || lane == 63 ? emin : Num<T>::min(emin, smin);  // (these lack a face)
        floor_h = Num<T>::min(floor_h, Num<T>::min(e, dpp_left(e)) + Num<T>::min(Dmin, dpp_left(Dmin)));
        emin = Num<T>::big;
        smin = s2;
        Dmin = Num<T>::min(i1.D, i2.D);
    };
    // rows y0-3 .. y1+2: the halo rows at either end (and a last row without a partner)
    // with the stage conditions, the steady state without them.  A strip of up to 8 rows is
    // one window (a window costs its chain of rows 0.1 to 0.2 us).
    int r = y0 - 3;
#pragma unroll 1
    for (; r <= y0 + 1; r++) row(r, Edge{});
    if (rows > 8) window();
    while (r < y1) {
        const int re = min(r + 7, y1);
#pragma unroll 1
        for (; r < re; r += 2) {
            row(r, Steady{});
            row(r + 1, Steady{});
        }
        if (rows > 8) window();
    }
#pragma unroll 1
    for (; r <= y1 + 2; r++) row(r, Edge{});
    window();
    const T h_last = buf.e + buf.D;
    floor_h = Num<T>::min(floor_h, Num<T>::min(h_last, dpp_left(h_last)));
    const bool valid = __all(lane == 0 || floor_h > tmax(a.hpos, T(0)));
    // a strip whose check failed is redone, and checked, as general tiles
    if (valid) raise_health(a, out_col && nan_acc != nan_acc);
    dtmin_out = out_col ? dtmin : 3.0e38f;
    return valid;
}

// One workgroup's share of a step.  A tile item: the general tile (x0, y0, rows).  A deep
// item: the strip (x0, y0, rows) of each wavefront; a strip whose check fails is redone
// here, tile by tile, by the whole workgroup (the values it has stored are overwritten;
// its metric updates used the state before the step and stand).
template <typename T>
__device__ __forceinline__ float tile_or_strips(const ArgsAt<T> args, const BlockCtl<T> &bc, const bool tile, int x0, int y0,
                                                int rows, TileLds<T> &s, int *s_fail) {
    float dtmin = 3.0e38f;
    if (!tile) {
        const int wv = threadIdx.x >> 6;
        bool ok = true;
        if (x0 >= 0) ok = deep_strip(again<T>(args), bc, x0, y0, rows, dtmin);
        if (!ok) {
            dtmin = 3.0e38f;
            // its stores reach the L2, through which every wavefront of the workgroup writes,
            // before those that replace them (a fence would write the L2 back for other XCDs:
            // every strip failing, 2000x2000, 264 us a step with it and 182 without)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if ((threadIdx.x & 63) == 0) {
            s_fail[3 * wv] = x0;
            s_fail[3 * wv + 1] = y0;
            s_fail[3 * wv + 2] = ok ? 0 : rows;
        }
        __syncthreads();
    }
    for (int w = 0, t = 0;;) {
        if (!tile) {  // tile t of the strip of wavefront w
            int n = 0, tiles = 0;
            for (; w < SW_WAVES; w++, t = 0) {
                n = __builtin_amdgcn_readfirstlane(s_fail[3 * w + 2]);
                tiles = (n + kTileRows - 1) / kTileRows;
                if (t < tiles) break;
            }
            if (w == SW_WAVES) break;
            const int d = n * t / tiles;
            x0 = __builtin_amdgcn_readfirstlane(s_fail[3 * w]);
            y0 = __builtin_amdgcn_readfirstlane(s_fail[3 * w + 1]) + d;
            rows = n * (t + 1) / tiles - d;
            t++;
            __syncthreads();  // the tile before still uses the rows in LDS
        }
        dtmin = fminf(dtmin, general_tile(args, bc, x0, y0, rows, s));
        if (tile) break;
    }
    return dtmin;
}

// Work items, one per workgroup: a general tile (x0, y0 << 4 | rows), or four deep-water
// strips (index of the first in the strip list, 0).  `strip`: a deep item's strip of this
// wavefront; x0 < 0: none.  flip > 0: the strips in reverse order, in place of the item's
// those mirrored over the list's `flip` groups of 8 items (an item of the same XCD).
template <typename T>
__device__ __forceinline__ int2 item_origin(const StepArgs<T> &a, const int2 it, bool &tile, int &rows, const int flip) {
    rows = it.y & 15;
    tile = rows != 0;
    if (tile) return make_int2(it.x, it.y >> 4);
    const int g = it.x / SW_WAVES;
    const int first = flip > 0 ? ((flip - 1 - (g >> 3)) * 8 + (g & 7)) * SW_WAVES : it.x;
    const int2 strip = uniform_load(a.deep + first + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    rows = strip.y & 2047;
    return make_int2(strip.x, strip.y >> 11);
}

// One step of one grid in one launch, a workgroup per work item.  Workgroup 0 is the
// step's writer.
template <typename T>
__global__ void __launch_bounds__(64 * SW_WAVES, sizeof(T) == 4 ? 5 : 2) k_sweep(const StepArgs<T> args_, const int slot, const int flip) {
    __shared__ TileLds<T> s;
    __shared__ BlockCtl<T> bc;
    __shared__ float s_red[SW_WAVES];
    __shared__ int s_fail[3 * SW_WAVES];
    (void)args_;  // the first kernel argument, read through its address
    const ArgsAt<T> args = (ArgsAt<T>)__builtin_amdgcn_kernarg_segment_ptr();
    const StepArgs<T> &a = again<T>(args);
    const int tid = threadIdx.x, bid = blockIdx.x;
    const int2 w = uniform_load(a.items + bid);
    if (tid == 0) begin_step(a, slot, bid == 0, bc, kDtParts);
    bool tile;
    int rows;
    const int2 o = item_origin(a, w, tile, rows, flip);
    __syncthreads();
    if (!bc.run) return;
    if (bid == 0) {
        const bool c1 = bc.cur != 0;
        gather_gauges(a, bc, c1 ? a.e[1] : a.e[0], c1 ? a.qx[1] : a.qx[0], c1 ? a.qy[1] : a.qy[0], tid, 64 * SW_WAVES);
    }
    const float dtmin = tile_or_strips<T>(args, bc, tile, o.x, o.y, rows, s, s_fail);
    block_dt_min(again<T>(args), slot, dtmin, s_red, bid);
}

// ---------------------------------------------------------------------------
// Many grids per launch.  Each scenario keeps its own state, control block and dt slots; a
// step of the batch advances every running scenario by one of its own steps in one launch:
// their deep-water strips, four of one scenario to a workgroup, and among them the general
// tiles of all, costliest first.  The item flagged as its scenario's writer publishes the next
// control block.  Item counts are read on the device, so one captured launch sequence serves a
// changing item list up to the captured grid size.
// ---------------------------------------------------------------------------
struct BatchItem {
    int slot;    // scenario slot (-1: padding)
    int writer;
    int2 it;     // the work item, as in the scenario's own list
};

struct BatchArgs {
    const StepArgs<float> *args;  // per scenario slot (zeroed while the slot is free)
    const BatchItem *items;
    const int *n_items;
};

__global__ void __launch_bounds__(64 * SW_WAVES, 5) k_batch(const BatchArgs q, const int slot) {
    __shared__ TileLds<float> s;
    __shared__ BlockCtl<float> bc;
    __shared__ float s_red[SW_WAVES];
    __shared__ int s_fail[3 * SW_WAVES];
    const int tid = threadIdx.x;
    if ((int)blockIdx.x >= __builtin_amdgcn_readfirstlane(*q.n_items)) return;
    const BatchItem w = uniform_load(q.items + blockIdx.x);
    if (w.slot < 0) return;
    const ArgsAt<float> args = (ArgsAt<float>)(q.args + w.slot);
    const StepArgs<float> &a = again<float>(args);
    if (!a.ctrl) return;
    if (tid == 0) begin_step(a, slot, w.writer != 0, bc, kDtParts);
    bool tile;
    int rows;
    const int2 o = item_origin(a, w.it, tile, rows, 0);
    __syncthreads();
    if (!bc.run) return;
    if (w.writer) {
        const bool c1 = bc.cur != 0;
        gather_gauges(a, bc, c1 ? a.e[1] : a.e[0], c1 ? a.qx[1] : a.qx[0], c1 ? a.qy[1] : a.qy[0], tid, 64 * SW_WAVES);
    }
    const float dtmin = tile_or_strips<float>(args, bc, tile, o.x, o.y, rows, s, s_fail);
    block_dt_min(again<float>(args), slot, dtmin, s_red, blockIdx.x);
}

// control blocks of the scenarios at launch slot `slot`, gathered for one copy (a free
// scenario slot has a zeroed argument block and is skipped)
__global__ void k_gather_ctrl(const StepArgs<float> *args, const int n, const int slot, Ctrl *out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && args[i].ctrl) out[i] = args[i].ctrl[slot];
}

}  // namespace thy
