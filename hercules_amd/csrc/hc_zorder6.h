// 6th-order wall-normal operators (hc_params.zorder = 6), column side.
//
// The reference is 2nd order in z (src/module_cnvdiff.f90:89,121,
// src/module_poisson_solver.f90:32-122).  With zorder = 6 the implicit
// operators of a column are
//   u, v, t:  I + rc (-hxy - kappa Z)      Z = ZO_C2_* (7-point d2/dz2, centres)
//   w:        I + rc (-hxy - kappa Z)      Z = ZO_F2   (7-point d2/dz2, faces)
//   p:        rc (hxy + ZO_P)              ZO_P = ZO_D o ZO_G
// with hxy the horizontal symbol the 2nd-order rows use.  They are banded
// (half band 5, and 7 for ZO_P) and solved directly, one thread per column
// (k_z6_band, hc_band6.h).  A column pass of the step is a sequence of
// launches, each one thread per (l, m) column streaming along z:
// right-hand sides (spectral path), the Helmholtz solves, the divergence,
// the pressure solve, then the projection and the pressure increment.
// Arithmetic is FP64; the spectra are stored in FP64 or (mixed variant)
// FP32, the pressure correction phi always in FP64.
#pragma once

#include "hc_band6.h"

// The 6th-order interpolants of the substep's fields, once per point, for
// the right-hand-side kernels: u, v at the w face of level k (the top wall
// face included), w at the centre of level k, t at the interior w face k.
// One thread per (i, j) column, field (blockIdx.y: u, v, w, t) and z chunk
// (blockIdx.z of gridDim.z) streams along z with a window of kIntWin levels,
// k-kIntHW .. k+kIntHW around the row k being formed, and applies the band
// rows ZB_IU_* and ZB_IFC, staged in LDS (FP64 at 256x256x257 423 -> 207 us,
// 9.2 fields of 135 MB; see z6_stream).  The window holds the wall
// data of the C convention at levels -1 and nz (u: -u_mrf, and -u_mrf or
// du/dz = 0 at the top; v: 0; t: tbot, and ttop or the wall gradient) and
// zero beyond; w is zero outside its interior faces 0..nz-2.  The band rows
// list the stencil weights in the stencils' own order with zeros between
// them, so each value equals the accessor's sum term for term, in the stored
// type R.
constexpr int kIntWin = 2 * kIntHW + 1;
template <class R>
__global__ __launch_bounds__(256) void k_zinterp6(StepArgsT<R> A, R *fu, R *fv, R *cw, R *ft)
{
    constexpr int PF = 8;
    extern __shared__ double band_sm[];
    const int nz = A.nz, f = (int)blockIdx.y;
    const size_t plane = (size_t)A.nx * A.ny;
    const size_t col = blockIdx.x * (size_t)256 + threadIdx.x;
    const ZChunk z = z_chunk(nz);
    const int band = f == 2 ? ZB_IFC : (f == 3 ? A.tbc_top : A.ochannel) ? ZB_IU_DN : ZB_IU_DD;
    stage_bands(A.zband, nz, z, {band}, band_sm);
    if (col >= plane || (f == 3 && !ft) || z.kb >= z.ke) return;
    const int kb = z.kb, ke = z.ke;
    const R zero = R(0.0);
    // the field's data, its stored levels lo .. nlev-1, wall data at levels
    // -1 and nz, band and output
    const R *src;
    R *dst, wb = zero, wt = zero;
    int nlev = nz;
    if (f == 0) {
        src = A.u; dst = fu;
        wb = R(-A.u_mrf);
        wt = A.ochannel == 0 ? R(-A.u_mrf) : zero;
    } else if (f == 1) {
        src = A.v; dst = fv;
    } else if (f == 2) {
        src = A.w; dst = cw; nlev = nz - 1;
    } else {
        src = A.t; dst = ft;
        wb = A.tbot;
        wt = A.tbc_top ? R(A.gdz_top * A.lev[LV_IDZT * nz + nz - 1]) : A.ttop;
    }
    if (f == 2) wb = wt = zero;  // w: zero at both wall faces
    auto load = [&](int li) __attribute__((always_inline)) { return src[(size_t)min(max(li, 0), nlev - 1) * plane + col]; };
    auto level = [&](int li, R v) __attribute__((always_inline)) {
        return li >= 0 && li < nlev ? v : (li == -1 ? wb : (li == nz ? wt : zero));
    };
    R win[kIntWin], ring[PF], first[kIntWin - 1];
#pragma unroll
    for (int t = 0; t < kIntWin - 1; ++t) first[t] = load(kb - kIntHW + t);
#pragma unroll
    for (int u = 0; u < PF; ++u) ring[u] = load(kb + kIntHW + u);
#pragma unroll
    for (int t = 0; t < kIntWin - 1; ++t) win[t + 1] = level(kb - kIntHW + t, first[t]);
    for (int k0 = kb; k0 < ke; k0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int k = k0 + u;
            if (k >= ke) return;
#pragma unroll
            for (int t = 0; t < kIntWin - 1; ++t) win[t] = win[t + 1];
            win[kIntWin - 1] = level(k + kIntHW, ring[u]);
            ring[u] = load(k + PF + kIntHW);
            R acc = zero;
            const double *b = band_row(band_sm, z, 0, k) + kBandMax - kIntHW;
#pragma unroll
            for (int t = 0; t < kIntWin; ++t) acc += R(b[t]) * win[t];
            dst[(size_t)k * plane + col] = f == 3 && k == nz - 1 ? zero : acc;
        }
    }
}

// ---------------------------------------------------------------------------
// z terms of the FD right-hand sides (get_momentum_cnvdiff,
// get_temperature_cnvdiff with the 6th-order operators), once per point for
// the tiles that add the horizontal ones (k_rhs_mom_march with ZO = 6, k_rhs_t2):
//   e = 0, 1: d(uw)/dz, d2u/dz2 (of v) into ff, qu (gg, qv)
//   e = 2:    d(ww)/dz - got (t - t_ref), and nu dt/2 d2w/dz2 - dt dp/dz over
//             rc into hh, qw (levels below the top)
//   e = 3:    d(tw)/dz, d2t/dz2 into ss, qt
// One thread per (i, j) column, equation (e0 + blockIdx.y) and z chunk streams
// along z with windows of kWin levels, as the spectral path's column kernels
// (192x128x129: 259 us a substep with the band rows read in the loop, 141 so).
// The fluxes through a face are formed once, where the accessors formed six
// per point; a wall face carries none.
// The window of a face quantity holds face kw at level kw; the band rows ZB_D
// and ZB_F2 leave out the wall faces, ZB_C2_* the wall data, whose terms
// zwall adds.
template <class R>
HC_DEV R zwall(const StepArgsT<R> &A, int op, int k, R bot, R top, bool has_top)
{
    if (k >= 4 && k < A.nz - 4) return R(0);  // no stencil of these reaches a wall
    const size_t e = (size_t)op * A.nz + k;
    const int s = A.zst[e], jt = A.nz + 1 - s;
    const double *w = A.zwt + e * kZW;
    R v = R(0);
    if (s == 0) v += R(w[0]) * bot;
    if (has_top && jt < A.zn2) v += R(w[jt]) * top;
    return v;
}
// NR stored values per level (load, of any level 0 .. nrows) become NW window
// entries (make); NP values of the row itself (point).  The loads run PF rows
// ahead, as z6_stream's.
template <int NR, int NW, int NP, class R, class Load, class Make, class Point, class Row>
HC_DEV void zterm_stream(const ZChunk &z, int nlev, Load &&load, Make &&make, Point &&point, Row &&row)
{
    constexpr int PF = 4;
    const int kb = z.kb, ke = z.ke;
    R win[NW][kWin], ring[PF][NR], pring[PF][NP];
    auto lev = [&](int li) { return min(max(li, 0), nlev - 1); };
    auto enter = [&](int li, const R (&v)[NR]) __attribute__((always_inline)) {
        R in[NW];
        make(li, v, in);
#pragma unroll
        for (int f = 0; f < NW; ++f) {
#pragma unroll
            for (int t = 0; t < kWin - 1; ++t) win[f][t] = win[f][t + 1];
            win[f][kWin - 1] = in[f];
        }
    };
#pragma unroll
    for (int f = 0; f < NW; ++f)
#pragma unroll
        for (int t = 0; t < kWin; ++t) win[f][t] = R(0);
    static_assert((kWin - 1) % 2 == 0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        R first[(kWin - 1) / 2][NR];
#pragma unroll
        for (int t = 0; t < (kWin - 1) / 2; ++t) load(lev(kb - kBandMax + h * (kWin - 1) / 2 + t), first[t]);
#pragma unroll
        for (int t = 0; t < (kWin - 1) / 2; ++t) enter(kb - kBandMax + h * (kWin - 1) / 2 + t, first[t]);
    }
#pragma unroll
    for (int u = 0; u < PF; ++u) {
        load(lev(kb + kBandMax + u), ring[u]);
        point(min(kb + u, ke - 1), pring[u]);
    }
    for (int k0 = kb; k0 < ke; k0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int k = k0 + u;
            if (k >= ke) return;
            enter(k + kBandMax, ring[u]);
            R pt[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) pt[p] = pring[u][p];
            load(lev(k + PF + kBandMax), ring[u]);
            point(min(k + PF, ke - 1), pring[u]);
            row(k, win, pt);
        }
    }
}
template <class R>
HC_DEV R zdot(const double *b, const R (&x)[kWin])
{
    R acc = R(0);
#pragma unroll
    for (int t = 0; t < kWin; ++t) acc += R(b[t]) * x[t];
    return acc;
}

template <int CDS, class R>
__global__ __launch_bounds__(256) void k_z6_terms(StepArgsT<R> A, int e0)
{
    const int nx = A.nx, ny = A.ny, nz = A.nz, e = e0 + (int)blockIdx.y;
    const size_t plane = (size_t)nx * ny, col = blockIdx.x * (size_t)256 + threadIdx.x;
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(e == 2 ? nz - 1 : nz);
    const bool grad = e == 3 ? A.tbc_top != 0 : A.ochannel != 0;
    stage_bands(A.zband, nz, z, {e == 2 ? ZB_G : ZB_D, e == 2 ? ZB_F2 : grad ? ZB_C2_DN : ZB_C2_DD}, band_sm);
    if (col >= plane || z.kb >= z.ke) return;
    const int j = (int)(col / nx), i = (int)(col - (size_t)j * nx);
    auto none = [](int, R (&p)[1]) { p[0] = R(0); };
    auto dot = [&](int b, int k, const R (&x)[kWin]) __attribute__((always_inline)) { return zdot(band_row(band_sm, z, b, k), x); };
    if (e < 2) {
        // neighbours of w across x (u) or y (v): the face interpolant whx, why
        const R *f = e == 0 ? A.u : A.v, *zf = e == 0 ? A.zfu : A.zfv;
        R *conv = e == 0 ? A.ff : A.gg, *dif = reinterpret_cast<R *>(e == 0 ? A.s0 : A.s1);
        size_t o[4];
#pragma unroll
        for (int d = 0; d < 4; ++d)
            o[d] = e == 0 ? (size_t)j * nx + wrapi(i + d - 1, nx) : (size_t)wrapi(j + d - 1, ny) * nx + i;
        const R wall = e == 0 ? R(-A.u_mrf) : R(0);
        const int op = A.ochannel ? ZO_C2_DN : ZO_C2_DD;
        zterm_stream<6, 2, 1, R>(z, nz,
            [&](int li, R (&v)[6]) __attribute__((always_inline)) {
                const size_t b = (size_t)li * plane;
                v[0] = f[b + col];
                v[1] = zf[b + col];
#pragma unroll
                for (int d = 0; d < 4; ++d) v[2 + d] = A.w[b + o[d]];
            },
            [&](int li, const R (&v)[6], R (&in)[2]) __attribute__((always_inline)) {
                in[0] = li >= 0 && li < nz ? v[0] : R(0);
                const R wh = CDS == 1 ? R(0.5) * (v[4] + v[3])
                                      : (-v[5] + R(9.0) * v[4] + R(9.0) * v[3] - v[2]) / R(16.0);
                in[1] = li >= 0 && li < nz - 1 ? v[1] * wh : R(0);
            },
            none,
            [&](int k, const R (&win)[2][kWin], const R (&)[1]) __attribute__((always_inline)) {
                const size_t c = (size_t)k * plane + col;
                conv[c] = dot(0, k, win[1]);
                dif[c] = dot(1, k, win[0]) + zwall<R>(A, op, k, wall, wall, A.ochannel == 0);
            });
    } else if (e == 2) {
        R *qw = reinterpret_cast<R *>(A.s2);
        const R cn = R(0.5) * A.dt * A.nu;
        const R *zt = A.isscalar ? A.zft : A.zcw;
        zterm_stream<3, 3, 1, R>(z, nz,
            [&](int li, R (&v)[3]) __attribute__((always_inline)) {
                const size_t b = (size_t)li * plane + col;
                v[0] = A.w[b];
                v[1] = A.p[b];
                v[2] = A.zcw[b];
            },
            [&](int li, const R (&v)[3], R (&in)[3]) __attribute__((always_inline)) {
                const bool on = li >= 0 && li < nz;
                in[0] = on && li < nz - 1 ? v[0] : R(0);
                in[1] = on ? v[1] : R(0);
                in[2] = on ? sq(v[2]) : R(0);
            },
            // without temperature a value that is there and is not used
            [&](int k, R (&p)[1]) __attribute__((always_inline)) { p[0] = zt[(size_t)k * plane + col]; },
            [&](int k, const R (&win)[3][kWin], const R (&p)[1]) __attribute__((always_inline)) {
                const size_t c = (size_t)k * plane + col;
                R con = dot(0, k, win[2]);
                if (A.isscalar) con -= A.got * (p[0] - A.t_ref);
                A.hh[c] = con;
                qw[c] = cn * dot(1, k, win[0]) - A.dt * dot(0, k, win[1]);
            });
    } else {
        R *qt = reinterpret_cast<R *>(A.s0);
        const R top = A.tbc_top ? R(A.gdz_top * A.lev[LV_IDZT * nz + nz - 1]) : A.ttop;
        const int op = A.tbc_top ? ZO_C2_DN : ZO_C2_DD;
        zterm_stream<3, 2, 1, R>(z, nz,
            [&](int li, R (&v)[3]) __attribute__((always_inline)) {
                const size_t b = (size_t)li * plane + col;
                v[0] = A.t[b];
                v[1] = A.zft[b];
                v[2] = A.w[b];
            },
            [&](int li, const R (&v)[3], R (&in)[2]) __attribute__((always_inline)) {
                in[0] = li >= 0 && li < nz ? v[0] : R(0);
                in[1] = li >= 0 && li < nz - 1 ? v[1] * v[2] : R(0);
            },
            none,
            [&](int k, const R (&win)[2][kWin], const R (&)[1]) __attribute__((always_inline)) {
                const size_t c = (size_t)k * plane + col;
                A.ss[c] = dot(0, k, win[1]);
                qt[c] = dot(1, k, win[0]) + zwall<R>(A, op, k, A.tbot, top, true);
            });
    }
}
