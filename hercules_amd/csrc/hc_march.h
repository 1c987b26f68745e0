// Momentum right-hand side of the FD substep on x-y tiles that march up a run
// of levels (get_momentum_cnvdiff, src/module_cnvdiff.f90:35-374, with the
// interpolants of src/module_tools.f90:410-470 and the wall rules of
// src/module_boundary.f90:33-290).
#pragma once

#include "hc_xfer.h"

// The multiply-adds of the interpolants are written out, so that a value is
// rounded the same wherever it is formed (a run's first level forms the
// fluxes of the level below, which other runs carry).
HC_DEV double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
HC_DEV float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// value halfway between f0 and f1 of four consecutive entries
template <int CDS, class R>
HC_DEV R mid4(R fm, R f0, R f1, R f2)
{
    if (CDS == 1) return R(0.5) * (f0 + f1);
    return (fma_(R(9.0), f0, fma_(R(9.0), f1, -f2)) - fm) * R(0.0625);
}
// value at a level's face from the levels above and below it
template <class R>
HC_DEV R zface(R up, R dn, R lt) { return fma_(up, lt, dn * (R(1.0) - lt)); }
// difference across the middle of four consecutive face values, without the spacing
template <int CDS, class R>
HC_DEV R dif4(R fm, R f0, R f1, R f2)
{
    if (CDS == 1) return f1 - f0;
    return -f2 + R(27.0) * f1 - R(27.0) * f0 + fm;
}

// the parts of a point's equations are kept apart in the schedule: all of
// their LDS reads issued at once take 214 VGPRs (FP64), in parts 149
#define HC_SB __builtin_amdgcn_sched_barrier(0)

// LDS rows of S = TX + 6 points (x halo 3) of one level
template <int TX, int TY>
struct MarchTile {
    static constexpr int S = TX + 6;
    static constexpr int RU = TY + 6;  // u, v, w: rows j0-3 .. j0+TY+2
    static constexpr int RP = TY + 3;  // p:       rows j0-1 .. j0+TY+1
    static constexpr int OU = 0, OV = RU, OW = 2 * RU, OP = 3 * RU, NRAW = 3 * RU + RP;
    static constexpr int RF = TY + 3;  // uhy*vhx: rows j0-2 .. j0+TY, columns i0-2 .. i0+TX
};

// One thread per point of a TX x TY tile.  A block forms levels k0 .. k1-1 in
// turn: LDS holds the raw u, v, w, p rows of levels k and k+1, registers the
// loads of level k+2 (issued before level k is formed, stored after it) and,
// from the level below, the point's u, v, w and its vertical fluxes.  So a
// value is fetched once per block and its z neighbours cost no load, and the
// address of each staged value is a pointer that advances by one plane.
// uhy*vhx, which eight points share, goes through LDS; the other
// interpolants are formed where they are used from the rows the Laplacians
// read anyway.  f, g, h are stored; qu, qv, qw go as physical rows into the
// storage of their spectra (a row of nx values takes the bytes of its nx/2
// modes), which launch_r2c_n then transforms in place.
// ZO = 6 (6th- and 4th-order z): the z terms at a point are k_z6_terms', left
// where the outputs go, and the rows of level k+1 give way to those of u and v
// at the faces of level k (zfu, zfv).
// A level costs a thread 270 FP64 and 76 other VALU instructions and 56 LDS
// reads; HBM and the latency of its two barriers at three waves per SIMD
// bound it (held to 128 VGPRs for four waves, the loads in flight spill and
// the launch takes 0.81 instead of 0.47 ms at 256x256x257).  Tiles of 32x8
// are the fastest in FP64: with the x transform 0.61 ms per substep at
// 256x256x257 (64x4 0.64, 64x8 and 32x16, of 512 threads, 0.68), where the
// same tiles restaged level by level took 0.66 and whole rows fused with the
// transform 0.83; 3.9 ms at 512x512x385 (one row per block: 16.0).
template <int CDS, int TX, int TY, class R, int ZO = 2>
__global__ __launch_bounds__(TX * TY, sizeof(R) == 8 ? 3 : 4) void k_rhs_mom_march(StepArgsT<R> A)
{
    using Tl = MarchTile<TX, TY>;
    constexpr int D0 = CDS == 1 ? 1 : 0, D1 = CDS == 1 ? 3 : 4;  // faces at -2 .. 1 of a point (cds 1: -1, 0)
    constexpr int T = TX * TY, S = Tl::S, NV = Tl::NRAW * S, NU = Tl::RU * S, NPV = Tl::RP * S;
    constexpr int NF = ZO == 6 ? 5 : 3;
    constexpr int LEFT = NU % T, REST = NF * LEFT <= T ? LEFT : 0, NM = NU / T + (LEFT > REST ? 1 : 0);
    constexpr int NP = (NPV + T - 1) / T;
    __shared__ R raw[2][NV];
    __shared__ R fuv[Tl::RF * S];
    const int tid = threadIdx.x, nx = A.nx, ny = A.ny, nz = A.nz;
    const int ntx = nx / TX, ntile = ntx * (ny / TY);
    // tiles of one run of levels are neighbours in an XCD's L2
    const int logical = xcd_remap(blockIdx.x, (int)gridDim.x);
    const int run = logical / ntile, tl = logical - run * ntile;
    const int k0 = A.klo + run * A.kchunk, k1 = min(k0 + A.kchunk, A.klo + A.nlev);
    const int i0 = (tl % ntx) * TX, j0 = (tl / ntx) * TY;
    const int il = tid % TX, jj = tid / TX, i = i0 + il, j = j0 + jj, xl = il + 3;
    const size_t plane = (size_t)nx * ny;
    // staged values of a level: NM per thread and field of u, v, w (offsets
    // in the plane common to the three), what is left of each shared by the
    // threads of one more slot, and NP of p
    unsigned ouv[NM], op[NP];
    const R *rest = A.u;
    int rest_at = -1;
    auto src_off = [&](int r, int x) __attribute__((always_inline)) {
        return (unsigned)wrapi(r, ny) * (unsigned)nx + (unsigned)wrapi(i0 - 3 + x, nx);
    };
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const int q = min(tid + m * T, NU - 1), r = q / S;
        ouv[m] = src_off(j0 - 3 + r, q - r * S);
    }
#pragma unroll
    for (int m = 0; m < NP; ++m) {
        const int q = min(tid + m * T, NPV - 1), r = q / S;
        op[m] = src_off(j0 - 1 + r, q - r * S);
    }
    if constexpr (REST > 0) {
        if (tid < NF * REST) {
            const int fd = tid / REST, q = NM * T + tid - fd * REST, r = q / S;
            rest = (fd == 0 ? A.u : fd == 1 ? A.v : fd == 2 ? A.w : fd == 3 ? A.zfu : A.zfv) +
                   src_off(j0 - 3 + r, q - r * S);
            rest_at = fd < 3 ? fd * NU + q : NV + (fd - 3) * NU + q;
        }
    }
    struct Level {
        R f[NF][NM], p[NP], x;
    };
    auto fetch = [&](Level &v, int k) __attribute__((always_inline)) {
        const size_t lo = (size_t)k * plane;
        const R *ub = A.u + lo, *vb = A.v + lo, *wb = A.w + lo, *pb = A.p + lo;
#pragma unroll
        for (int m = 0; m < NM; ++m) { v.f[0][m] = ub[ouv[m]]; v.f[1][m] = vb[ouv[m]]; v.f[2][m] = wb[ouv[m]]; }
        if constexpr (ZO == 6) {
            const R *fu = A.zfu + lo, *fv = A.zfv + lo;
#pragma unroll
            for (int m = 0; m < NM; ++m) { v.f[3][m] = fu[ouv[m]]; v.f[4][m] = fv[ouv[m]]; }
        }
#pragma unroll
        for (int m = 0; m < NP; ++m) v.p[m] = pb[op[m]];
        if constexpr (REST > 0) v.x = rest_at >= 0 ? rest[lo] : R(0);
    };
    auto put = [&](R *dst, const Level &v) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NM; ++m)
            if (m < NM - 1 || NU >= NM * T || tid + m * T < NU) {
#pragma unroll
                for (int fd = 0; fd < NF; ++fd) dst[(fd < 3 ? fd * NU : NV + (fd - 3) * NU) + tid + m * T] = v.f[fd][m];
            }
#pragma unroll
        for (int m = 0; m < NP; ++m)
            if (m < NP - 1 || NPV >= NP * T || tid + m * T < NPV) dst[3 * NU + tid + m * T] = v.p[m];
        if constexpr (REST > 0)
            if (rest_at >= 0) dst[rest_at] = v.x;
    };
    const bool two = ZO == 2 && k0 + 1 < nz;
    {
        Level a;
        fetch(a, k0);
        put(raw[0], a);
        if (two) {
            fetch(a, k0 + 1);
            put(raw[1], a);
        }
    }
    // the level below: wall values (src/module_boundary.f90:52-107) or u, v, w
    // at k0-1 and the fluxes uhz*whx, vhz*why of its face
    const R um = A.u_mrf;
    const size_t cp = (size_t)j * nx + i;
    R ukm = R(0), vkm = R(0), wkm = R(0), fuw_km = R(0), fwv_km = R(0);
    R wx[4], wy[3];
    const bool bot = k0 == 0;
    if (ZO == 2 && !bot) {
        const size_t lo = (size_t)(k0 - 1) * plane;
        ukm = A.u[lo + cp];
        vkm = A.v[lo + cp];
#pragma unroll
        for (int d = 0; d < 4; ++d) wx[d] = A.w[lo + (size_t)j * nx + wrapi(i + d - 1, nx)];
        wy[0] = A.w[lo + (size_t)wrapi(j - 1, ny) * nx + i];
        wy[1] = A.w[lo + (size_t)wrapi(j + 1, ny) * nx + i];
        wy[2] = A.w[lo + (size_t)wrapi(j + 2, ny) * nx + i];
        wkm = wx[1];
    }
    size_t c = (size_t)k0 * plane + cp;
    R tk = A.isscalar ? A.t[c] : R(0);
    const R dpx = A.dp_opt == 2 ? R(A.scal[0]) : A.dpx;
    __syncthreads();
    if constexpr (ZO == 2) {
        const R u0 = raw[0][(Tl::OU + jj + 3) * S + xl], v0 = raw[0][(Tl::OV + jj + 3) * S + xl];
        if (bot) {
            ukm = -u0 - R(2.0) * um;
            vkm = -v0;
        } else {
            const R lt = A.lev[LV_LT * nz + k0 - 1];
            fuw_km = zface(u0, ukm, lt) * mid4<CDS>(wx[0], wx[1], wx[2], wx[3]);
            fwv_km = zface(v0, vkm, lt) * mid4<CDS>(wy[0], wx[1], wy[1], wy[2]);
        }
    }
    for (int k = k0, b = 0; k < k1; ++k, b ^= 1) {
        const R *cur = raw[ZO == 6 ? 0 : b], *nxt = raw[ZO == 6 ? 1 : b ^ 1];
        const bool top = k == nz - 1, more = k + 1 < k1, ahead = more && (ZO == 6 || k + 2 < nz);
        Level pre;
        if (ahead) fetch(pre, ZO == 6 ? k + 1 : k + 2);
        R o0 = R(0), o1 = R(0), o2 = R(0), tkp = R(0);
        if (A.use_f0) { o0 = A.ff0[c]; o1 = A.gg0[c]; o2 = A.hh0[c]; }
        if (ZO == 2 && A.isscalar && !top) tkp = A.t[c + plane];
        R z[6];  // ZO = 6: k_z6_terms' values at the point
        if constexpr (ZO == 6) {
            z[0] = A.ff[c]; z[1] = A.gg[c]; z[2] = A.hh[c];
            z[3] = reinterpret_cast<const R *>(A.s0)[c];
            z[4] = reinterpret_cast<const R *>(A.s1)[c];
            z[5] = reinterpret_cast<const R *>(A.s2)[c];
        }
        // uhy*vhx, which the points of two rows and columns on either side read
        for (int e = tid; e < Tl::RF * (TX + 3); e += T) {
            const int r = e / (TX + 3), x = 1 + e - r * (TX + 3);
            const R *pu = cur + (Tl::OU + r + 1) * S + x, *pv = cur + (Tl::OV + r + 1) * S + x;
            fuv[r * S + x] = mid4<CDS>(pu[-S], pu[0], pu[S], pu[2 * S]) * mid4<CDS>(pv[-1], pv[0], pv[1], pv[2]);
        }
        __syncthreads();
        const R *pu = cur + (Tl::OU + jj + 3) * S + xl, *pv = cur + (Tl::OV + jj + 3) * S + xl;
        const R *pw = cur + (Tl::OW + jj + 3) * S + xl, *pp = cur + (Tl::OP + jj + 1) * S + xl;
        const R *qu_ = nxt + (Tl::OU + jj + 3) * S + xl, *qv_ = nxt + (Tl::OV + jj + 3) * S + xl;
        const R *F = fuv + (jj + 2) * S + xl;
        const R idz = A.lev[LV_IDZ * nz + k], idzt = A.lev[LV_IDZT * nz + k], idzb = A.lev[LV_IDZB * nz + k];
        const R lt = A.lev[LV_LT * nz + k];
        const R cn = A.rc * R(0.5) * A.dt * A.nu, cdt = A.rc * A.dt;
        const R u0 = pu[0], v0 = pv[0], w0 = pw[0];
        R f, g, h = R(0), qu, qv, qw = R(0);
        R fuw = R(0), fwv = R(0);  // fluxes through this level's face (zero on the top wall, as w)
        if (!top) {  // ---- W equation (:274-370), k < kend3
            R con, wx_, lap;
            {
                R r[7], m[4] = {}, x[4] = {};
#pragma unroll
                for (int d = 0; d < 7; ++d) r[d] = pw[d - 3];
#pragma unroll
                for (int d = D0; d < D1; ++d) {
                    m[d] = mid4<CDS>(r[d], r[d + 1], r[d + 2], r[d + 3]);
                    x[d] = (ZO == 6 ? qu_[d - 2] : zface(qu_[d - 2], pu[d - 2], lt)) * m[d];
                }
                fuw = x[2];
                con = dif4<CDS>(x[0], x[1], x[2], x[3]) * (CDS == 1 ? A.idx : A.c24x);
                wx_ = dif4<CDS>(m[0], m[1], m[2], m[3]) * (CDS == 1 ? A.idx : A.c24x);
                lap = CDS == 1 ? (r[4] - R(2.0) * w0 + r[2]) * A.idx2
                               : (-r[5] + R(16.0) * r[4] - R(30.0) * w0 + R(16.0) * r[2] - r[1]) * A.c12x2;
            }
            HC_SB;
            {
                R r[7], x[4] = {};
#pragma unroll
                for (int d = 0; d < 7; ++d) r[d] = pw[(d - 3) * S];
#pragma unroll
                for (int d = D0; d < D1; ++d)
                    x[d] = (ZO == 6 ? qv_[(d - 2) * S] : zface(qv_[(d - 2) * S], pv[(d - 2) * S], lt)) *
                           mid4<CDS>(r[d], r[d + 1], r[d + 2], r[d + 3]);
                fwv = x[2];
                con += dif4<CDS>(x[0], x[1], x[2], x[3]) * (CDS == 1 ? A.idy : A.c24y);
                lap += CDS == 1 ? (r[4] - R(2.0) * w0 + r[2]) * A.idy2
                                : (-r[5] + R(16.0) * r[4] - R(30.0) * w0 + R(16.0) * r[2] - r[1]) * A.c12y2;
            }
            if constexpr (ZO == 6) {
                h = -con - z[2] - um * wx_;
                qw = w0 + A.dt * (A.ra * h + A.rb * o2) + cn * lap + A.rc * z[5];
            } else {
                const R wkp = k + 1 == nz - 1 ? R(0) : nxt[(Tl::OW + jj + 3) * S + xl];
                const R pkp = nxt[(Tl::OP + jj + 1) * S + xl];
                const R wwz = (sq(R(0.5) * (w0 + wkp)) - sq(R(0.5) * (w0 + wkm))) * idzt;
                const R wzz = ((wkp - w0) * A.lev[LV_IDZ * nz + k + 1] - (w0 - wkm) * idz) * idzt;
                h = -con - wwz - um * wx_;
                if (A.isscalar) h += A.got * (zface(tkp, tk, lt) - A.t_ref);
                qw = w0 + A.dt * (A.ra * h + A.rb * o2) + cn * (lap + wzz) - cdt * ((pkp - pp[0]) * idzt);
            }
        }
        A.hh[c] = h;
        reinterpret_cast<R *>(A.s2)[c] = qw;
        HC_SB;
        {   // ---- U equation (:55-161)
            R con, ux, lap, dpdx;
            {
                R r[7];
#pragma unroll
                for (int d = 0; d < 7; ++d) r[d] = pu[d - 3];
                R m[4] = {};
#pragma unroll
                for (int d = D0; d < D1; ++d) m[d] = mid4<CDS>(r[d], r[d + 1], r[d + 2], r[d + 3]);
                if (CDS == 1) {  // faces between i-1, i and i, i+1
                    con = (sq(m[2]) - sq(m[1])) * A.idx;
                    ux = (m[2] - m[1]) * A.idx;
                    lap = (r[4] - R(2.0) * u0 + r[2]) * A.idx2;
                    dpdx = (pp[1] - pp[0]) * A.idx;
                } else {
                    con = dif4<2>(sq(m[0]), sq(m[1]), sq(m[2]), sq(m[3])) * A.c24x;
                    ux = dif4<2>(m[0], m[1], m[2], m[3]) * A.c24x;
                    lap = (-r[5] + R(16.0) * r[4] - R(30.0) * u0 + R(16.0) * r[2] - r[1]) * A.c12x2;
                    dpdx = dif4<2>(pp[-1], pp[0], pp[1], pp[2]) * A.c24x;
                }
            }
            HC_SB;
            if (CDS == 1) {
                con += (F[0] - F[-S]) * A.idy;
                lap += (pu[S] - R(2.0) * u0 + pu[-S]) * A.idy2;
            } else {
                con += dif4<2>(F[-2 * S], F[-S], F[0], F[S]) * A.c24y;
                lap += (-pu[2 * S] + R(16.0) * pu[S] - R(30.0) * u0 + R(16.0) * pu[-S] - pu[-2 * S]) * A.c12y2;
            }
            const R ukp = top ? (A.ochannel == 0 ? -u0 - R(2.0) * um : u0) : qu_[0];
            const R uwz = ZO == 6 ? z[0] : (fuw - fuw_km) * idz;
            const R uzz = ZO == 6 ? z[3] : ((ukp - u0) * idzt - (u0 - ukm) * idzb) * idz;
            if (A.dp_opt == 3) {
                const R x0 = mid4<CDS>(pv[-1], v0, pv[1], pv[2]), x1 = mid4<CDS>(pv[-S - 1], pv[-S], pv[-S + 1], pv[-S + 2]);
                f = -con - uwz - um * ux + A.fc * (R(0.5) * (x0 + x1) - A.vg);
            } else {
                f = -con - uwz + dpx - um * ux;
            }
            qu = u0 + A.dt * (A.ra * f + A.rb * o0) + cn * (lap + uzz) - cdt * dpdx;
            A.ff[c] = f;
            reinterpret_cast<R *>(A.s0)[c] = qu;
        }
        HC_SB;
        {   // ---- V equation (:166-270)
            R con, vx = R(0), lap, dpdy;
            {
                R r[7], m[4] = {};
#pragma unroll
                for (int d = 0; d < 7; ++d) r[d] = pv[(d - 3) * S];
#pragma unroll
                for (int d = D0; d < D1; ++d) m[d] = sq(mid4<CDS>(r[d], r[d + 1], r[d + 2], r[d + 3]));
                con = dif4<CDS>(m[0], m[1], m[2], m[3]) * (CDS == 1 ? A.idy : A.c24y);
                lap = CDS == 1 ? (r[4] - R(2.0) * v0 + r[2]) * A.idy2
                               : (-r[5] + R(16.0) * r[4] - R(30.0) * v0 + R(16.0) * r[2] - r[1]) * A.c12y2;
                dpdy = CDS == 1 ? (pp[S] - pp[0]) * A.idy : dif4<2>(pp[-S], pp[0], pp[S], pp[2 * S]) * A.c24y;
            }
            HC_SB;
            con += CDS == 1 ? (F[0] - F[-1]) * A.idx : dif4<2>(F[-2], F[-1], F[0], F[1]) * A.c24x;
            if (um != R(0)) {
                R m[4] = {};
#pragma unroll
                for (int d = D0; d < D1; ++d) m[d] = mid4<CDS>(pv[d - 3], pv[d - 2], pv[d - 1], pv[d]);
                vx = dif4<CDS>(m[0], m[1], m[2], m[3]) * (CDS == 1 ? A.idx : A.c24x);
            }
            lap += CDS == 1 ? (pv[1] - R(2.0) * v0 + pv[-1]) * A.idx2
                            : (-pv[2] + R(16.0) * pv[1] - R(30.0) * v0 + R(16.0) * pv[-1] - pv[-2]) * A.c12x2;
            const R vkp = top ? (A.ochannel == 0 ? -v0 : v0) : qv_[0];
            const R vwz = ZO == 6 ? z[1] : (fwv - fwv_km) * idz;
            const R vzz = ZO == 6 ? z[4] : ((vkp - v0) * idzt - (v0 - vkm) * idzb) * idz;
            g = -con - vwz - um * vx;
            if (A.dp_opt == 3) {
                const R a0 = mid4<CDS>(pu[-S], u0, pu[S], pu[2 * S]), a1 = mid4<CDS>(pu[-S - 1], pu[-1], pu[S - 1], pu[2 * S - 1]);
                g += A.fc * (A.ug - R(0.5) * (a0 + a1) - um);
            }
            qv = v0 + A.dt * (A.ra * g + A.rb * o1) + cn * (lap + vzz) - cdt * dpdy;
            A.gg[c] = g;
            reinterpret_cast<R *>(A.s1)[c] = qv;
        }
        c += plane;
        ukm = u0; vkm = v0; wkm = w0;
        fuw_km = fuw; fwv_km = fwv;
        tk = tkp;
        if (!more) break;
        __syncthreads();
        if (ahead) put(raw[ZO == 6 ? 0 : b], pre);
        if (ZO == 6) __syncthreads();
    }
}
