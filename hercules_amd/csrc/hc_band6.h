// Direct solves of the 6th-order implicit z systems (zorder = 6), one thread
// per (l, m) column.
//
// Every system of the step is real and banded,
//   u, v, t:  (1 - rc hxy) I - rc kappa Z      Z = ZO_C2_* on the levels
//   w:        (1 - rc hxy) I - rc kappa Z      Z = ZO_F2 on the interior faces
//   p:        rc (hxy I + ZO_P)                ZO_P = ZO_D o ZO_G
// and differs between columns only through the horizontal symbol hxy.  Z has
// half band 3 (7-point stencils) but for the first and last two rows, whose
// stencils shift inwards at the walls and reach 5; ZO_P half band 5, and 7 in
// those rows.  Gaussian elimination without pivoting is stable for all of
// them (growth factor below 1.7 on the channel grids), so each thread factors
// its column's matrix row by row while eliminating the right-hand sides.
// U's rows (half band and 1/diagonal) and the eliminated right-hand sides of
// a whole column are more bytes than the right-hand sides themselves, so they
// are not kept: the levels are cut into the first PB, a remainder and segments
// of kBandSeg,
//   pass 1  eliminates from the bottom and keeps, at each segment's start,
//           the rows that the next one depends on (scratch, scr),
//   pass 2  takes the segments from the top: eliminates one again from its
//           start, its rows of U into LDS, and back-substitutes through it.
// Consecutive threads own consecutive l, so every load and store of a level
// is one coalesced line across the wavefront.  The (0,0) mode adds the wall
// data of u and t to the first right-hand side (the Crank-Nicolson implicit
// half) and replaces the first pressure row by the delnull row.
#pragma once


// CI: the stored complex type of the right-hand sides (double2, or float2 in
// the mixed variant); the factorisation and the solve run in FP64.
template <class CI>
struct BandSys {
    const CI *in[2];  // right-hand sides (k, j, l)
    CI *f[2];         // solutions (may be in[])
    double *scr;    // segment starts: PI (PI + 1 + 2 nr) doubles per segment and column
    int nr;         // right-hand sides sharing the matrix: 1 or 2
    int eq;         // 0 u/v, 1 w, 2 p, 3 t
    int fix;        // apply the (0,0)-mode wall data / delnull row
    int trunc;      // zero the columns outside the 2/3 rule on output
};
template <class CI>
struct BandArgs {
    BandSys<CI> s[2];  // one system per blockIdx.y
};

// Wall data of the (0,0) mode for row k of the u (eq 0) or t (eq 3)
// equation: rc kappa times the weight of the wall datum times its value
// (bottom: -u_mrf or tbot; top: -u_mrf for a closed channel, ttop or the
// gradient for t), i.e. the implicit half of the Crank-Nicolson wall terms.
HC_DEV double z6_wall_rhs(const StepArgs &A, int eq, int op, double ck, int k)
{
    const int nz = A.nz;
    if (k >= 4 && k < nz - 4) return 0.0;  // no stencil of these reaches a wall
    double bot, top;
    bool has_top;
    if (eq == 0) {
        bot = -A.u_mrf;
        top = -A.u_mrf;
        has_top = A.ochannel == 0;
    } else {
        bot = A.tbot;
        top = A.tbc_top ? A.gdz_top * A.lev[LV_IDZT * nz + nz - 1] : A.ttop;
        has_top = true;
    }
    const size_t e = (size_t)op * nz + k;
    const int s = A.zst[e];
    const double *w = A.zwt + e * kZW;
    double v = 0.0;
    if (s == 0) v += ck * w[0] * bot;
    const int jt = nz + 1 - s;
    if (has_top && jt < 7) v += ck * w[jt] * top;
    return v;
}

constexpr int kBandSeg = 12;  // levels of a segment
// bytes of LDS of one block (one wavefront): the rows of a segment, the four
// entries of the first two rows beyond the half band, the segment's band rows
template <int PI>
constexpr size_t band_lds(int nr)
{
    return (size_t)((kBandSeg * (PI + 1 + 2 * nr) + 4) + (kBandSeg * (2 * PI + 1) + 63) / 64) * 64 * sizeof(double);
}

// PI: half band of all rows but the first and last two, whose band is PI + 2.
// NR: right-hand sides.  A launch has about one wavefront per SIMD (33,024
// columns at 256x256), so the loads in flight carry the rate: the elimination
// of a segment is straight-line code that loads the next one's right-hand
// sides and band rows as it goes, without a branch around a load, after which
// a wait would be for all of them.  12 levels: U's rows of three blocks fill a
// CU's LDS.  The solves of one step at 256x256x257 (three substeps, u, v, w,
// t, p): 5.5 ms with U kept in memory, 4.9 ms with loads behind branches, 2.0
// ms so (FP32 spectra 4.7 -> 1.6 ms).
template <int PI, int NR, class CI>
HC_DEV void band_solve(const StepArgs &A, const BandSys<CI> &S)
{
    constexpr int PB = PI + 2, SG = kBandSeg, NS = PI * (PI + 1 + 2 * NR), NL_ = PI + 1 + 2 * NR;
    constexpr int W = 2 * PI + 1, TQ = (SG * W + 63) / 64;
    static_assert(SG >= 9);  // the last two rows' stencils stay within the top segment
    extern __shared__ double band_sm[];
    const int lane = threadIdx.x, nl = A.nl, ny = A.ny, nz = A.nz;
    const int ncol = nl * ny;
    // lanes beyond the last column repeat it (same wavefront, same values)
    const int col = min((int)blockIdx.x * 64 + lane, ncol - 1);
    const int l = col % nl, jm = col / nl;
    const size_t plane = (size_t)ncol;
    const bool face = S.eq == 1, pres = S.eq == 2;
    const int n = face ? nz - 1 : nz;
    int band, op;
    double hxy, kap;
    switch (S.eq) {
    case 0:
        band = A.ochannel ? ZB_C2_DN : ZB_C2_DD;
        op = A.ochannel ? ZO_C2_DN : ZO_C2_DD;
        hxy = A.symx[SY_HU * nl + l] + A.symy[SY_HU * ny + jm];
        kap = 0.5 * A.dt * A.nu;
        break;
    case 1:
        band = ZB_F2;
        op = ZO_F2;
        hxy = A.symx[SY_HU * nl + l] + A.symy[SY_HU * ny + jm];
        kap = 0.5 * A.dt * A.nu;
        break;
    case 2:
        band = ZB_P;
        op = ZO_P;
        hxy = A.symx[SY_PX * nl + l] + A.symy[SY_PX * ny + jm];
        kap = 0.0;
        break;
    default:
        band = A.tbc_top ? ZB_C2_DN : ZB_C2_DD;
        op = A.tbc_top ? ZO_C2_DN : ZO_C2_DD;
        hxy = A.symx[SY_HT * nl + l] + A.symy[SY_HT * ny + jm];
        kap = 0.5 * A.dt * A.alpha;
        break;
    }
    const double rc = A.rc, ck = rc * kap;
    const double cdiag = pres ? rc * hxy : 1.0 - rc * hxy, coff = pres ? rc : -ck;
    const bool is00 = S.fix && l == 0 && jm == 0;
    const bool walls = is00 && (S.eq == 0 || S.eq == 3);
    const double *bt = A.zband + (size_t)band * nz * kBandRow + kBandMax;
    // rows 0 .. PB-1, then nrem, then nfull segments.  n >= 15 (16 for p), so
    // the top one, of SG or (nfull = 0) nrem rows, has PB + 2 and more.
    const int nfull = (n - PB) / SG, nrem = n - PB - nfull * SG;
    // LDS: row i of the segment, entry e (U's PI, 1/diagonal, the right-hand
    // sides), and the two entries beyond PI of rows 0 and 1
    auto row = [&](int i, int e) -> double & { return band_sm[(4 + i * NL_ + e) * 64 + lane]; };
    auto wide = [&](int k, int e) -> double & { return band_sm[(2 * k + e) * 64 + lane]; };
    double *tab = band_sm + (4 + SG * NL_) * 64;
    // Every row is rounded as the elimination over the full band rounds it, so
    // that segments of any position agree to the last bit: an entry is the
    // product coff w (the diagonal fma(coff, w, cdiag)), rounded unless its
    // first update is not zero, which takes the product unrounded.
    auto prod = [](double x, double y) -> double {
#pragma clang fp contract(off)
        return x * y;
    };
    auto entry = [&](double w, int d) -> double { return d ? prod(coff, w) : fma(coff, w, cdiag); };
    // band rows of the segment at k0: loaded a segment ahead, then through LDS
    double tq[TQ];
    auto tab_load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TQ; ++j) {
            const int e = lane + 64 * j;
            tq[j] = bt[min(k0 + e / W, nz - 1) * kBandRow + e % W - PI];
        }
    };
    auto tab_put = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < TQ; ++j) tab[lane + 64 * j] = tq[j];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // the PI rows before the current one, oldest first
    struct Win {
        double U[PI][PI], dv[PI];
        double2 y[NR][PI];
    };
    Win w;
    CI ring[SG][NR];
    auto load_rhs = [&](int k, CI (&r)[NR]) __attribute__((always_inline)) {
        const size_t o = (size_t)min(k, n - 1) * plane + col;
#pragma unroll
        for (int e = 0; e < NR; ++e) r[e] = S.in[e][o];
    };
    auto fill = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < SG; ++u) load_rhs(k0 + u, ring[u]);
    };
    auto keep = [&](int i, const double (&u)[PI], double dk, const double2 (&r)[NR]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < PI; ++c) row(i, c) = u[c];
        row(i, PI) = dk;
#pragma unroll
        for (int e = 0; e < NR; ++e) { row(i, PI + 1 + 2 * e) = r[e].x; row(i, PI + 2 + 2 * e) = r[e].y; }
    };
    // rows 0 .. PB-1 from ring with the full band: rows 0 and 1 reach PB to the right
    auto bottom = [&](bool store) __attribute__((always_inline)) {
        double U[PB][PB], dv[PB];
        double2 y[NR][PB];
#pragma unroll
        for (int t = 0; t < PB; ++t) {
            dv[t] = 0.0;
#pragma unroll
            for (int e = 0; e < NR; ++e) y[e][t] = make_double2(0.0, 0.0);
#pragma unroll
            for (int c = 0; c < PB; ++c) U[t][c] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < PB; ++k) {
            double a[2 * PB + 1];
#pragma unroll
            for (int d = -PB; d <= PB; ++d) a[d + PB] = entry(bt[k * kBandRow + d], d);
            double2 r[NR];
#pragma unroll
            for (int e = 0; e < NR; ++e) r[e] = ccast<double2>(ring[k][e]);
            if (k < 3 && walls) r[0].x += z6_wall_rhs(A, S.eq, op, ck, k);
            if (k == 0 && is00 && pres) {  // delnull: b0 phi(0) = 0 (src/module_poisson_solver.f90:558-564)
#pragma unroll
                for (int d = 0; d <= 2 * PB; ++d) a[d] = 0.0;
                a[PB] = rc * (hxy + A.lev[LV_DP00 * nz]);
                r[0] = make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int t = 0; t < PB; ++t) {
                const double lt = a[t] * dv[t];
#pragma unroll
                for (int c = 1; c <= PB; ++c)
                    if (c == PB && t > 0 && k > 0) a[t + PB] = fma(coff, bt[k * kBandRow + t], -prod(lt, U[t][PB - 1]));
                    else a[t + c] -= lt * U[t][c - 1];
#pragma unroll
                for (int e = 0; e < NR; ++e) { r[e].x -= lt * y[e][t].x; r[e].y -= lt * y[e][t].y; }
            }
            const double dk = 1.0 / a[PB];
#pragma unroll
            for (int t = 0; t < PB - 1; ++t) {
                dv[t] = dv[t + 1];
#pragma unroll
                for (int e = 0; e < NR; ++e) y[e][t] = y[e][t + 1];
#pragma unroll
                for (int c = 0; c < PB; ++c) U[t][c] = U[t + 1][c];
            }
            dv[PB - 1] = dk;
#pragma unroll
            for (int e = 0; e < NR; ++e) y[e][PB - 1] = r[e];
#pragma unroll
            for (int c = 0; c < PB; ++c) U[PB - 1][c] = a[PB + 1 + c];
            if (store) {
                double u[PI];
#pragma unroll
                for (int c = 0; c < PI; ++c) u[c] = a[PB + 1 + c];
                keep(k, u, dk, r);
                if (k < 2) { wide(k, 0) = a[PB + 1 + PI]; wide(k, 1) = a[PB + 2 + PI]; }
            }
        }
#pragma unroll
        for (int t = 0; t < PI; ++t) {
            w.dv[t] = dv[t + 2];
#pragma unroll
            for (int e = 0; e < NR; ++e) w.y[e][t] = y[e][t + 2];
#pragma unroll
            for (int c = 0; c < PI; ++c) w.U[t][c] = U[t + 2][c];
        }
    };
    // row k, the i-th of its segment, from the right-hand sides q; into LDS if
    // store; edge: one of the column's last three rows, tail: of its last two
    auto step = [&](int k, int i, const CI (&q)[NR], bool store, bool edge, bool tail) __attribute__((always_inline)) {
        double a[W];
#pragma unroll
        for (int d = -PI; d <= PI; ++d) a[d + PI] = entry(tab[i * W + d + PI], d);
        double2 r[NR];
#pragma unroll
        for (int e = 0; e < NR; ++e) r[e] = ccast<double2>(q[e]);
        if (edge && walls) r[0].x += z6_wall_rhs(A, S.eq, op, ck, k);
        if (tail) {  // these reach PB to the left: older rows of the segment from LDS
            const double far = entry(bt[k * kBandRow - PB], -PB);
#pragma unroll
            for (int d = PB; d > PI; --d) {
                double lt = far;
                if (d == PB - 1) {
                    const double lo = far * row(i - PB, PI);  // what the row before took from this entry
                    lt = fma(coff, bt[k * kBandRow - d], -prod(lo, row(i - PB, 0)));
                }
                lt *= row(i - d, PI);
#pragma unroll
                for (int c = 1; c <= PI; ++c)
                    if (c - d + PI >= 0) {
                        if (d == PB) a[c - d + PI] = fma(coff, tab[i * W + c - d + PI], -prod(lt, row(i - d, c - 1)));
                        else a[c - d + PI] -= lt * row(i - d, c - 1);
                    }
#pragma unroll
                for (int e = 0; e < NR; ++e) {
                    r[e].x -= lt * row(i - d, PI + 1 + 2 * e);
                    r[e].y -= lt * row(i - d, PI + 2 + 2 * e);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < PI; ++t) {
            const double lt = a[t] * w.dv[t];
#pragma unroll
            for (int c = 1; c <= PI; ++c) a[t + c] -= lt * w.U[t][c - 1];
#pragma unroll
            for (int e = 0; e < NR; ++e) { r[e].x -= lt * w.y[e][t].x; r[e].y -= lt * w.y[e][t].y; }
        }
        const double dk = 1.0 / a[PI];
        double u[PI];
#pragma unroll
        for (int c = 0; c < PI; ++c) u[c] = a[PI + 1 + c];
        if (store) keep(i, u, dk, r);
#pragma unroll
        for (int t = 0; t < PI - 1; ++t) {
            w.dv[t] = w.dv[t + 1];
#pragma unroll
            for (int e = 0; e < NR; ++e) w.y[e][t] = w.y[e][t + 1];
#pragma unroll
            for (int c = 0; c < PI; ++c) w.U[t][c] = w.U[t + 1][c];
        }
        w.dv[PI - 1] = dk;
#pragma unroll
        for (int e = 0; e < NR; ++e) w.y[e][PI - 1] = r[e];
#pragma unroll
        for (int c = 0; c < PI; ++c) w.U[PI - 1][c] = u[c];
    };
    // a segment of SG rows at k0; loads the right-hand sides of the one at next
    auto segment = [&](int k0, int next, bool store, bool top) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < SG; ++u) {
            step(k0 + u, u, ring[u], store, u >= SG - 3 && top, u >= SG - 2 && top);
            load_rhs(next + u, ring[u]);
        }
    };
    auto remainder = [&](bool store, bool top) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < SG - 1; ++u)
            if (u < nrem) step(PB + u, u, ring[u], store, top && u >= nrem - 3, top && u >= nrem - 2);
    };
    // start of the remainder (slot 0) or of full segment slot - 1: PI rows of PI + 1 + 2 NR values
    auto start = [&](int slot, bool put) __attribute__((always_inline)) {
        double *p = S.scr + (size_t)slot * NS * plane + col;
        auto move = [&](int e, double &v) __attribute__((always_inline)) {
            if (put) p[(size_t)e * plane] = v;
            else v = p[(size_t)e * plane];
        };
#pragma unroll
        for (int t = 0; t < PI; ++t) {
#pragma unroll
            for (int c = 0; c < PI; ++c) move(t * NL_ + c, w.U[t][c]);
            move(t * NL_ + PI, w.dv[t]);
#pragma unroll
            for (int e = 0; e < NR; ++e) {
                move(t * NL_ + PI + 1 + 2 * e, w.y[e][t].x);
                move(t * NL_ + PI + 2 + 2 * e, w.y[e][t].y);
            }
        }
    };
    // ---- pass 1
    const int kf = PB + nrem;  // first row of the full segments
    tab_load(PB);
    fill(0);
    bottom(false);
    fill(PB);
    if (nfull > 0 && nrem > 0) {
        start(0, true);
        tab_put();
        remainder(false, false);
        tab_load(kf);
        fill(kf);
    }
    for (int g = 0; g < nfull - 1; ++g) {
        const int k0 = kf + g * SG;
        start(1 + g, true);
        tab_put();
        tab_load(k0 + SG);
        segment(k0, k0 + SG, false, false);
    }
    // ---- pass 2; the top segment's start is the window as it stands
    const int mw = jm < ny / 2 ? jm : jm - ny;
    const bool zero_out = S.trunc && !(l < A.lc && mw < A.mc && mw > -A.mc);
    const CI zero = czero_t<CI>();
    double2 xs[NR][PI];  // x at k+1 .. k+PI
#pragma unroll
    for (int e = 0; e < NR; ++e)
#pragma unroll
        for (int c = 0; c < PI; ++c) xs[e][c] = make_double2(0.0, 0.0);
    // x of row i of the segment, level k; x4 and x5 (rows 0 and 1): x at the
    // levels PI + 1 and PI + 2 above
    auto back = [&](int k, int i, const double2 (&x4)[NR], const double2 (&x5)[NR], int nwide) __attribute__((always_inline)) {
        const double dk = row(i, PI);
        double2 r[NR];
#pragma unroll
        for (int e = 0; e < NR; ++e)  // rounded to the stored type first: with FP32 spectra the last bits of u, v, w move p by 1e-4
            r[e] = ccast<double2>(ccast<CI>(make_double2(row(i, PI + 1 + 2 * e), row(i, PI + 2 + 2 * e))));
#pragma unroll
        for (int c = 0; c < PI; ++c) {
            const double u = row(i, c);
#pragma unroll
            for (int e = 0; e < NR; ++e) { r[e].x -= u * xs[e][c].x; r[e].y -= u * xs[e][c].y; }
        }
        if (nwide > 0) {
            const double u4 = wide(i, 0);
#pragma unroll
            for (int e = 0; e < NR; ++e) { r[e].x -= u4 * x4[e].x; r[e].y -= u4 * x4[e].y; }
        }
        if (nwide > 1) {
            const double u5 = wide(i, 1);
#pragma unroll
            for (int e = 0; e < NR; ++e) { r[e].x -= u5 * x5[e].x; r[e].y -= u5 * x5[e].y; }
        }
        const size_t o = (size_t)k * plane + col;
#pragma unroll
        for (int e = 0; e < NR; ++e) {
            r[e] = make_double2(r[e].x * dk, r[e].y * dk);
#pragma unroll
            for (int c = PI - 1; c > 0; --c) xs[e][c] = xs[e][c - 1];
            xs[e][0] = r[e];
            S.f[e][o] = zero_out ? zero : ccast<CI>(r[e]);
        }
    };
    const double2 none[NR] = {};
    if (face) {  // w at the top wall face
#pragma unroll
        for (int e = 0; e < NR; ++e) S.f[e][(size_t)(nz - 1) * plane + col] = zero;
    }
    for (int g = nfull - 1; g >= 0; --g) {
        const int k0 = kf + g * SG, next = g > 0 ? k0 - SG : nrem > 0 ? PB : 0;
        tab_put();
        tab_load(next);
        segment(k0, next, true, g == nfull - 1);
        if (next > 0) start(g, false);  // while this one is back-substituted
#pragma unroll
        for (int u = SG - 1; u >= 0; --u) back(k0 + u, u, none, none, 0);
    }
    if (nrem > 0) {
        tab_put();
        remainder(true, nfull == 0);
        fill(0);
        for (int u = nrem - 1; u >= 0; --u) back(PB + u, u, none, none, 0);
    }
    bottom(true);
    double2 xb[NR], xa[NR];  // x at levels PB and PB - 1
#pragma unroll
    for (int e = 0; e < NR; ++e) xb[e] = xs[e][0];
#pragma unroll
    for (int k = PB - 1; k >= 0; --k) {
        if (k == 0) back(0, 0, xa, xb, 2);
        else if (k == 1) back(1, 1, xb, none, 1);
        else back(k, k, none, none, 0);
        if (k == PB - 1) {
#pragma unroll
            for (int e = 0; e < NR; ++e) xa[e] = xs[e][0];
        }
    }
}

template <int PI, class CI>
__global__ __launch_bounds__(64) void k_z6_band(StepArgs A, BandArgs<CI> B)
{
    const BandSys<CI> S = B.s[blockIdx.y];
    if constexpr (PI == 3) {
        if (S.nr > 1) {
            band_solve<PI, 2, CI>(A, S);
            return;
        }
    }
    band_solve<PI, 1, CI>(A, S);
}

// ---------------------------------------------------------------------------
// Explicit column operations of the 6th-order step, one thread per (l, m)
// column streaming along z.  A thread keeps a window of kWin levels of the
// fields that an operator reaches (levels k-7 .. k+7 around the row k being
// formed) and applies band rows (ZB_* tables) to it.  Loads run PF levels
// ahead through a ring indexed by the unrolled loop position.  The loop holds
// no other load and no branch around one, which a wait would not tell from
// those in flight: the band rows of the block's levels are staged in LDS,
// levels out of range are loaded from the nearest one and dropped.  What bounds
// these kernels then is HBM: at 256x256x257 w's right-hand side moves 8.8 fields
// of 136 MB in 234 us (294 with the band rows read in the loop), the projection
// 9.4 in 217 (267), the divergence 4.4 in 109 (130); with FP32 spectra t's
// right-hand side 82 us (147), the divergence 62 (145).
constexpr int kWin = 2 * kBandMax + 1;

// A block forms the rows kb .. ke-1 of its columns (blockIdx.z of gridDim.z
// equal chunks), so that a launch has several wavefronts per SIMD.
constexpr int kStreamRowsPerChunk = 32;
inline int stream_chunks(int nz) { return nz / kStreamRowsPerChunk < 1 ? 1 : (nz / kStreamRowsPerChunk > 8 ? 8 : nz / kStreamRowsPerChunk); }
struct ZChunk {
    int kb, ke, csz;
};
HC_DEV ZChunk z_chunk(int nrows)
{
    const int csz = (nrows + (int)gridDim.z - 1) / (int)gridDim.z, kb = (int)blockIdx.z * csz;
    return {kb, min(kb + csz, nrows), csz};
}
// bytes of LDS that nb bands of a chunk take
inline size_t stream_lds(int nz, int nb)
{
    const int nc = stream_chunks(nz);
    return (size_t)nb * ((nz + nc - 1) / nc) * kBandRow * sizeof(double);
}
// rows kb .. ke-1 of band b of this launch's NB bands at sm + b csz kBandRow;
// every thread of the block calls this (it ends in a barrier)
template <int NB>
HC_DEV void stage_bands(const double *zband, int nz, const ZChunk &z, const int (&band)[NB], double *sm)
{
    const int n = (z.ke - z.kb) * kBandRow;
#pragma unroll
    for (int b = 0; b < NB; ++b)
        for (int q = threadIdx.x; q < n; q += 256)
            sm[b * z.csz * kBandRow + q] = zband[((size_t)band[b] * nz + z.kb) * kBandRow + q];
    __syncthreads();
}
HC_DEV const double *band_row(const double *sm, const ZChunk &z, int b, int k)
{
    return sm + (b * z.csz + k - z.kb) * kBandRow;
}

// Row k is formed by row(k, win, pts) with win[kBandMax + t] = level k + t
// (zero outside 0 .. wlev[f] - 1; a chunk reads kBandMax levels beyond each
// end) and pts the point fields at k.  Fields are stored as CI (double2 or
// float2) and held in FP64.  A kernel writes only its point fields' rows or
// fields it does not read.
template <int N, class CI = double2>
struct FieldSet {
    const CI *p[N > 0 ? N : 1];
    int n[N > 0 ? N : 1];  // levels of a window field
};
template <int NW, int NP, int PF, class CW, class CP, class Row>
HC_DEV void z6_stream(size_t plane, size_t col, const ZChunk &z, const FieldSet<NW, CW> ws, const FieldSet<NP, CP> ps,
                      Row &&row)
{
    const double2 zero = make_double2(0.0, 0.0);
    const int kb = z.kb, ke = z.ke;
    if (kb >= ke) return;
    auto load_w = [&](int f, int li) __attribute__((always_inline)) {
        return ws.p[f][(size_t)min(max(li, 0), ws.n[f] - 1) * plane + col];
    };
    auto load_p = [&](int p, int k) __attribute__((always_inline)) { return ps.p[p][(size_t)min(k, ke - 1) * plane + col]; };
    auto level = [&](int f, int li, const CW &v) __attribute__((always_inline)) {
        return li >= 0 && li < ws.n[f] ? ccast<double2>(v) : zero;
    };
    // the ring holds the stored type: widening to FP64 happens when a level
    // leaves the ring, so no conversion waits on a load in flight
    double2 win[NW][kWin];
    CW fw[NW][PF], first[NW][kWin - 1];
    CP fp[PF][NP > 0 ? NP : 1];
#pragma unroll
    for (int f = 0; f < NW; ++f)
#pragma unroll
        for (int t = 0; t < kWin - 1; ++t) first[f][t] = load_w(f, kb - kBandMax + t);
#pragma unroll
    for (int u = 0; u < PF; ++u) {
#pragma unroll
        for (int f = 0; f < NW; ++f) fw[f][u] = load_w(f, kb + u + kBandMax);
#pragma unroll
        for (int p = 0; p < NP; ++p) fp[u][p] = load_p(p, kb + u);
    }
#pragma unroll
    for (int f = 0; f < NW; ++f)
#pragma unroll
        for (int t = 0; t < kWin - 1; ++t) win[f][t + 1] = level(f, kb - kBandMax + t, first[f][t]);
    for (int k0 = kb; k0 < ke; k0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int k = k0 + u;
            if (k >= ke) return;
            double2 pts[NP > 0 ? NP : 1];
#pragma unroll
            for (int f = 0; f < NW; ++f) {
#pragma unroll
                for (int t = 0; t < kWin - 1; ++t) win[f][t] = win[f][t + 1];
                win[f][kWin - 1] = level(f, k + kBandMax, fw[f][u]);
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) pts[p] = ccast<double2>(fp[u][p]);
#pragma unroll
            for (int f = 0; f < NW; ++f) fw[f][u] = load_w(f, k + PF + kBandMax);
#pragma unroll
            for (int p = 0; p < NP; ++p) fp[u][p] = load_p(p, k + PF);
            row(k, win, pts);
        }
    }
}

// sum_t band(k, t) x(k + t) over the stored band
HC_DEV double2 band_dot(const double *brow, const double2 (&x)[kWin])
{
    double2 acc = make_double2(0.0, 0.0);
#pragma unroll
    for (int t = 0; t < kWin; ++t) {
        const double b = brow[t];
        acc.x += b * x[t].x;
        acc.y += b * x[t].y;
    }
    return acc;
}

struct ColIdx {
    int l, jm;
    size_t col, plane;
};
HC_DEV bool col_idx(const StepArgs &A, ColIdx &c)
{
    const int ncol = A.nl * A.ny;
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= ncol) return false;
    c.l = q % A.nl;
    c.jm = q / A.nl;
    c.col = (size_t)q;
    c.plane = (size_t)ncol;
    return true;
}

// Divergence D_x u + D_y v + D_z w of a column times `scale` into the FP64
// spectrum dst (get_p_eqn_src / get_div_spec with ZO_D over the interior
// faces).
template <class CI>
__global__ __launch_bounds__(256, 2) void k_z6s_div(StepArgs A, const CI *u, const CI *v, const CI *w, double2 *dst,
                                                 double scale)
{
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(A.nz);
    stage_bands(A.zband, A.nz, z, {ZB_D}, band_sm);
    ColIdx c;
    if (!col_idx(A, c)) return;
    const int nl = A.nl, ny = A.ny, nz = A.nz;
    const double2 sdx = make_double2(A.symx[SY_DRE * nl + c.l], A.symx[SY_DIM * nl + c.l]);
    const double2 sdy = make_double2(A.symy[SY_DRE * ny + c.jm], A.symy[SY_DIM * ny + c.jm]);
    const FieldSet<1, CI> ws = {{w}, {nz - 1}};
    const FieldSet<2, CI> ps = {{u, v}, {0, 0}};
    z6_stream<1, 2, 8>(c.plane, c.col, z, ws, ps, [&](int k, const double2 (&win)[1][kWin], const double2 (&p)[2]) __attribute__((always_inline)) {
        const double2 dz = band_dot(band_row(band_sm, z, 0, k), win[0]);
        const double2 d = cadd(cadd(cmul(sdx, p[0]), cmul(sdy, p[1])), dz);
        dst[(size_t)k * c.plane + c.col] = make_double2(d.x * scale, d.y * scale);
    });
}

// Projection u, v, w -= cdt grad phi (calculate_uvw, ZO_G at the interior
// faces), phi an FP64 spectrum.  mode 0 (FD substep, cdt = rc dt): the
// pressure increment phi - rc dt nu / 2 (hxy_L + ZO_P) phi (calculate_new_p)
// goes to `pinc`; mode 1 (projection of a state, cdt = 1); mode 2 (spectral
// substep, cdt = rc dt): the increment is added to c_p in `pinc` and the
// columns outside the 2/3 rule are zeroed.
template <class CI>
__global__ __launch_bounds__(256, 2) void k_z6s_proj(StepArgs A, CI *u, CI *v, CI *w, const double2 *phi, CI *pinc,
                                                  int mode)
{
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(A.nz);
    stage_bands(A.zband, A.nz, z, {ZB_G, ZB_P}, band_sm);
    ColIdx c;
    if (!col_idx(A, c)) return;
    const int nl = A.nl, ny = A.ny, nz = A.nz;
    const double2 sgx = make_double2(A.symx[SY_GRE * nl + c.l], A.symx[SY_GIM * nl + c.l]);
    const double2 sgy = make_double2(A.symy[SY_GRE * ny + c.jm], A.symy[SY_GIM * ny + c.jm]);
    const double slap = A.symx[SY_L * nl + c.l] + A.symy[SY_L * ny + c.jm];
    const double cdt = mode == 1 ? 1.0 : A.rc * A.dt, cnu = A.rc * 0.5 * A.dt * A.nu;
    const int mw = c.jm < ny / 2 ? c.jm : c.jm - ny;
    const bool kept = mode != 2 || (c.l < A.lc && mw < A.mc && mw > -A.mc);
    const CI zero = czero_t<CI>();
    const FieldSet<1> ws = {{phi}, {nz}};
    // the fourth point field is read only in mode 2 (c_p); u stands in otherwise
    const FieldSet<4, CI> ps = {{u, v, w, mode == 2 ? pinc : u}, {0, 0, 0, 0}};
    z6_stream<1, 4, 4>(c.plane, c.col, z, ws, ps, [&](int k, const double2 (&win)[1][kWin], const double2 (&p)[4]) __attribute__((always_inline)) {
        const size_t o = (size_t)k * c.plane + c.col;
        const double2 ph = win[0][kBandMax];
        double2 uu = csub(p[0], cscale(cmul(sgx, ph), cdt));
        double2 vv = csub(p[1], cscale(cmul(sgy, ph), cdt));
        double2 ww = p[2];
        if (k < nz - 1) {
            const double2 g = band_dot(band_row(band_sm, z, 0, k), win[0]);
            ww = make_double2(ww.x - cdt * g.x, ww.y - cdt * g.y);
        }
        u[o] = kept ? ccast<CI>(uu) : zero;
        v[o] = kept ? ccast<CI>(vv) : zero;
        w[o] = kept ? ccast<CI>(ww) : zero;
        if (mode == 1) return;
        const double2 pz = band_dot(band_row(band_sm, z, 1, k), win[0]);
        const double2 inc = make_double2(ph.x - cnu * (slap * ph.x + pz.x), ph.y - cnu * (slap * ph.y + pz.y));
        if (mode == 0) pinc[o] = ccast<CI>(inc);
        else pinc[o] = kept ? ccast<CI>(cadd(p[3], inc)) : zero;
    });
}

// Right-hand sides of the spectral substep's Helmholtz systems
// (get_momentum_cnvdiff_spec, src/module_spectral.f90:35-504, with the
// 6th-order z operators) for u, v (blockIdx.y = 0, 1; into sp[3], sp[4]) or
// w (k_z6s_rhs_w; into sp[7]):
//   q = c + hxy c + dif Z c - cdt grad_e p + rb dt f_old + ra dt f
//   f = -u_mrf i kx c - coe (i kx X + i ky Y) + coe R
// with X, Y, R the transformed products of the component; f replaces f_old.
// The (0,0) mode adds the explicit half of the wall data of u.
template <class CI>
__global__ __launch_bounds__(256, 2) void k_z6s_rhs_uv(StepArgs A, SpecIO<real_of<CI>> io)
{
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(A.nz);
    stage_bands(A.zband, A.nz, z, {A.ochannel ? ZB_C2_DN : ZB_C2_DD}, band_sm);
    ColIdx c;
    if (!col_idx(A, c)) return;
    const int e = blockIdx.y;
    const int nl = A.nl, ny = A.ny, nz = A.nz;
    const double kx = A.symx[SY_GIM * nl + c.l], ky = A.symy[SY_GIM * ny + c.jm];
    const double hxy = A.rc * (A.symx[SY_HU * nl + c.l] + A.symy[SY_HU * ny + c.jm]);
    const double dif = A.rc * 0.5 * A.dt * A.nu, coe = A.coe, um = A.u_mrf, cdt = A.rc * A.dt;
    const double rb = A.rb * A.dt, ra = A.ra * A.dt, kk = e == 0 ? kx : ky;
    const bool is00 = e == 0 && c.l == 0 && c.jm == 0;
    const int op = A.ochannel ? ZO_C2_DN : ZO_C2_DD;
    // q goes over R_u / R_v (read at the same row by the same thread): c_u,
    // c_v stay intact for the neighbouring z chunks' windows
    CI *cs = e == 0 ? io.cu : io.cv, *fo = e == 0 ? io.cff : io.cgg, *qo = e == 0 ? io.sp[3] : io.sp[4];
    const FieldSet<1, CI> ws = {{cs}, {nz}};
    const FieldSet<5, CI> ps = {{io.sp[e == 0 ? 0 : 1], io.sp[e == 0 ? 1 : 2], io.sp[e == 0 ? 3 : 4], io.cp, fo},
                                {0, 0, 0, 0, 0}};
    z6_stream<1, 5, 3>(c.plane, c.col, z, ws, ps, [&](int k, const double2 (&win)[1][kWin], const double2 (&p)[5]) __attribute__((always_inline)) {
        const double2 x = win[0][kBandMax];
        const double2 t = band_dot(band_row(band_sm, z, 0, k), win[0]);
        double2 q = make_double2(x.x + hxy * x.x + dif * t.x, x.y + hxy * x.y + dif * t.y);
        if (is00) q.x += z6_wall_rhs(A, 0, op, dif, k);
        double2 f = times_i(x, -um * kx);
        f = csub(f, times_i(p[0], coe * kx));
        f = csub(f, times_i(p[1], coe * ky));
        f = make_double2(f.x + coe * p[2].x, f.y + coe * p[2].y);
        q = csub(q, times_i(p[3], cdt * kk));
        q = make_double2(q.x + rb * p[4].x + ra * f.x, q.y + rb * p[4].y + ra * f.y);
        const size_t o = (size_t)k * c.plane + c.col;
        fo[o] = ccast<CI>(f);
        qo[o] = ccast<CI>(q);
    });
}
template <class CI>
__global__ __launch_bounds__(256, 2) void k_z6s_rhs_w(StepArgs A, SpecIO<real_of<CI>> io)
{
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(A.nz);
    stage_bands(A.zband, A.nz, z, {ZB_F2, ZB_G}, band_sm);
    ColIdx c;
    if (!col_idx(A, c)) return;
    const int nl = A.nl, ny = A.ny, nz = A.nz;
    const double kx = A.symx[SY_GIM * nl + c.l], ky = A.symy[SY_GIM * ny + c.jm];
    const double hxy = A.rc * (A.symx[SY_HU * nl + c.l] + A.symy[SY_HU * ny + c.jm]);
    const double dif = A.rc * 0.5 * A.dt * A.nu, coe = A.coe, um = A.u_mrf, cdt = A.rc * A.dt;
    const double rb = A.rb * A.dt, ra = A.ra * A.dt;
    const FieldSet<2, CI> ws = {{io.cw, io.cp}, {nz - 1, nz}};
    const FieldSet<4, CI> ps = {{io.sp[5], io.sp[6], io.sp[7], io.chh}, {0, 0, 0, 0}};
    z6_stream<2, 4, 2>(c.plane, c.col, z, ws, ps, [&](int k, const double2 (&win)[2][kWin], const double2 (&p)[4]) __attribute__((always_inline)) {
        const size_t o = (size_t)k * c.plane + c.col;
        const double2 x = win[0][kBandMax];
        double2 f = times_i(x, -um * kx);
        f = csub(f, times_i(p[0], coe * kx));
        f = csub(f, times_i(p[1], coe * ky));
        f = make_double2(f.x + coe * p[2].x, f.y + coe * p[2].y);
        io.chh[o] = ccast<CI>(f);
        if (k == nz - 1) return;  // the top wall face: no equation
        const double2 t = band_dot(band_row(band_sm, z, 0, k), win[0]);
        const double2 g = band_dot(band_row(band_sm, z, 1, k), win[1]);
        double2 q = make_double2(x.x + hxy * x.x + dif * t.x - cdt * g.x, x.y + hxy * x.y + dif * t.y - cdt * g.y);
        q = make_double2(q.x + rb * p[3].x + ra * f.x, q.y + rb * p[3].y + ra * f.y);
        io.sp[7][o] = ccast<CI>(q);  // over R_w, as for u and v
    });
}

// Right-hand side of the spectral temperature system
// (get_temperature_cnvdiff_spec with the 6th-order z operator) into sp[2];
// the new s replaces the old one in c_ss; the (0,0) mode adds the explicit
// half of the wall data.
template <class CI>
__global__ __launch_bounds__(256, 2) void k_z6s_rhs_t(StepArgs A, SpecIO<real_of<CI>> io)
{
    extern __shared__ double band_sm[];
    const ZChunk z = z_chunk(A.nz);
    stage_bands(A.zband, A.nz, z, {A.tbc_top ? ZB_C2_DN : ZB_C2_DD}, band_sm);
    ColIdx c;
    if (!col_idx(A, c)) return;
    const int nl = A.nl, ny = A.ny, nz = A.nz;
    const double kx = A.symx[SY_GIM * nl + c.l], ky = A.symy[SY_GIM * ny + c.jm];
    const double hxy = A.rc * (A.symx[SY_HT * nl + c.l] + A.symy[SY_HT * ny + c.jm]);
    const double dif = A.rc * 0.5 * A.dt * A.alpha, um = A.u_mrf;
    const double rb = A.rb * A.dt, ra = A.ra * A.dt;
    const bool is00 = c.l == 0 && c.jm == 0;
    const int op = A.tbc_top ? ZO_C2_DN : ZO_C2_DD;
    const FieldSet<1, CI> ws = {{io.ct}, {nz}};
    const FieldSet<4, CI> ps = {{io.sp[0], io.sp[1], io.sp[2], io.css}, {0, 0, 0, 0}};
    z6_stream<1, 4, 4>(c.plane, c.col, z, ws, ps, [&](int k, const double2 (&win)[1][kWin], const double2 (&p)[4]) __attribute__((always_inline)) {
        const double2 x = win[0][kBandMax];
        const double2 t = band_dot(band_row(band_sm, z, 0, k), win[0]);
        double2 d = make_double2(x.x + hxy * x.x + dif * t.x, x.y + hxy * x.y + dif * t.y);
        if (is00) d.x += z6_wall_rhs(A, 3, op, dif, k);
        double2 f = times_i(x, -um * kx);
        f = csub(f, times_i(p[0], kx));
        f = csub(f, times_i(p[1], ky));
        f = cadd(f, p[2]);
        d = make_double2(d.x + rb * p[3].x + ra * f.x, d.y + rb * p[3].y + ra * f.y);
        const size_t o = (size_t)k * c.plane + c.col;
        io.css[o] = ccast<CI>(f);
        io.sp[2][o] = ccast<CI>(d);  // over the z flux term
    });
}
