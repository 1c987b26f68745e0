// Column kernels of the 2nd-order z operators: the fused momentum column
// pass, the temperature solve, the projection of initial states and the
// standalone poisson_solver_fft, FP64 or with FP32 storage.
#include "hc_host.h"

// Columns per block of k_column_mom: four, so that two blocks share a CU (a
// block's loads and stores then overlap the other's solves); the two halves
// of a 128-byte line belong to neighbouring blocks of one XCD.  Two beyond
// 512 levels, whose tiles would not fit, and from 342 levels on where the
// runtime has refused more than 64 KB of dynamic LDS.
template <int L> constexpr int mom_waves() { return L > 8 ? 2 : 4; }
constexpr size_t kLdsDefault = 64 * 1024;  // dynamic LDS of any kernel

// One fused column pass of the substep: Helmholtz solves of u*, v*, w*, the
// divergence source, the pressure Poisson solve, the projection and the
// pressure increment (FP64).  A column lives in its block's LDS tiles (u, v,
// w; the increment in a fourth if A.ntile says so, else in u's after that is
// stored) and only the fields being solved for are in registers, which keeps
// up to 8 levels per lane below the 256 VGPRs of two waves per SIMD (156 VGPRs
// at 5 levels: three blocks of four waves).  Bound by HBM and, less, VALU
// issue (2060 instructions per column at 5 levels): 335 us per substep at
// 256x256x257 FP64 (0.94 GB, 2.8 TB/s; with every field in registers, 247
// VGPRs and one block of eight columns per CU, 473 us),
// 47 us at 128x128x129 (91), 3.0 ms at 512x512x385 (6.2, spilling).
template <int L, int W = mom_waves<L>()>
__global__ __launch_bounds__(64 * W, 2) void k_column_mom(StepArgs A, ColIO<double> io)
{
    using RC = double;
    using CC = double2;
    constexpr int T = 64 * W;
    extern __shared__ double2 tile_raw[];
    CC *tile = tile_raw;
    const ColPos pos = col_pos<W>(io, A.ny);
    if (pos.skip) return;  // block-uniform, before any barrier
    // nl is a multiple of kColWaves: every wavefront owns a column
    const int w = threadIdx.x >> 6, l = pos.bx * W + w, jm = pos.jm;
    const ColMap m = col_map<L>(A.nz);
    const int nz = A.nz, nl = A.nl, ny = A.ny;
    const bool is00 = (l == 0 && jm == 0);
    const size_t plane = (size_t)ny * nl, col0 = (size_t)jm * nl + (size_t)pos.bx * W;
    const int sub = (int)col_sub<W>(nz);
    CC *const tu = tile, *const tv = tile + sub, *const tw = tile + 2 * sub;
    {   // all three inputs, every load before the first LDS store
        CC v[3][L];
#pragma unroll
        for (int it = 0; it < L; ++it) {
            const int q = threadIdx.x + it * T, k = q / W, c = q - k * W;
            const size_t o = (size_t)k * plane + col0 + c;
            v[0][it] = v[1][it] = v[2][it] = czero();
            if (q < nz * W) { v[0][it] = io.s0[o]; v[1][it] = io.s1[o]; v[2][it] = io.s2[o]; }
        }
#pragma unroll
        for (int it = 0; it < L; ++it) {
            const int q = threadIdx.x + it * T, k = q / W, c = q - k * W;
            if (q < nz * W) {
                const int at = col_tidx<L, true, W>(k, c);
                tu[at] = v[0][it]; tv[at] = v[1][it]; tw[at] = v[2][it];
            }
        }
    }
    __syncthreads();
    // this column's entries of a tile: read and written by this wave alone
    int at[L];
#pragma unroll
    for (int r = 0; r < L; ++r) at[r] = col_tidx<L, true, W>(min(m.k0 + r, nz - 1), w);
    RC a[L], b[L], c[L];
    {   // u and v share the matrix (assign_abc(aa_u,...) for both, :291-299)
        CC d[2][L];
#pragma unroll
        for (int r = 0; r < L; ++r) {
            d[0][r] = r < m.cnt ? tu[at[r]] : czero();
            d[1][r] = r < m.cnt ? tv[at[r]] : czero();
        }
        assemble<L>(A, 0, l, jm, is00, m, a, b, c);
        if (is00) fixups<L>(A, 0, m, d[0]);
        wave_tridiag<L, 2>(a, b, c, d);
#pragma unroll
        for (int r = 0; r < L; ++r)
            if (r < m.cnt) { tu[at[r]] = d[0][r]; tv[at[r]] = d[1][r]; }
    }
    const CC sdx = mk2<CC>(RC(A.symx[SY_DRE * nl + l]), RC(A.symx[SY_DIM * nl + l]));
    const CC sdy = mk2<CC>(RC(A.symy[SY_DRE * ny + jm]), RC(A.symy[SY_DIM * ny + jm]));
    CC dp[1][L];
    {   // w (:302-304): kend3 row is trivial and its right-hand side is unused
        CC d[1][L];
#pragma unroll
        for (int r = 0; r < L; ++r) d[0][r] = m.k0 + r < nz - 1 ? tw[at[r]] : czero();
        assemble<L>(A, 1, l, jm, is00, m, a, b, c);
        wave_tridiag<L, 1>(a, b, c, d);
        // divergence source /dt (get_p_eqn_src, :127-176) in spectral form
        CC wm = col_before<L>(m, d[0]);
        if (m.lane == 0) wm = czero();
#pragma unroll
        for (int r = 0; r < L; ++r) {
            dp[0][r] = czero();
            if (r < m.cnt) {
                tw[at[r]] = d[0][r];
                const RC idz = RC(col_lev<L>(A, m, LV_IDZ, r));
                CC dv = cadd(cmul(sdx, tu[at[r]]), cmul(sdy, tv[at[r]]));
                dv.x += (d[0][r].x - wm.x) * idz;
                dv.y += (d[0][r].y - wm.y) * idz;
                dp[0][r] = cscale(dv, RC(A.idt));
            }
            wm = d[0][r];
        }
    }
    // pressure Poisson (:312-314)
    assemble<L>(A, 2, l, jm, is00, m, a, b, c);
    if (is00) fixups<L>(A, 2, m, dp[0]);
    wave_tridiag_refined<L, 1>(a, b, c, dp);
    // projection (calculate_uvw, :659-734) and pressure increment
    // (calculate_new_p, :739-808)
    const RC cdt = RC(A.rc * A.dt), cnu = RC(A.rc * 0.5 * A.dt * A.nu);
    const RC slap = RC(A.symx[SY_L * nl + l] + A.symy[SY_L * ny + jm]);
    const CC sgx = mk2<CC>(RC(A.symx[SY_GRE * nl + l]), RC(A.symx[SY_GIM * nl + l]));
    const CC sgy = mk2<CC>(RC(A.symy[SY_GRE * ny + jm]), RC(A.symy[SY_GIM * ny + jm]));
    CC pm = col_before<L>(m, dp[0]);
    const CC pnext = col_after<L>(m, dp[0]);
    if (m.lane == 0) pm = dp[0][0];
    const bool four = A.ntile >= 4;
    CC inc[L];
#pragma unroll
    for (int r = 0; r < L; ++r) {
        const CC ph = dp[0][r];
        inc[r] = czero();
        if (r < m.cnt) {
            const int k = m.k0 + r;
            const CC pn = col_next<L>(m, nz, dp[0], r, pnext);
            const RC idzt = RC(col_lev<L>(A, m, LV_IDZT, r)), idzb = RC(col_lev<L>(A, m, LV_IDZB, r));
            const RC idz = RC(col_lev<L>(A, m, LV_IDZ, r));
            const CC lz = mk2<CC>(((pn.x - ph.x) * idzt - (ph.x - pm.x) * idzb) * idz,
                                  ((pn.y - ph.y) * idzt - (ph.y - pm.y) * idzb) * idz);
            inc[r] = mk2<CC>(ph.x - cnu * (slap * ph.x + lz.x), ph.y - cnu * (slap * ph.y + lz.y));
            if (four) tile[3 * sub + at[r]] = inc[r];
            tu[at[r]] = csub(tu[at[r]], cscale(cmul(sgx, ph), cdt));
            tv[at[r]] = csub(tv[at[r]], cscale(cmul(sgy, ph), cdt));
            if (k < nz - 1) {
                const RC f = cdt * idzt;
                const CC ww = tw[at[r]];
                tw[at[r]] = mk2<CC>(ww.x - f * (pn.x - ph.x), ww.y - f * (pn.y - ph.y));
            }
        }
        pm = ph;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < nz * W; q += T) {
        const int k = q / W, cl = q - k * W, e = col_tidx<L, true, W>(k, cl);
        const size_t o = (size_t)k * plane + col0 + cl;
        io.s0[o] = tu[e];
        io.s1[o] = tv[e];
        io.s2[o] = tw[e];
        if (four) io.s3[o] = tile[3 * sub + e];
    }
    if (four) return;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < L; ++r)
        if (r < m.cnt) tu[at[r]] = inc[r];
    __syncthreads();
    for (int q = threadIdx.x; q < nz * W; q += T) {
        const int k = q / W, cl = q - k * W;
        io.s3[(size_t)k * plane + col0 + cl] = tu[col_tidx<L, true, W>(k, cl)];
    }
}

// The same pass over FP32 spectra (mixed variant), in FP64 for the
// low-wavenumber blocks and FP32 for the rest: every field in registers, eight
// columns per block, the operations of lane_tridiag.
template <int L, class RC>
__global__ __launch_bounds__(64 * kColWaves) void k_column_mom_mixed(StepArgs A, ColIO<float> io)
{
    using CI = float2;
    using CC = cplx<RC>;
    extern __shared__ double2 tile_raw[];
    CI *tile = reinterpret_cast<CI *>(tile_raw);
    const ColPos pos = col_pos(io, A.ny);
    if (pos.skip) return;  // block-uniform, before any barrier
    // nl is a multiple of kColWaves: every wavefront owns a column
    const int l = pos.bx * kColWaves + (threadIdx.x >> 6), jm = pos.jm;
    const auto m = col_map<L, false>(A.nz);
    const int nz = A.nz, nl = A.nl, ny = A.ny;
    const bool is00 = (l == 0 && jm == 0);
    const size_t plane = (size_t)ny * nl, col0 = (size_t)jm * nl + (size_t)pos.bx * kColWaves;
    CC duv[2][L], dw[1][L], dp[1][L];
    // all three inputs in one phase when the tile holds them (A.ntile sub-tiles)
    const size_t sub = (size_t)nz * kColWaves;
    if (A.ntile >= 3) {
        const CI *srcs[3] = {io.s0, io.s1, io.s2};
        col_fill_n<L, 3, false>(srcs, tile, nz, plane, col0);
        __syncthreads();
        col_take<L>(tile, m, duv[0]);
        col_take<L>(tile + sub, m, duv[1]);
        col_take<L>(tile + 2 * sub, m, dw[0]);
        __syncthreads();
    } else {
        col_load<L>(io.s0, tile, nz, plane, col0, m, duv[0]);
        col_load<L>(io.s1, tile, nz, plane, col0, m, duv[1]);
        col_load<L>(io.s2, tile, nz, plane, col0, m, dw[0]);
    }
    RC a[L], b[L], c[L];
    // u and v share the matrix (assign_abc(aa_u,...) for both, :291-299)
    assemble<L>(A, 0, l, jm, is00, m, a, b, c);
    if (is00) fixups<L>(A, 0, m, duv[0]);
    lane_tridiag<L, 2>(m.cnt, a, b, c, duv);
    // w (:302-304): kend3 row is trivial and its right-hand side is unused
#pragma unroll
    for (int r = 0; r < L; ++r)
        if (r < m.cnt && m.k0 + r == nz - 1) dw[0][r] = czero_t<CC>();
    assemble<L>(A, 1, l, jm, is00, m, a, b, c);
    lane_tridiag<L, 1>(m.cnt, a, b, c, dw);
    // divergence source /dt (get_p_eqn_src, :127-176) in spectral form
    col_divergence<L>(A, m, l, jm, duv[0], duv[1], dw[0], RC(A.idt), dp[0]);
    // pressure Poisson (:312-314)
    assemble<L>(A, 2, l, jm, is00, m, a, b, c);
    if (is00) fixups<L>(A, 2, m, dp[0]);
    lane_tridiag_refined<L, 1>(m.cnt, a, b, c, dp);
    // projection (calculate_uvw, :659-734) and pressure increment
    // (calculate_new_p, :739-808)
    const RC cdt = RC(A.rc * A.dt);
    col_project<L>(A, m, l, jm, cdt, dp[0], duv[0], duv[1], dw[0]);
    const RC slap = RC(A.symx[SY_L * nl + l] + A.symy[SY_L * ny + jm]);
    CC pprev = shfl_up_c(last_of<L>(dp[0], m.cnt), 1);
    CC pnext = shfl_dn_c(dp[0][0], 1);
    const RC cnu = RC(A.rc * 0.5 * A.dt * A.nu);
    CC dpn[L];
#pragma unroll
    for (int r = 0; r < L; ++r) {
        dpn[r] = czero_t<CC>();
        if (r < m.cnt) {
            int k = m.k0 + r;
            CC ph = dp[0][r];
            CC pm = r == 0 ? (m.lane == 0 ? ph : pprev) : dp[0][r > 0 ? r - 1 : 0];
            CC pn = col_next<L>(m, nz, dp[0], r, pnext);
            RC idzt = RC(A.lev[LV_IDZT * nz + k]), idzb = RC(A.lev[LV_IDZB * nz + k]), idz = RC(A.lev[LV_IDZ * nz + k]);
            CC lz;
            lz.x = ((pn.x - ph.x) * idzt - (ph.x - pm.x) * idzb) * idz;
            lz.y = ((pn.y - ph.y) * idzt - (ph.y - pm.y) * idzb) * idz;
            CC lap = mk2<CC>(slap * ph.x + lz.x, slap * ph.y + lz.y);
            dpn[r] = mk2<CC>(ph.x - cnu * lap.x, ph.y - cnu * lap.y);
        }
    }
    if (A.ntile >= 4) {
        col_put<L>(tile, m, duv[0]);
        col_put<L>(tile + sub, m, duv[1]);
        col_put<L>(tile + 2 * sub, m, dw[0]);
        col_put<L>(tile + 3 * sub, m, dpn);
        __syncthreads();
        col_drain<L, false>(io.s0, tile, nz, plane, col0);
        col_drain<L, false>(io.s1, tile + sub, nz, plane, col0);
        col_drain<L, false>(io.s2, tile + 2 * sub, nz, plane, col0);
        col_drain<L, false>(io.s3, tile + 3 * sub, nz, plane, col0);
    } else {
        col_store<L>(io.s0, tile, nz, plane, col0, m, duv[0]);
        col_store<L>(io.s1, tile, nz, plane, col0, m, duv[1]);
        col_store<L>(io.s2, tile, nz, plane, col0, m, dw[0]);
        col_store<L>(io.s3, tile, nz, plane, col0, m, dpn);
    }
}

// Temperature Helmholtz solve in place on s0 (:335-337).
template <int L, class RIO, class RC>
__global__ __launch_bounds__(64 * kColWaves) void k_column_t(StepArgs A, ColIO<RIO> io)
{
    using CI = cplx<RIO>;
    extern __shared__ double2 tile_raw[];
    CI *tile = reinterpret_cast<CI *>(tile_raw);
    const ColPos pos = col_pos(io, A.ny);
    if (pos.skip) return;
    const int l = pos.bx * kColWaves + (threadIdx.x >> 6), jm = pos.jm;
    const auto m = col_map<L, sizeof(RIO) == 8>(A.nz);
    const bool is00 = (l == 0 && jm == 0);
    const size_t plane = (size_t)A.ny * A.nl, col0 = (size_t)jm * A.nl + (size_t)pos.bx * kColWaves;
    cplx<RC> d[1][L];
    col_load<L>(io.s0, tile, A.nz, plane, col0, m, d[0]);
    RC a[L], b[L], c[L];
    assemble<L>(A, 3, l, jm, is00, m, a, b, c);
    if (is00) fixups<L>(A, 3, m, d[0]);
    if constexpr (decltype(m)::parts) wave_tridiag<L, 1>(a, b, c, d);
    else lane_tridiag<L, 1>(m.cnt, a, b, c, d);
    col_store<L>(io.s0, tile, A.nz, plane, col0, m, d[0]);
}

// How the two kernels below spread a column of FP64 spectra.  Beyond 896 levels
// both keep a, b, c and two vectors of 16 levels per lane in scratch, and lanes
// that share the levels evenly touch less of it than parts of 16 (900 levels,
// 128x128: pressure solve 469 against 500 us, projection 4.51 against 4.60 ms).
template <int L, class RIO>
constexpr bool solve_by_parts() { return sizeof(RIO) == 8 && L < 16; }

// Projection of (u, v, w) spectra in s0, s1, s2 onto discretely
// divergence-free fields with the pressure operator at rk_c = 1:
// phi = L^{-1} div u, u -= G phi (the operators of get_p_eqn_src,
// poisson_solver_fft and calculate_uvw).  Used to prepare initial states.
template <int L, class RIO, class RC>
__global__ __launch_bounds__(64 * kColWaves) void k_column_project(StepArgs A, ColIO<RIO> io)
{
    using CI = cplx<RIO>;
    using CC = cplx<RC>;
    extern __shared__ double2 tile_raw[];
    CI *tile = reinterpret_cast<CI *>(tile_raw);
    const ColPos pos = col_pos(io, A.ny);
    if (pos.skip) return;
    const int l = pos.bx * kColWaves + (threadIdx.x >> 6), jm = pos.jm;
    const auto m = col_map<L, solve_by_parts<L, RIO>()>(A.nz);
    const bool is00 = (l == 0 && jm == 0);
    const size_t plane = (size_t)A.ny * A.nl, col0 = (size_t)jm * A.nl + (size_t)pos.bx * kColWaves;
    CC u[1][L], v[1][L], w[1][L], ph[1][L];
    col_load<L>(io.s0, tile, A.nz, plane, col0, m, u[0]);
    col_load<L>(io.s1, tile, A.nz, plane, col0, m, v[0]);
    col_load<L>(io.s2, tile, A.nz, plane, col0, m, w[0]);
#pragma unroll
    for (int r = 0; r < L; ++r)
        if (r < m.cnt && m.k0 + r == A.nz - 1) w[0][r] = czero_t<CC>();
    col_divergence<L>(A, m, l, jm, u[0], v[0], w[0], RC(1), ph[0]);
    RC a[L], b[L], c[L];
    assemble<L>(A, 2, l, jm, is00, m, a, b, c);
    if (is00) fixups<L>(A, 2, m, ph[0]);
    if constexpr (decltype(m)::parts) wave_tridiag_refined<L, 1>(a, b, c, ph);
    else lane_tridiag_refined<L, 1>(m.cnt, a, b, c, ph);
    col_project<L>(A, m, l, jm, RC(1), ph[0], u[0], v[0], w[0]);
    col_store<L>(io.s0, tile, A.nz, plane, col0, m, u[0]);
    col_store<L>(io.s1, tile, A.nz, plane, col0, m, v[0]);
    col_store<L>(io.s2, tile, A.nz, plane, col0, m, w[0]);
}

// Standalone poisson_solver_fft for one equation, in place on s0.
// eq: 0 u (ubnd), 1 v, 2 w (zstagger), 3 p (delnull), 4 t (tbnd).
template <int L, class RIO, class RC>
__global__ __launch_bounds__(64 * kColWaves) void k_column_solve(StepArgs A, ColIO<RIO> io, int eq)
{
    using CI = cplx<RIO>;
    extern __shared__ double2 tile_raw[];
    CI *tile = reinterpret_cast<CI *>(tile_raw);
    const ColPos pos = col_pos(io, A.ny);
    if (pos.skip) return;
    const int l = pos.bx * kColWaves + (threadIdx.x >> 6), jm = pos.jm;
    const auto m = col_map<L, solve_by_parts<L, RIO>()>(A.nz);
    const bool is00 = (l == 0 && jm == 0);
    const size_t plane = (size_t)A.ny * A.nl, col0 = (size_t)jm * A.nl + (size_t)pos.bx * kColWaves;
    cplx<RC> d[1][L];
    col_load<L>(io.s0, tile, A.nz, plane, col0, m, d[0]);
#pragma unroll
    for (int r = 0; r < L; ++r)
        if (eq == 2 && r < m.cnt && m.k0 + r == A.nz - 1) d[0][r] = czero_t<cplx<RC>>();
    const int meq = eq == 0 || eq == 1 ? 0 : (eq == 2 ? 1 : (eq == 3 ? 2 : 3));
    RC a[L], b[L], c[L];
    assemble<L>(A, meq, l, jm, is00, m, a, b, c);
    if (is00 && eq != 1 && eq != 2) fixups<L>(A, meq, m, d[0]);
    if constexpr (decltype(m)::parts) {
        if (meq == 2) wave_tridiag_refined<L, 1>(a, b, c, d);
        else wave_tridiag<L, 1>(a, b, c, d);
    } else {
        if (meq == 2) lane_tridiag_refined<L, 1>(m.cnt, a, b, c, d);
        else lane_tridiag<L, 1>(m.cnt, a, b, c, d);
    }
    col_store<L>(io.s0, tile, A.nz, plane, col0, m, d[0]);
}

// k_column_mom with W columns per block in at most lim bytes of LDS: the fourth
// tile unless it does not fit or more blocks share a CU with three (the
// registers hold four blocks up to 3 levels per lane, three up to 5)
template <int L, int W>
static void mom_kernel(dim3 g, size_t lim, hipStream_t st, const StepArgs &A, const ColIO<double> &io)
{
    const size_t one = col_sub<W>(A.nz) * sizeof(double2), regs = L <= 3 ? 4 : L <= 5 ? 3 : 2;
    StepArgs M = A;
    M.ntile = 4 * one > lim || std::min(regs, kColLds / (3 * one)) > std::min(regs, kColLds / (4 * one)) ? 3 : 4;
    hipLaunchKernelGGL((k_column_mom<L, W>), dim3(g.x * (kColWaves / W), g.y), dim3(64 * W), M.ntile * one, st, M, io);
}

// Column kernels: kind 0 k_column_mom, 1 k_column_t, 2 k_column_project,
// 3 k_column_solve (equation eq).
template <int L, class RIO, class RC>
static void col_kernel(int kind, dim3 g, size_t lds, bool big, hipStream_t st, const StepArgs &A, const ColIO<RIO> &io,
                       int eq)
{
    const dim3 b(64 * kColWaves);
    switch (kind) {
    case 0:
        if constexpr (sizeof(RIO) == 4) {
            hipLaunchKernelGGL((k_column_mom_mixed<L, RC>), g, b, lds, st, A, io);
        } else {
            constexpr int W = mom_waves<L>();
            const size_t lim = big ? kColLds : kLdsDefault;
            if constexpr (L == 7 || L == 8)
                if (3 * col_sub<W>(A.nz) * sizeof(double2) > lim) {
                    mom_kernel<L, 2>(g, lim, st, A, io);
                    break;
                }
            mom_kernel<L, W>(g, lim, st, A, io);
        }
        break;
    case 1: hipLaunchKernelGGL((k_column_t<L, RIO, RC>), g, b, lds, st, A, io); break;
    case 2: hipLaunchKernelGGL((k_column_project<L, RIO, RC>), g, b, lds, st, A, io); break;
    default: hipLaunchKernelGGL((k_column_solve<L, RIO, RC>), g, b, lds, st, A, io, eq); break;
    }
}
// One column pass over spectra s[0..3] of V.  FP64 storage: every block in
// FP64.  Mixed: the low-wavenumber blocks in FP64, then the rest in FP32.
template <class R>
int launch_columns(hc_ctx *c, int kind, StepArgs A, const View<R> &V, int nfields, int eq)
{
    ColIO<R> io;
    io.s0 = V.s[0]; io.s1 = V.s[1]; io.s2 = V.s[2]; io.s3 = V.s[3];
    io.lo_l = c->lo_l; io.lo_m = c->lo_m;
    io.remap = c->tune.col_remap;
    if (A.zorder == 6) {  // 6th/4th-order z operators: every column in FP64 arithmetic
        launch_col6<R>(kind, c->stream, A, io, eq);
        return 0;
    }
    A.ntile = col_tiles(c, nfields, sizeof(cplx<R>));
    const size_t lds = col_lds(c, nfields, sizeof(cplx<R>));
    const dim3 gfull((c->nl + kColWaves - 1) / kColWaves, c->ny);
    if constexpr (std::is_same<R, double>::value) {
        io.sel = 0;
#define HC_CK(L_) col_kernel<L_, double, double>(kind, gfull, lds, c->big_lds, c->stream, A, io, eq);
        HC_DISPATCH_L(c->Lcol, HC_CK)
#undef HC_CK
    } else {
        if (c->lo_l > 0) {
            io.sel = 1;
            const dim3 glo(c->lo_l, 2 * c->lo_m + 1);
#define HC_CK(L_) col_kernel<L_, float, double>(kind, glo, lds, c->big_lds, c->stream, A, io, eq);
            HC_DISPATCH_L_MIXED(c->Lcol, HC_CK)
#undef HC_CK
        }
        io.sel = c->lo_l > 0 ? 2 : 0;
#define HC_CK(L_) col_kernel<L_, float, float>(kind, gfull, lds, c->big_lds, c->stream, A, io, eq);
        HC_DISPATCH_L_MIXED(c->Lcol, HC_CK)
#undef HC_CK
    }
    return 0;
}

template int launch_columns<double>(hc_ctx *, int, StepArgs, const View<double> &, int, int);
template int launch_columns<float>(hc_ctx *, int, StepArgs, const View<float> &, int, int);

hipError_t columns_set_lds(int L, bool mixed, int bytes)
{
    hipError_t e = hipSuccess;
#define HC_A1(K_)                                                                                                   \
    if (e == hipSuccess)                                                                                            \
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&K_), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
#define HC_A(L_) HC_A1((k_column_mom<L_>))
#define HC_AM(L_) HC_A1((k_column_mom_mixed<L_, float>)) HC_A1((k_column_mom_mixed<L_, double>))
    switch (L) {
    HC_CASES_L(HC_A)
    case 7: HC_A(7); break;
    case 10: HC_A(10); break;
    case 12: HC_A(12); break;
    case 14: HC_A(14); break;
    default: return hipErrorInvalidValue;
    }
    if (mixed)
        switch (L) {
        HC_CASES_L(HC_AM)
        default: return hipErrorInvalidValue;
        }
#undef HC_AM
#undef HC_A
#undef HC_A1
    return e;
}
