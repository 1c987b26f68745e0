// The divergence screen of time_advancement_fd / _sp: screen_div_error
// (src/module_io.f90:85-206), called after every substep with isfinal = 1
// (src/module_navier_stokes.f90:344-350) and at start-up with isfinal = 0.
//
// The reference scans the points in (k, j, i) order and keeps
//   div_avg      = sum |d| / (nx ny nz)
//   div_max      : starts at 0; at each point with |d| > div_max, div_max = d
//   div_hist_max : the same rule, kept across calls, updated when isfinal = 1
// and stops on the first NaN in u, v or w (screen_div_error_spec,
// src/module_spectral.f90:899-1007, stores |d|: plain maxima).  div_max and div_hist_max are
// therefore SIGNED and depend on the scan order: after a negative d is stored
// the next point always replaces it.
//
// Parallel form.  After a point is taken the state is its d, so the next
// point taken is the first later one with |d'| > d: a pointer that does not
// depend on how the scan got there.  A run of points therefore maps an
// incoming state S through the first point with |d| > S, which is one of the
// run's records (strict prefix maxima of |d|, about ln n of them), to the d
// where that point's chain of pointers ends.  Three launches:
//   k_div_units   d of 2048 consecutive points (scan order is memory order)
//                 in LDS, 32 chunks of 64.  Per chunk and point, the end of
//                 its chain within the chunk (next-greater search over a
//                 table of shuffled maxima, then pointer doubling).  One lane
//                 per record then walks the chunks to the end of the unit:
//                 records and their final states, sum of |d|, NaN flag.
//   k_div_groups  the same walk over the records of 64 units
//   k_div_final   one wavefront applies the groups to div_max and
//                 div_hist_max in order.
// The spectral path's states are plain maxima of |d|, which need no order:
//   k_div_max     sum, largest |d| and NaN flag of a block's share of the points
//   k_div_max_final  the blocks' to div_avg, div_max and div_hist_max
// A unit with more than kRec records (long monotone |d|) or a group of such
// units is walked by k_div_final point by point instead.  At 128x128x129 the
// three take 62 + 36 + 18 us; one wavefront that visited every taken point
// (a state that a negative d resets takes ~10% of all points) took 2350 us
// after a 28 us pass for the row maxima.
#include "hc_host.h"

#include <algorithm>
#include <mutex>

namespace {
constexpr int kScrLen = 32;
constexpr int kChunk = 64;                 // points of a chunk, units of a group
constexpr int kChunks = 32;                // chunks of a batch
constexpr int kBatch = kChunks * kChunk;   // points held in LDS at a time
constexpr int kRec = 32;                   // records kept per unit / group
// a unit's or group's summary: sum |d|, max |d|, NaN flag, number of records
// (-1: more than kRec, or a member had), records, final states
constexpr int kSum = 4 + 2 * kRec;

__global__ void k_scr_zero(double *f, int n)
{
    if ((int)threadIdx.x < n) f[threadIdx.x] = 0.0;
}

// signed divergence of point q (scan order) as the states keep it and the
// magnitude it is compared by; a NaN is never taken
template <int CDS, class R>
HC_DEV void point_div(const StepArgsT<R> &F, const StepArgs &D, unsigned q, double &d, double &a)
{
    const unsigned row = q / (unsigned)D.nx, i = q - row * (unsigned)D.nx;
    const unsigned k = row / (unsigned)D.ny, j = row - k * (unsigned)D.ny;
    d = div_at<CDS, R>(F, D, (int)i, (int)j, (int)k);
    a = fabs(d);
}

// One lane's walk state: lane r < nrec follows record r.
struct Walk {
    double S, rec, gmax;  // state, the record's magnitude, largest |d| so far (uniform)
    int nrec;             // uniform; -1 once there are more than kRec
};
// Lanes whose state the run [pm] (kChunk nondecreasing prefix maxima) beats:
// position of the first entry above S
HC_DEV int first_above(const double *pm, int n2, double S)
{
    int pos = 0;
    for (int st = n2 >> 1; st > 0; st >>= 1)
        if (!(pm[pos + st - 1] > S)) pos += st;
    return pos;
}
// new records of a run: bit set where entry `i` of the lanes is one; out = its final state
HC_DEV void add_records(Walk &w, unsigned long long m, double mag, double out, int lane)
{
    while (m) {
        const int b = __ffsll((long long)m) - 1;
        m &= m - 1;
        const double g = __shfl(mag, b, 64), o = __shfl(out, b, 64);
        if (w.nrec >= 0) {
            if (w.nrec == kRec) { w.nrec = -1; return; }
            if (lane == w.nrec) { w.rec = g; w.S = o; }
            ++w.nrec;
        }
    }
}
HC_DEV void write_summary(const Walk &w, double *o, double sum, int nan, int lane)
{
    if (lane == 0) { o[0] = sum; o[1] = w.gmax; o[2] = (double)nan; o[3] = (double)w.nrec; }
    if (lane < kRec) {
        const bool on = lane < w.nrec;
        o[4 + lane] = on ? w.rec : HUGE_VAL;
        o[4 + kRec + lane] = on ? w.S : 0.0;
    }
}

// Bound by the walk's LDS latency and the shuffles of the chunk tables, not
// by HBM: 2048 points keep 35 KB of LDS, four blocks per CU that hide each
// other's walks (128x128x129: 62 us; 107 with 4096 points, two blocks per CU,
// where four of the 516 blocks ran by themselves).
template <int CDS, class R>
__global__ __launch_bounds__(256) void k_div_units(StepArgsT<R> F, StepArgs D, unsigned N, int nb, double *units)
{
    __shared__ double dd[kBatch], pm[kBatch], cmax[kChunks], rs[4];
    __shared__ unsigned char ex[kBatch];
    __shared__ int rn[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const double ninf = -HUGE_VAL;
    double s = 0.0;
    int nan = 0;
    Walk w{0.0, 0.0, ninf, 0};
    for (int bt = 0; bt < nb; ++bt) {
        const size_t base = ((size_t)blockIdx.x * nb + bt) * kBatch;
        if (base >= N) break;
        for (int c = wv; c < kChunks; c += 4) {
            const size_t q = base + (size_t)c * kChunk + lane;
            double d = 0.0, a = ninf;
            if (q < N) {
                double mag;
                point_div<CDS, R>(F, D, (unsigned)q, d, mag);
                s += mag;
                if (mag >= 0.0) a = mag;
                const R u0 = F.u[q], v0 = F.v[q], w0 = F.w[q];
                if (u0 != u0 || v0 != v0 || w0 != w0) nan = 1;
            }
            // t[e] = max over the 2^e points after this one
            double t[6];
            t[0] = __shfl_down(a, 1, 64);
            if (lane == 63) t[0] = ninf;
#pragma unroll
            for (int e = 1; e < 6; ++e) {
                const int h = 1 << (e - 1);
                const double o = __shfl_down(t[e - 1], h, 64);
                t[e] = fmax(t[e - 1], lane + h < 64 ? o : ninf);
            }
            // the first later point with |d| > d, or this one
            int pos = lane;
#pragma unroll
            for (int e = 5; e >= 0; --e) {
                const double o = __shfl(t[e], pos & 63, 64);
                if (pos < 64 && !(o > d)) pos += 1 << e;
            }
            int p = pos + 1 < 64 ? pos + 1 : lane;
#pragma unroll
            for (int e = 0; e < 6; ++e) p = __shfl(p, p, 64);
            double m = a;
#pragma unroll
            for (int e = 1; e < 64; e <<= 1) {
                const double o = __shfl_up(m, e, 64);
                if (lane >= e) m = fmax(m, o);
            }
            const int at = c * kChunk + lane;
            dd[at] = d;
            pm[at] = m;
            ex[at] = (unsigned char)p;
            if (lane == 63) cmax[c] = m;
        }
        __syncthreads();
        if (wv == 0) {
            for (int c = 0; c < kChunks; ++c) {
                const double cm = cmax[c];
                const int at = c * kChunk;
                if (lane < w.nrec && cm > w.S) w.S = dd[at + ex[at + first_above(pm + at, kChunk, w.S)]];
                if (cm > w.gmax) {
                    const double mine = pm[at + lane], prev = lane ? pm[at + lane - 1] : ninf;
                    add_records(w, __ballot(mine > fmax(w.gmax, prev)), mine, dd[at + ex[at + lane]], lane);
                    w.gmax = cm;
                }
            }
        }
        __syncthreads();
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, 64);
        nan |= __shfl_xor(nan, o, 64);
    }
    if (lane == 0) { rs[wv] = s; rn[wv] = nan; }
    __syncthreads();
    if (wv == 0)
        write_summary(w, units + (size_t)blockIdx.x * kSum, (rs[0] + rs[1]) + (rs[2] + rs[3]),
                      rn[0] | rn[1] | rn[2] | rn[3], lane);
}

// 64 units to one summary, the same walk over their records
__global__ __launch_bounds__(64) void k_div_groups(const double *units, int nunit, double *groups)
{
    __shared__ double rec[kChunk][kRec], out[kChunk][kRec];
    const int lane = threadIdx.x, u0 = blockIdx.x * kChunk, n = min(kChunk, nunit - u0);
    const double ninf = -HUGE_VAL;
    for (int q = lane; q < n * 2 * kRec; q += 64) {
        const int u = q / (2 * kRec), r = q - u * 2 * kRec;
        const double v = units[(size_t)(u0 + u) * kSum + 4 + r];
        if (r < kRec) rec[u][r] = v;
        else out[u][r - kRec] = v;
    }
    double sum = 0.0, mx = ninf, cnt = 0.0;
    int nan = 0;
    if (lane < n) {
        const double *h = units + (size_t)(u0 + lane) * kSum;
        sum = h[0];
        mx = h[1];
        nan = h[2] != 0.0;
        cnt = h[3];
    }
    const bool bad = __any(cnt < 0.0);
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o, 64);
        nan |= __shfl_xor(nan, o, 64);
    }
    __syncthreads();
    Walk w{0.0, 0.0, ninf, bad ? -1 : 0};
    for (int c = 0; c < n; ++c) {
        const double cm = __shfl(mx, c, 64);
        if (!bad) {
            if (lane < w.nrec && cm > w.S) w.S = out[c][first_above(rec[c], kRec, w.S)];
            if (cm > w.gmax) {
                const bool on = lane < (int)__shfl(cnt, c, 64);
                const double mine = on ? rec[c][lane] : 0.0;
                add_records(w, __ballot(on && mine > w.gmax), mine, on ? out[c][lane] : 0.0, lane);
            }
        }
        w.gmax = fmax(w.gmax, cm);
    }
    write_summary(w, groups + (size_t)blockIdx.x * kSum, sum, nan, lane);
}

// State of the scan: s[0] = div_max, s[1] = div_hist_max (updated when fin)
struct ScanState {
    double s[2];
    int n;
    HC_DEV bool hit(double a) const { return a > s[0] || (n > 1 && a > s[1]); }
};
// a summary's n records applied to the states: the first record above each
HC_DEV void apply(ScanState &S, int n, double rec, double out, int lane)
{
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const unsigned long long m = __ballot(e < S.n && lane < n && rec > S.s[e]);
        if (m) S.s[e] = __shfl(out, __ffsll((long long)m) - 1, 64);
    }
}
// points [q0, q1) one at a time, 64 loaded together
template <int CDS, class R>
HC_DEV void scan_points(const StepArgsT<R> &F, const StepArgs &D, size_t q0, size_t q1, ScanState &S, int lane)
{
    for (size_t b = q0; b < q1; b += 64) {
        double d = 0.0, a = -HUGE_VAL;
        if (b + lane < q1) point_div<CDS, R>(F, D, (unsigned)(b + lane), d, a);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            int pos = -1;
            while (true) {
                const unsigned long long m = __ballot(e < S.n && lane > pos && a > S.s[e]);
                if (!m) break;
                pos = __ffsll((long long)m) - 1;
                S.s[e] = __shfl(d, pos, 64);
            }
        }
    }
}

// state[0]: div_hist_max before the call (updated in place when fin)
template <int CDS, class R>
__global__ __launch_bounds__(64) void k_div_final(StepArgsT<R> F, StepArgs D, unsigned N, int nb, const double *units,
                                                  int nunit, const double *groups, int ngroup, double *state,
                                                  double *rec, int fin)
{
    const int lane = threadIdx.x;
    double s = 0.0;
    int nan = 0;
    for (int g = lane; g < ngroup; g += 64) {
        s += groups[(size_t)g * kSum];
        nan |= groups[(size_t)g * kSum + 2] != 0.0;
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, 64);
        nan |= __shfl_xor(nan, o, 64);
    }
    ScanState S{{0.0, state[0]}, fin ? 2 : 1};
    if (!nan) {
        constexpr int U = 8;  // summaries loaded ahead of their use
        for (int g0 = 0; g0 < ngroup; g0 += U) {
            double mx[U], ct[U], rc[U], ou[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double *h = groups + (size_t)min(g0 + u, ngroup - 1) * kSum;
                mx[u] = h[1];
                ct[u] = h[3];
                rc[u] = h[4 + (lane & (kRec - 1))];
                ou[u] = h[4 + kRec + (lane & (kRec - 1))];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int g = g0 + u;
                if (g >= ngroup || !S.hit(mx[u])) continue;
                if (ct[u] >= 0.0) {
                    apply(S, (int)ct[u], rc[u], ou[u], lane);
                    continue;
                }
                for (int q = g * kChunk; q < min((g + 1) * kChunk, nunit); ++q) {
                    const double *h = units + (size_t)q * kSum;
                    if (!S.hit(h[1])) continue;
                    if (h[3] >= 0.0) {
                        apply(S, (int)h[3], h[4 + (lane & (kRec - 1))], h[4 + kRec + (lane & (kRec - 1))], lane);
                    } else {
                        const size_t per = (size_t)nb * kBatch, q0 = q * per;
                        scan_points<CDS, R>(F, D, q0, q0 + per < N ? q0 + per : (size_t)N, S, lane);
                    }
                }
            }
        }
    }
    if (lane == 0) {
        rec[0] = s / ((double)D.nx * D.ny * D.nz);
        rec[1] = S.s[0];
        rec[2] = S.s[1];
        rec[3] = nan;
        if (fin && !nan) state[0] = S.s[1];
    }
}

// The largest |d| of the spectral path (screen_div_error_spec stores |d|,
// src/module_spectral.f90:931-946), whose divergence lies in F.aux: a NaN is
// never taken.  Bound by HBM: four reads of every point, four points of a
// thread in flight (256x256x257: 122 us, 4.4 TB/s; a whole screen of that grid
// 351 us, 501 with the units and records of the signed states, and 71 against
// 151 at 128x128x129).
constexpr int kMaxBlocks = 2048;  // eight blocks of four wavefronts per CU
template <class R>
__global__ __launch_bounds__(256) void k_div_max(StepArgsT<R> F, unsigned N, double *part)
{
    __shared__ double rs[4], rm[4];
    __shared__ int rn[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double s = 0.0, m = -HUGE_VAL;
    int nan = 0;
    constexpr int U = 4;
    for (size_t q0 = (size_t)blockIdx.x * 256 * U + threadIdx.x; q0 < N; q0 += (size_t)gridDim.x * 256 * U) {
        R d[U], u[U], v[U], w[U];
#pragma unroll
        for (int e = 0; e < U; ++e) {
            const size_t q = min(q0 + 256 * e, (size_t)N - 1);
            d[e] = F.aux[q]; u[e] = F.u[q]; v[e] = F.v[q]; w[e] = F.w[q];
        }
#pragma unroll
        for (int e = 0; e < U; ++e) {
            if (q0 + 256 * e >= N) continue;
            const double a = fabs((double)d[e]);
            s += a;
            if (a > m) m = a;
            if (u[e] != u[e] || v[e] != v[e] || w[e] != w[e]) nan = 1;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, 64);
        m = fmax(m, __shfl_xor(m, o, 64));
        nan |= __shfl_xor(nan, o, 64);
    }
    if (lane == 0) { rs[wv] = s; rm[wv] = m; rn[wv] = nan; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double *o = part + 3 * (size_t)blockIdx.x;
        o[0] = (rs[0] + rs[1]) + (rs[2] + rs[3]);
        o[1] = fmax(fmax(rm[0], rm[1]), fmax(rm[2], rm[3]));
        o[2] = (double)(rn[0] | rn[1] | rn[2] | rn[3]);
    }
}

// state and rec as k_div_final's
__global__ __launch_bounds__(256) void k_div_max_final(const double *part, int nblk, double np, double *state,
                                                       double *rec, int fin)
{
    __shared__ double rs[4], rm[4];
    __shared__ int rn[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double s = 0.0, m = -HUGE_VAL;
    int nan = 0;
    for (int b = threadIdx.x; b < nblk; b += 256) {
        s += part[3 * (size_t)b];
        m = fmax(m, part[3 * (size_t)b + 1]);
        nan |= part[3 * (size_t)b + 2] != 0.0;
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, 64);
        m = fmax(m, __shfl_xor(m, o, 64));
        nan |= __shfl_xor(nan, o, 64);
    }
    if (lane == 0) { rs[wv] = s; rm[wv] = m; rn[wv] = nan; }
    __syncthreads();
    if (threadIdx.x == 0) {
        nan = rn[0] | rn[1] | rn[2] | rn[3];
        m = fmax(fmax(rm[0], rm[1]), fmax(rm[2], rm[3]));
        const double hist = state[0], h = fin && !nan && m > hist ? m : hist;
        rec[0] = ((rs[0] + rs[1]) + (rs[2] + rs[3])) / np;
        rec[1] = !nan && m > 0.0 ? m : 0.0;
        rec[2] = h;
        rec[3] = nan;
        state[0] = h;
    }
}

__global__ void k_scr_set(double *f, double v)
{
    if (threadIdx.x == 0) f[0] = v;
}

// Partials of one screen: the units' and groups' summaries
struct ScreenBufs {
    double *units, *groups, *state, *rec;
    int nb;  // batches of 2048 points per unit
};
inline int screen_units(const hc_ctx *c, int nb)
{
    const size_t N = (size_t)c->nx * c->ny * c->nz, per = (size_t)nb * kBatch;
    return (int)((N + per - 1) / per);
}
inline int screen_groups(int nunit) { return (nunit + kChunk - 1) / kChunk; }

template <int CDS, class R>
void launch_screen(hc_ctx *c, const StepArgsT<R> &F, const StepArgs &D, const ScreenBufs &B, int fin)
{
    const unsigned N = (unsigned)c->nx * (unsigned)c->ny * (unsigned)c->nz;
    const int nu = screen_units(c, B.nb), ng = screen_groups(nu);
    hipLaunchKernelGGL((k_div_units<CDS, R>), dim3(nu), dim3(256), 0, c->stream, F, D, N, B.nb, B.units);
    hipLaunchKernelGGL(k_div_groups, dim3(ng), dim3(64), 0, c->stream, B.units, nu, B.groups);
    hipLaunchKernelGGL((k_div_final<CDS, R>), dim3(1), dim3(64), 0, c->stream, F, D, N, B.nb, B.units, nu, B.groups, ng,
                       B.state, B.rec, fin);
}

// the spectral path: three values per block, fewer than a unit's summary each
template <class R>
void launch_screen_max(hc_ctx *c, const StepArgsT<R> &F, const ScreenBufs &B, int fin)
{
    const unsigned N = (unsigned)c->nx * (unsigned)c->ny * (unsigned)c->nz;
    const int nblk = (int)std::min((N + 1023) / 1024, (unsigned)kMaxBlocks);
    hipLaunchKernelGGL((k_div_max<R>), dim3(nblk), dim3(256), 0, c->stream, F, N, B.units);
    hipLaunchKernelGGL(k_div_max_final, dim3(1), dim3(256), 0, c->stream, B.units, nblk,
                       (double)c->nx * c->ny * c->nz, B.state, B.rec, fin);
}

// Queue a screen of the context's current fields with the partials in B.
int queue_screen(hc_ctx *c, const ScreenBufs &B, int fin)
{
    StepArgs A = base_args(c);
    if (c->prm.cds == 3)
        if (int e = spec_divergence(c)) return e;
    if (c->mixed) {
        StepArgsT<float> F = rows_args<float>(A, c->m32);
        F.aux = c->m32.ptmp;
        if (c->prm.cds == 1) launch_screen<1, float>(c, F, A, B, fin);
        else if (c->prm.cds == 2) launch_screen<2, float>(c, F, A, B, fin);
        else launch_screen_max<float>(c, F, B, fin);
    } else {
        A.aux = c->ptmp;
        if (c->prm.cds == 1) launch_screen<1, double>(c, A, A, B, fin);
        else if (c->prm.cds == 2) launch_screen<2, double>(c, A, A, B, fin);
        else launch_screen_max<double>(c, A, B, fin);
    }
    HIPCHK(hipGetLastError());
    return 0;
}
}  // namespace

int screen_alloc(hc_ctx *c)
{
    if (c->scr) return 0;
    const int nu = screen_units(c, 1), ng = screen_groups(nu);
    int e = dalloc(c, (void **)&c->scr, kScrLen * sizeof(double));
    if (!e) e = dalloc(c, (void **)&c->scr_units, (size_t)nu * kSum * sizeof(double));
    if (!e) e = dalloc(c, (void **)&c->scr_groups, (size_t)ng * kSum * sizeof(double));
    if (!e) {
        // div_hist_max starts at 0 (module_io's save variable)
        hipLaunchKernelGGL(k_scr_zero, dim3(1), dim3(64), 0, c->stream, c->scr, kScrLen);
        HIPCHK(hipGetLastError());
    }
    return e;
}

// Queue the screen of the current fields into record slot `slot` (4 doubles
// at c->scr + 4 + 4 slot: div_avg, div_max, div_hist_max, NaN flag).
int screen_queue(hc_ctx *c, int slot, int fin)
{
    if (int e = screen_alloc(c)) return e;
    return queue_screen(c, ScreenBufs{c->scr_units, c->scr_groups, c->scr, c->scr + 4 + 4 * slot, 1}, fin);
}

// ---------------------------------------------------------------------------
// The screen without allocation: its partials live in `scratch`, a
// file-scope device array that every GPU the library runs on holds until the
// process ends.  Host code never passes the array's name to a kernel (that is
// a host-side stand-in, not a device address): the device address is looked
// up once per device with hipGetSymbolAddress and kept in g_scratch.
namespace {
constexpr size_t kScratchDoubles = (size_t)1 << 19;  // 4 MiB
constexpr int kMaxDevices = 64;
__device__ __align__(256) double scratch[kScratchDoubles];
double *g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mu;

int scratch_ptr(int device, double **out)
{
    if (device < 0 || device >= kMaxDevices) return set_err(HC_ERR_ARG, "device %d out of range", device);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[device]) {
        void *p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_err(HC_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch[device] = (double *)p;
    }
    *out = g_scratch[device];
    return 0;
}
}  // namespace

extern "C" int hc_screen_div_error_noalloc(hc_ctx *c, int isfinal, double *div_avg, double *div_max,
                                           double *div_hist_max)
{
    if (!c || !div_hist_max) return set_err(HC_ERR_ARG, "null argument");
    if (isfinal != 0 && isfinal != 1) return set_err(HC_ERR_ARG, "isfinal must be 0 or 1");
    // the grids that are taken: the limit is that of row maxima and block sums
    // (ny nz rows and 3 values for 16 rows of a level), which the summaries of
    // units no longer need and which stays so that no answer changes
    const size_t need = 8 + (size_t)c->ny * c->nz + 3 * (size_t)((c->ny + 15) / 16) * c->nz;
    // units of as many batches as make their summaries fit: 1 to 16 (a grid of
    // this size has nx <= 512, so under 2^28 points)
    int nb = 1, nu = screen_units(c, 1);
    while (nb < 64 && 8 + (size_t)(nu + screen_groups(nu)) * kSum > kScratchDoubles) {
        nb *= 2;
        nu = screen_units(c, nb);
    }
    if (need > kScratchDoubles || 8 + (size_t)(nu + screen_groups(nu)) * kSum > kScratchDoubles)
        return set_err(HC_ERR_ARG, "screen partials of %zu doubles (ny=%d, nz=%d) exceed the scratch of %zu doubles",
                       need, c->ny, c->nz, kScratchDoubles);
    int dev = -1;
    HIPCHK(hipGetDevice(&dev));
    if (dev != c->device) return set_err(HC_ERR_ARG, "the context lives on device %d, current is %d", c->device, dev);
    double *ptr = nullptr;
    if (int e = scratch_ptr(dev, &ptr)) return e;
    // scratch layout: [0] div_hist_max in/out, [4..7] the record, then the
    // units' and the groups' summaries (both fully rewritten by each call)
    const ScreenBufs B{ptr + 8, ptr + 8 + (size_t)nu * kSum, ptr, ptr + 4, nb};
    hipLaunchKernelGGL(k_scr_set, dim3(1), dim3(64), 0, c->stream, ptr, *div_hist_max);
    HIPCHK(hipGetLastError());
    if (int e = queue_screen(c, B, isfinal)) return e;
    double rec[4];
    HIPCHK(hipMemcpyAsync(rec, ptr + 4, sizeof rec, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (div_avg) *div_avg = rec[0];
    if (div_max) *div_max = rec[1];
    *div_hist_max = rec[2];
    if (rec[3] != 0.0) return set_err(HC_ERR_NAN, "NaN error!");
    return 0;
}
