// sn_aux_kernels.h -- kernels beside the tile sweep (gfx950, FP64):
// sweep-counter bump, the site_energy batch, sequential replay, energy /
// adjoint beyond cut-off 5, reductions, moment, device lattices, the random
// initial lattice and the recombination sums.  Included by sn_api.hip only
// (non-template kernels: one definition).
#pragma once
#include "sn_kernels.h"

namespace sn {
__global__ void bump_sweep_kernel(unsigned *sweep_ctr, int R, unsigned n)
{
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < R) sweep_ctr[r] += n;
}

// Local field pieces of one site (the site_energy batch), and by direct
// gathers from HBM (energy / adjoint beyond cut-off 5).
struct FieldOut {
    double hx, hy, hz;  // sum_r L_j (p_j - 3 n (n.p_j)) / d^3
    double gx, gy, gz;  // sum_{|r|=1} p_j
};

__device__ __forceinline__ void site_field(const double4 *lat, const RepDev &rep, const PairDev *offs,
                                           int noff, int x, int y, int z, FieldOut &f)
{
    f.hx = f.hy = f.hz = f.gx = f.gy = f.gz = 0.0;
    for (int i = 0; i < noff; i++) {
        const PairDev o = offs[i];
        int gx = wrap_once(x + o.dx, rep.X), gy = wrap_once(y + o.dy, rep.Y), gz = wrap_once(z + o.dz, rep.Z);
        double4 t = lat[((long long)gx * rep.Y + gy) * rep.Z + gz];
        double s = o.nx * t.x + o.ny * t.y + o.nz * t.z;
        double wl = o.w * t.w;
        double ts = -3.0 * wl * s;
        f.hx += wl * t.x + ts * o.nx;
        f.hy += wl * t.y + ts * o.ny;
        f.hz += wl * t.z + ts * o.nz;
        if (o.nn) { f.gx += t.x; f.gy += t.y; f.gz += t.z; }
    }
}

// Energy differences of proposed moves.  G lanes share a move: lanes next to
// each other read offsets next to each other, mostly one run along z, so a
// gather touches a third of the cache lines that 64 moves a wave did, and a
// single move has its neighbours in flight together.  The offset table is in
// LDS, padded with zero weights to a whole number of rounds; groups take moves
// in turn until none is left.  100000 moves of a 64^3 lattice at cut-off 3:
// 53 us (99 us with a move per lane), one move 2.8 us (10 us); bound by the
// gathers' cache lines.  G is the power of two, at most 16, that leaves about
// four rounds, whose gathers are in flight together: fewer lanes for short
// tables, since a move's own work (site, proposal, result) is done by each of
// its lanes.  A call of 200000 moves: 64^3, cut-off 1, 354 us with 2 lanes, 367
// with 16; 2D, cut-off 2, 358 us with 4, 369 with 16 (mostly copies).
constexpr int kMoveThreads = 256;
constexpr int kMoveBlocks = 2048;   // eight workgroups a CU

__host__ __device__ inline int move_lanes(int noff)
{
    int G = 1;
    while (G < 16 && 4 * G < noff) G *= 2;
    return G;
}
__host__ __device__ inline int move_rounds(int noff, int G)
{
    const int rounds = (noff + G - 1) / G;
    return rounds < 4 ? 4 : rounds;
}
inline size_t move_lds(int noff)
{
    const int G = move_lanes(noff);
    return (size_t)move_rounds(noff, G) * G * (sizeof(double2) + sizeof(int2));
}

// q = s / d and the remainder, for 0 <= s < 2^31: id = 1 / d is within an ulp,
// so the quotient is at most one off.
__device__ __forceinline__ int divide(int s, int d, double id, int &rest)
{
    int q = (int)(s * id);
    rest = s - q * d;
    if (rest < 0) { q--; rest += d; }
    if (rest >= d) { q++; rest -= d; }
    return q;
}

template <int G>
__global__ __launch_bounds__(kMoveThreads) void site_energy_batch_kernel(
    const double4 *__restrict__ lat, const RepDev *__restrict__ reps, int replica,
    const PairDev *__restrict__ offs, int noff, long long n, const int *__restrict__ site,
    const double *__restrict__ prop, double *__restrict__ dE)
{
    extern __shared__ double2 s_w[];   // w, 3 w / |r|^2
    const int rounds = move_rounds(noff, G);
    int2 *const s_d = (int2 *)(s_w + rounds * G);   // dx, dy; dz, nearest neighbour
    for (int i = threadIdx.x; i < rounds * G; i += kMoveThreads) {
        double2 w = make_double2(0.0, 0.0);
        int2 d = make_int2(0, 0);
        if (i < noff) {
            const PairDev o = offs[i];
            w = make_double2(o.w, 3.0 * o.w / (double)(o.dx * o.dx + o.dy * o.dy + o.dz * o.dz));
            d = make_int2((o.dx & 0xFFFF) | (o.dy << 16), (o.dz & 0xFFFF) | (o.nn << 16));
        }
        s_w[i] = w;
        s_d[i] = d;
    }
    __syncthreads();
    const RepDev rep = reps[replica];
    const double4 *L = lat + rep.base;
    const long long N = (long long)rep.X * rep.Y * rep.Z;
    const double iY = 1.0 / rep.Y, iZ = 1.0 / rep.Z;
    const int lane = threadIdx.x % G;
    const long long step = (long long)gridDim.x * (kMoveThreads / G);
    for (long long k = (long long)blockIdx.x * (kMoveThreads / G) + threadIdx.x / G; k < n; k += step) {
        const int s = site[k];
        const double px = prop[3 * k], py = prop[3 * k + 1], pz = prop[3 * k + 2];
        // an index outside the replica reads nothing and yields NaN
        if (s < 0 || s >= N) {
            if (lane == 0) dE[k] = __builtin_nan("");
            continue;
        }
        int z, y;
        const int x = divide(divide(s, rep.Z, iZ, z), rep.Y, iY, y);
        const double4 o = L[s];
        const double dx = px - o.x, dy = py - o.y, dz = pz - o.z;
        FieldOut f = {};
        auto offset = [&](int i, int2 &d) __attribute__((always_inline)) {
            d = s_d[i];
            const int gx = wrap_once(x + (short)d.x, rep.X), gy = wrap_once(y + (d.x >> 16), rep.Y),
                      gz = wrap_once(z + (short)d.y, rep.Z);
            return L[((long long)gx * rep.Y + gy) * rep.Z + gz];
        };
        auto add = [&](int i, const int2 &d, const double4 &q) __attribute__((always_inline)) {
            const double2 w = s_w[i];
            const double rx = (short)d.x, ry = d.x >> 16, rz = (short)d.y;
            const double wl = w.x * q.w, ts = -(w.y * q.w) * (rx * q.x + ry * q.y + rz * q.z);
            f.hx += wl * q.x + ts * rx;
            f.hy += wl * q.y + ts * ry;
            f.hz += wl * q.z + ts * rz;
            if (d.y >> 16) { f.gx += q.x; f.gy += q.y; f.gz += q.z; }
        };
        int t = 0;
        for (; t + 4 <= rounds; t += 4) {
            int2 d[4];
            double4 q[4];
#pragma unroll
            for (int j = 0; j < 4; j++) q[j] = offset((t + j) * G + lane, d[j]);
#pragma unroll
            for (int j = 0; j < 4; j++) add((t + j) * G + lane, d[j], q[j]);
        }
        for (; t < rounds; t++) {
            int2 d;
            const double4 q = offset(t * G + lane, d);
            add(t * G + lane, d, q);
        }
        f.hx = group_sum_dpp<G>(f.hx);
        f.hy = group_sum_dpp<G>(f.hy);
        f.hz = group_sum_dpp<G>(f.hz);
        f.gx = group_sum_dpp<G>(f.gx);
        f.gy = group_sum_dpp<G>(f.gy);
        f.gz = group_sum_dpp<G>(f.gz);
        double e = o.w * (dx * f.hx + dy * f.hy + dz * f.hz) - rep.J * (dx * f.gx + dy * f.gy + dz * f.gz) +
                   (dx * rep.E[0] + dy * rep.E[1] + dz * rep.E[2]);
        if (rep.K > 0.0) e += -rep.K * (fabs(px) - fabs(o.x) + fabs(py) - fabs(o.y));
        if (lane == 0) dE[k] = e;
    }
}

// Sequential replay of recorded moves: one workgroup, one move at a time;
// lanes split the neighbour list, a workgroup reduction gives h, g and the
// rounding scale, lane 0 decides and writes.
__global__ __launch_bounds__(256) void replay_kernel(double4 *lat, const RepDev *reps, int replica,
                                                     const PairDev *offs, int noff, long long n,
                                                     const int *site, const double *prop,
                                                     const double *u, const unsigned char *u_drawn,
                                                     const unsigned char *ref_accept,
                                                     unsigned char *decision,
                                                     unsigned long long *stats)
{
    __shared__ double red[7][256];
    const int tid = threadIdx.x;
    const RepDev rep = reps[replica];
    double4 *L = lat + rep.base;
    unsigned long long mism = 0, ties = 0, nacc = 0, nrej = 0;
    for (long long k = 0; k < n; k++) {
        const int s = site[k];
        const int z = s % rep.Z, q = s / rep.Z, y = q % rep.Y, x = q / rep.Y;
        const double4 o = L[s];
        const double px = prop[3 * k], py = prop[3 * k + 1], pz = prop[3 * k + 2];
        double v[7] = {0, 0, 0, 0, 0, 0, 0};
        for (int i = tid; i < noff; i += 256) {
            const PairDev of = offs[i];
            int gx = wrap_once(x + of.dx, rep.X), gy = wrap_once(y + of.dy, rep.Y), gz = wrap_once(z + of.dz, rep.Z);
            double4 t = L[((long long)gx * rep.Y + gy) * rep.Z + gz];
            double s_ = of.nx * t.x + of.ny * t.y + of.nz * t.z;
            double wl = of.w * t.w;
            double ts = -3.0 * wl * s_;
            v[0] += wl * t.x + ts * of.nx;
            v[1] += wl * t.y + ts * of.ny;
            v[2] += wl * t.z + ts * of.nz;
            if (of.nn) { v[3] += t.x; v[4] += t.y; v[5] += t.z; }
            // rounding scale of the reference's float terms for this neighbour
            double pn = fabs(px * t.x + py * t.y + pz * t.z), po = fabs(o.x * t.x + o.y * t.y + o.z * t.z);
            double an = fabs(of.nx * px + of.ny * py + of.nz * pz), ao = fabs(of.nx * o.x + of.ny * o.y + of.nz * o.z);
            v[6] += fabs(o.w * t.w) * of.w * (pn + po + 3.0 * fabs(s_) * (an + ao));
            if (of.nn) v[6] += fabs(rep.J) * (pn + po);
        }
        for (int c = 0; c < 7; c++) red[c][tid] = v[c];
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if (tid < st)
                for (int c = 0; c < 7; c++) red[c][tid] += red[c][tid + st];
            __syncthreads();
        }
        if (tid == 0) {
            const double dx = px - o.x, dy = py - o.y, dz = pz - o.z;
            double e = o.w * (dx * red[0][0] + dy * red[1][0] + dz * red[2][0]) -
                       rep.J * (dx * red[3][0] + dy * red[4][0] + dz * red[5][0]) +
                       (dx * rep.E[0] + dy * rep.E[1] + dz * rep.E[2]);
            double scale = red[6][0] + fabs(px * rep.E[0] + py * rep.E[1] + pz * rep.E[2]) +
                           fabs(o.x * rep.E[0] + o.y * rep.E[1] + o.z * rep.E[2]);
            if (rep.K > 0.0) {
                e += -rep.K * (fabs(px) - fabs(o.x) + fabs(py) - fabs(o.y));
                scale += rep.K * (fabs(px) + fabs(o.x) + fabs(py) + fabs(o.y));
            }
            // float rounding bound of the reference's dE (terms in float,
            // summed in double, result rounded to float)
            const double delta = 4e-6 * scale + 2e-7 * fabs(e);
            const int ref = ref_accept[k] ? 1 : 0;
            int mine = -1;   // -1: undecidable without a u the reference never drew
            bool tie = false;
            if (e < 0.0) mine = 1;
            else if (u_drawn[k]) mine = exp(-e * rep.beta) > u[k];
            if (fabs(e) <= delta) tie = true;
            if (u_drawn[k] && !__builtin_isinf(rep.beta)) {
                double g = exp(-e * rep.beta);
                double bound = rep.beta * delta * exp(-(e - delta) * rep.beta);
                if (fabs(g - u[k]) <= bound) tie = true;
            }
            int apply = ref;
            if (mine != ref) {
                if (tie) ties++;
                else mism++;
            }
            if (o.w != 0.0) {
                if (apply) { L[s] = make_double4(px, py, pz, o.w); nacc++; }
                else nrej++;
            }
            decision[k] = (unsigned char)apply;
        }
        __syncthreads();
    }
    if (tid == 0) { stats[0] = mism; stats[1] = ties; stats[2] = nacc; stats[3] = nrej; }
}

// Energy and adjoint at cut-offs beyond energy_kernel's: one site per lane; per-site gradient dE/dp_i and
// per-workgroup partial sums of
//   {E_dd, E_cage, E_field, E_K, dE/dJ, dE/dEx, dE/dEy, dE/dEz, dE/ds, dE/dK}.
constexpr int kNPart = 10;

__global__ __launch_bounds__(256) void energy_grad_kernel(const double4 *lat, const RepDev *reps,
                                                          int replica, const PairDev *offs, int noff,
                                                          double *grad, double *partials)
{
    __shared__ double red[kNPart][256];
    const int tid = threadIdx.x;
    const RepDev rep = reps[replica];
    const double4 *L = lat + rep.base;
    const long long N = (long long)rep.X * rep.Y * rep.Z;
    long long s = (long long)blockIdx.x * blockDim.x + tid;
    double v[kNPart];
    for (int c = 0; c < kNPart; c++) v[c] = 0.0;
    if (s < N) {
        int z = (int)(s % rep.Z), q = (int)(s / rep.Z), y = q % rep.Y, x = q / rep.Y;
        double4 p = L[s];
        FieldOut f;
        site_field(L, rep, offs, noff, x, y, z, f);
        double ph = p.x * f.hx + p.y * f.hy + p.z * f.hz;
        double pg = p.x * f.gx + p.y * f.gy + p.z * f.gz;
        double gx = p.w * f.hx - rep.J * f.gx + rep.E[0];
        double gy = p.w * f.hy - rep.J * f.gy + rep.E[1];
        double gz = p.w * f.hz - rep.J * f.gz + rep.E[2];
        double ak = fabs(p.x) + fabs(p.y);
        if (rep.K > 0.0) {
            gx -= rep.K * ((p.x > 0.0) - (p.x < 0.0));
            gy -= rep.K * ((p.y > 0.0) - (p.y < 0.0));
        }
        if (grad) { grad[3 * s] = gx; grad[3 * s + 1] = gy; grad[3 * s + 2] = gz; }
        v[0] = 0.5 * p.w * ph;
        v[1] = -0.5 * rep.J * pg;
        v[2] = p.x * rep.E[0] + p.y * rep.E[1] + p.z * rep.E[2];
        v[3] = rep.K > 0.0 ? -rep.K * ak : 0.0;
        v[4] = -0.5 * pg;
        v[5] = p.x; v[6] = p.y; v[7] = p.z;
        v[8] = p.w * ph;
        v[9] = rep.K > 0.0 ? -ak : 0.0;
    }
    for (int c = 0; c < kNPart; c++) red[c][tid] = v[c];
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st)
            for (int c = 0; c < kNPart; c++) red[c][tid] += red[c][tid + st];
        __syncthreads();
    }
    if (tid < kNPart) partials[(long long)blockIdx.x * kNPart + tid] = red[tid][0];
}

// Fixed-order sum of per-block partials (deterministic).  Workgroup (g, y)
// sums columns [g*kReduceCols, (g+1)*kReduceCols) of rows [seg[y], seg[y+1])
// (all nblocks rows when seg is null) of the nblocks x width table into
// out[y * width + col].  A wave owns a column: its lanes Neumaier-sum every
// 64th row, four in flight, and one compensated xor butterfly joins them.
// Bound by latency (loads, six exchanges): 2.8 us for 240 rows of 10 columns
// and 5.4 us for 256 of 162, against 8.3 and 16.6 us with every lane on all
// columns of its rows and a butterfly for each.
constexpr int kReduceCols = 16;
constexpr int kReduceThreads = 64 * kReduceCols;

__device__ __forceinline__ void neumaier_add(double &s, double &c, double v)
{
    const double t = s + v;
    c += (fabs(s) >= fabs(v)) ? (s - t) + v : (v - t) + s;
    s = t;
}

__global__ __launch_bounds__(kReduceThreads) void reduce_partials_kernel(const double *__restrict__ partials,
                                                                         int nblocks, int width,
                                                                         double *__restrict__ out, const int *seg)
{
    const int lane = threadIdx.x & 63, col = blockIdx.x * kReduceCols + (threadIdx.x >> 6);
    if (col >= width) return;
    const int b0 = seg ? seg[blockIdx.y] : 0, b1 = seg ? seg[blockIdx.y + 1] : nblocks;
    const double *p = partials + col;
    double s = 0.0, c = 0.0;
    int b = b0 + lane;
    for (; b + 192 < b1; b += 256) {
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = p[(long long)(b + 64 * k) * width];
#pragma unroll
        for (int k = 0; k < 4; k++) neumaier_add(s, c, v[k]);
    }
    {   // the last rows, together as well (a row beyond the end adds nothing)
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = b + 64 * k < b1 ? p[(long long)(b + 64 * k) * width] : 0.0;
#pragma unroll
        for (int k = 0; k < 4; k++) neumaier_add(s, c, v[k]);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double v = __shfl_xor(s, o, 64), cv = __shfl_xor(c, o, 64);
        c += cv;
        neumaier_add(s, c, v);
    }
    if (lane == 0) out[(long long)blockIdx.y * width + col] = s + c;
}

// Sum of dipole vectors (partials per block, then reduce_partials_kernel).
__global__ __launch_bounds__(256) void moment_kernel(const double4 *lat, const RepDev *reps, int replica,
                                                     double *partials)
{
    __shared__ double red[3][256];
    const int tid = threadIdx.x;
    const RepDev rep = reps[replica];
    const long long N = (long long)rep.X * rep.Y * rep.Z;
    double v0 = 0, v1 = 0, v2 = 0;
    for (long long s = (long long)blockIdx.x * blockDim.x + tid; s < N; s += (long long)gridDim.x * blockDim.x) {
        double4 p = lat[rep.base + s];
        v0 += p.x; v1 += p.y; v2 += p.z;
    }
    red[0][tid] = v0; red[1][tid] = v1; red[2][tid] = v2;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) for (int c = 0; c < 3; c++) red[c][tid] += red[c][tid + st];
        __syncthreads();
    }
    if (tid < 3) partials[(long long)blockIdx.x * 3 + tid] = red[tid][0];
}

// Scan of a lattice written from device memory: per workgroup {count of
// non-finite values, min length, max length} (the checks sn_set_lattice makes
// on the host).
__global__ __launch_bounds__(256) void lattice_scan_kernel(const double4 *lat, long long N, double *partials)
{
    __shared__ double red[3][256];
    const int tid = threadIdx.x;
    double bad = 0.0, lo = INFINITY, hi = -INFINITY;
    for (long long s = (long long)blockIdx.x * blockDim.x + tid; s < N; s += (long long)gridDim.x * blockDim.x) {
        const double4 p = lat[s];
        if (!isfinite(p.x) || !isfinite(p.y) || !isfinite(p.z) || !isfinite(p.w)) bad += 1.0;
        lo = fmin(lo, p.w);
        hi = fmax(hi, p.w);
    }
    red[0][tid] = bad; red[1][tid] = lo; red[2][tid] = hi;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) {
            red[0][tid] += red[0][tid + st];
            red[1][tid] = fmin(red[1][tid], red[1][tid + st]);
            red[2][tid] = fmax(red[2][tid], red[2][tid + st]);
        }
        __syncthreads();
    }
    if (tid < 3) partials[(long long)blockIdx.x * 3 + tid] = red[tid][0];
}

// Second pass of a lattice written from device memory: every workgroup sums
// up the scan's partials, and copies its share if nothing was non-finite; the
// first also reports {count, min, max} to `verdict` (pinned host memory).
__global__ __launch_bounds__(256) void lattice_take_kernel(const double4 *src, double4 *dst, long long N,
                                                           const double *partials, int nblk, double *verdict)
{
    __shared__ double red[3][4];
    const int tid = threadIdx.x;
    double bad = 0.0, lo = INFINITY, hi = -INFINITY;
    for (int b = tid; b < nblk; b += 256) {
        bad += partials[3 * b];
        lo = fmin(lo, partials[3 * b + 1]);
        hi = fmax(hi, partials[3 * b + 2]);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        bad += __shfl_xor(bad, o, 64);
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
    }
    if ((tid & 63) == 0) { red[0][tid >> 6] = bad; red[1][tid >> 6] = lo; red[2][tid >> 6] = hi; }
    __syncthreads();
    bad = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    if (blockIdx.x == 0 && tid == 0) {
        verdict[0] = bad;
        verdict[1] = fmin(fmin(red[1][0], red[1][1]), fmin(red[1][2], red[1][3]));
        verdict[2] = fmax(fmax(red[2][0], red[2][1]), fmax(red[2][2], red[2][3]));
    }
    if (bad > 0.0) return;   // uniform
    for (long long s = (long long)blockIdx.x * 256 + tid; s < N; s += (long long)gridDim.x * 256) dst[s] = src[s];
}

// A replica's record, passed as an argument: in stream order, no copy to wait for.
__global__ void put_rep_kernel(RepDev *dst, RepDev rep) { *dst = rep; }

// Random initial lattice on the device: unit dipole from the counter RNG
// (stream tag 0xFFFFFFFF in the sweep slot) and a length drawn from the
// species table (cumulative prevalence walk, as solid_solution does).
__global__ void init_random_kernel(double4 *lat, const RepDev *reps, int replica, int nspec,
                                   const double *len, const double *cum)
{
    const RepDev rep = reps[replica];
    const long long N = (long long)rep.X * rep.Y * rep.Z;
    long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= N) return;
    double px, py, pz, u;
    counter_draw(rep.seed, (uint32_t)replica, 0xFFFFFFFFu, (uint32_t)s, 0, px, py, pz, u);
    int k = 0;
    while (k + 1 < nspec && u >= cum[k]) k++;
    lat[rep.base + s] = make_double4(px, py, pz, len[k]);
}

// recombination_calculator's sums (src/starrynight-analysis.c:97-164) over a
// potential map: per workgroup partial sums of {exp(-b p), exp(b p),
// 1 / (exp(b p) + 1), 1 / (exp(-b p) + 1), their product}, p = scale * pot.
constexpr int kRecombParts = 5;

__global__ __launch_bounds__(256) void recombination_kernel(const double *pot, long long N, double scale,
                                                            double beta, double *partials)
{
    __shared__ double red[kRecombParts][256];
    const int tid = threadIdx.x;
    double v[kRecombParts] = {0, 0, 0, 0, 0};
    for (long long i = (long long)blockIdx.x * 256 + tid; i < N; i += (long long)gridDim.x * 256) {
        const double p = scale * pot[i];
        const double ep = exp(p * beta), em = exp(-p * beta);
        const double fe = 1.0 / (ep + 1.0), fh = 1.0 / (em + 1.0);
        v[0] += em; v[1] += ep; v[2] += fe; v[3] += fh; v[4] += fe * fh;
    }
    for (int c = 0; c < kRecombParts; c++) red[c][tid] = v[c];
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st)
            for (int c = 0; c < kRecombParts; c++) red[c][tid] += red[c][tid + st];
        __syncthreads();
    }
    if (tid < kRecombParts) partials[(long long)blockIdx.x * kRecombParts + tid] = red[tid][0];
}

}  // namespace sn
