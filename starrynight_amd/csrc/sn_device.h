// sn_device.h -- device-side building blocks shared by the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sn {

// Per-replica parameters, resident in HBM so that sn_set_params reaches a
// captured graph without re-capture.
struct RepDev {
    int X, Y, Z, mixed;
    long long base;        // first site of this replica in the lattice buffer
    double beta, J, K, L0; // L0: the common dipole length when !mixed
    double E[3];
    unsigned long long seed;
    int constrain_to_x, pad;
};

// One tile of the schedule, with its replica's size and its own: the staging
// loads of a tile depend on this record alone, not on a chain of tables.
struct TileDev {
    int replica, x0, y0, z0, shape, X, Y, Z;
    long long base;        // first site of the replica in the lattice buffer
    int size;              // tx | ty << 10 | tz << 20
    int sites_off, first_chunks;   // the shape's site list; sites of its first two proposal chunks, n0 | n1 << 16
    int gstep_off, gsteps_n, nchunks;   // the shape's step table, its steps and proposal chunks
};
static_assert(sizeof(TileDev) == 64, "one scalar load");

struct ShapeDev {
    int tx, ty, tz, ncol;
    int nsteps, step_off;     // field kernel's step table (see sn_sweep_field.h)
    int typ, tzp, coord_off;  // field kernel's padded tile-order strides and coordinate table
};

// z stride of the gather kernel's staged region.  A row of a multiple of 8
// sites (16 for 8-site tiles at DipoleCutOff 4) is padded by one: with a
// stride of 16 doubles every neighbour at the same dz lands in the same LDS
// bank, whatever its dx and dy.
__host__ __device__ inline int gather_zstride(int rz) { return (rz > 1 && rz % 8 == 0) ? rz + 1 : rz; }

// One +-r neighbour pair (sweep kernel) or one offset (gather kernels).
struct PairDev {
    int dx, dy, dz, nn;
    double nx, ny, nz, w;  // unit vector r/|r| and 1/|r|^3
};

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11).  Each round's two
// 32 x 32 -> 64-bit products are formed as 64-bit multiplies (one
// v_mad_u64_u32 each) rather than separate high and low multiplies.
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0], p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// The disc coordinate of a Philox word: x = a 2^-26, a odd, |a| < 2^26.
__device__ __forceinline__ double disc_coordinate(uint32_t word)
{
    return (double)((int)((word >> 5) | 1u) - (1 << 26)) * (1.0 / 67108864.0);
}

// |x|^2 of a candidate: the squares have at most 52 bits and their sum fits in
// 53, so nothing rounds.
__device__ __forceinline__ double disc_norm2(double x1, double x2) { return fma(x1, x1, x2 * x2); }

// sqrt of x in [2^-52, 1], correctly rounded: Goldschmidt iterations from the
// hardware's reciprocal root and two residual corrections (Markstein).  The
// library's sqrt spends as much again on scaling denormals and on zero and
// infinity, none of which occur here.
__device__ __forceinline__ double sqrt_unit(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    return fma(fma(-g, g, x), h, g);
}

// ln u of u = j 2^-53, 0 < j < 2^53: u = 2^k m with m in [sqrt(1/2), sqrt 2),
// ln m = 2 atanh(t), t = (m - 1) / (m + 1) carried in two doubles (m - 1 is
// exact), atanh by its Taylor series (t^2 < 0.0295: eleven terms reach 2^-56),
// k ln 2 in two doubles.  At most 0.59 ulp off: the last rounding, 0.03 for
// t's low part entering the series in its first term only, and eight roundings
// of the small terms of at most 0.007 each (0.57 over 20 million arguments
// against an extended-precision log).  About 50 instructions against the
// library's 118, most of them a dependent chain that a wave waits for.
__device__ __forceinline__ double log_unit(double u)
{
    double m = __builtin_amdgcn_frexp_mant(u);   // [1/2, 1)
    int k = __builtin_amdgcn_frexp_exp(u);
    const bool low = m < 0.70710678118654752440;
    m = low ? 2.0 * m : m;
    k -= low ? 1 : 0;
    const double f = m - 1.0, d = m + 1.0, de = (1.0 - d) + m;   // d + de = m + 1
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    const double t = f * r, tl = fma(-de, t, fma(-d, t, f)) * r;   // t + tl = f / (m + 1)
    const double z = t * t, z2 = z * z, z4 = z2 * z2;
    const double a = fma(z2, fma(z, 1.0 / 9, 1.0 / 7), fma(z, 1.0 / 5, 1.0 / 3));
    const double b = fma(z4, fma(z, 1.0 / 21, 1.0 / 19),
                         fma(z2, fma(z, 1.0 / 17, 1.0 / 15), fma(z, 1.0 / 13, 1.0 / 11)));
    const double lo = fma(t * z, fma(z4, b, a), tl);
    const double kd = (double)k, h2 = 2.0 * t;
    const double kh = kd * 0x1.62e42fefa3800p-1;   // exact: the constant's low 11 bits are zero
    const double h = kh + h2;
    const double e = k != 0 ? (kh - h) + h2 : 0.0;   // (|kh| > |h2|)
    return h + (e + fma(kd, 0x1.ef35793c76730p-45, 2.0 * lo));
}

// Proposal and acceptance uniform for one visit of `site` in `sweep`:
// counter (site, sweep, replica, k), key = seed.  u = 53-bit uniform from words
// 2, 3 of k = 0; Marsaglia (1972) disc point from words 0, 1 of k = 0, then
// words 0, 1 and 2, 3 of k = 1, 2, ... (two candidates per retry call: a
// wave waits for its slowest lane, so fewer calls per rejection shorten every
// draw), with x = a 2^-26, a odd: the disc test and 1 - s, 1 - 2 s are exact,
// so only one sqrt and two products round.  The retry loop only finds the
// accepted words (the point's arithmetic, inlined at each test, ran up to
// four times per wave).
// N sites per lane: their chains of dependent multiplies and roots interleave,
// and a retry call serves whichever site of a lane still needs one.
template <int N>
__device__ __forceinline__ void counter_draws(unsigned long long seed, uint32_t replica, uint32_t sweep,
                                              const uint32_t (&site)[N], int constrain_to_x, double (&px)[N],
                                              double (&py)[N], double (&pz)[N], double (&u)[N])
{
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    double x1[N], x2[N], S[N];
    uint32_t w0[N];
#pragma unroll
    for (int n = 0; n < N; n++) {
        uint32_t w[4] = {site[n], sweep, replica, 0u};
        philox4x32_10(w, k0, k1);
        u[n] = ((double)(w[2] >> 5) * 67108864.0 + (double)(w[3] >> 6)) * (1.0 / 9007199254740992.0);
        x1[n] = disc_coordinate(w[0]);
        x2[n] = disc_coordinate(w[1]);
        S[n] = disc_norm2(x1[n], x2[n]);
        w0[n] = w[0];
    }
    if (constrain_to_x) {
#pragma unroll
        for (int n = 0; n < N; n++) {
            const uint32_t i = w0[n] % 6u;
            px[n] = (i == 0) ? 1.0 : (i == 1) ? -1.0 : 0.0;
            py[n] = (i == 2) ? 1.0 : (i == 3) ? -1.0 : 0.0;
            pz[n] = (i == 4) ? 1.0 : (i == 5) ? -1.0 : 0.0;
        }
        return;
    }
    // (a lane's sites retry in order: site 0 until it has its point, then 1)
    uint32_t k = 1;
    for (;;) {
        const bool two = N > 1 && S[0] < 1.0;   // site 0 is done
        const double s = two ? S[N - 1] : S[0];
        if (!(s >= 1.0)) break;
        uint32_t c[4] = {two ? site[N - 1] : site[0], sweep, replica, k};
        philox4x32_10(c, k0, k1);
        double y1 = disc_coordinate(c[0]), y2 = disc_coordinate(c[1]), T = disc_norm2(y1, y2);
        const double v1 = disc_coordinate(c[2]), v2 = disc_coordinate(c[3]), V = disc_norm2(v1, v2);
        if (T >= 1.0) { y1 = v1; y2 = v2; T = V; }
        if (T >= 1.0 && k == 32) { y1 = 0.0; y2 = 0.0; T = 0.0; }   // 65 rejections in a row (p ~ 1e-43): (0, 0, 1)
        k = T >= 1.0 ? k + 1 : 1;
        if (two) { x1[N - 1] = y1; x2[N - 1] = y2; S[N - 1] = T; }
        else { x1[0] = y1; x2[0] = y2; S[0] = T; }
    }
#pragma unroll
    for (int n = 0; n < N; n++) {
        const double r = sqrt_unit(1.0 - S[n]);
        px[n] = (2.0 * x1[n]) * r;
        py[n] = (2.0 * x2[n]) * r;
        pz[n] = 1.0 - 2.0 * S[n];
    }
}

__device__ __forceinline__ void counter_draw(unsigned long long seed, uint32_t replica, uint32_t sweep, uint32_t site,
                                             int constrain_to_x, double &px, double &py, double &pz, double &u)
{
    const uint32_t sites[1] = {site};
    double x[1], y[1], z[1], v[1];
    counter_draws<1>(seed, replica, sweep, sites, constrain_to_x, x, y, z, v);
    px = x[0]; py = y[0]; pz = z[0]; u = v[0];
}

// Metropolis threshold: exp(-beta dE) > u  <=>  dE < -ln(u)/beta, and the
// dE < 0 branch of src/starrynight-montecarlo-core.c:179 is covered because
// the threshold is >= 0.  beta = +inf (T = 0) gives 0: only dE < 0 accepted.
// rbeta = 1 / beta, rounded: the quotient is its product corrected by its own
// residual, which is the correctly rounded quotient (Markstein 1990) while
// nothing over- or underflows; a beta that could is divided by.
__device__ __forceinline__ double metropolis_threshold(double u, double beta, double rbeta)
{
    if (u <= 0.0 || beta <= 0.0) return __builtin_inf();
    if (__builtin_isinf(beta)) return 0.0;
    const double l = -log_unit(u);
    if (!(beta > 1e-200 && beta < 1e200)) return l / beta;
    const double q = l * rbeta;
    return fma(fma(-q, beta, l), rbeta, q);
}

__device__ __forceinline__ int wrap_once(int v, int L)
{
    v += (v < 0) ? L : 0;
    v -= (v >= L) ? L : 0;
    return v;
}

__device__ __forceinline__ int wrap_any(int v, int L)
{
    const int m = v % L;
    return m < 0 ? m + L : m;
}

// Consecutive workgroups go to the eight XCDs in turn; this numbering gives
// each XCD (each L2) a contiguous eighth of the work instead.
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned n)
{
    const unsigned xcd = b % 8, each = n / 8, rest = n % 8;
    return xcd * each + min(xcd, rest) + b / 8;
}

}  // namespace sn
