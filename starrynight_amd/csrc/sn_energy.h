// sn_energy.h -- energy and adjoint of whole lattices (gfx950, FP64).
//
// The Hamiltonian whose single-site differences are the reference's
// site_energy (src/starrynight-montecarlo-core.c:91-134):
//   E = 1/2 sum_i L_i p_i . h_i - J/2 sum_i p_i . g_i + sum_i p_i . E - [K>0] K sum_i (|p_ix| + |p_iy|)
// with h_i = sum_r L_j (p_j - 3 n (n . p_j)) / d^3 and g_i = sum_{|r|=1} p_j.
// The adjoint is dE/dp_i = L_i h_i - J g_i + E - [K>0] K (sgn p_ix, sgn p_iy, 0)
// (the local field is its negative), and
//   dE/dJ = -1/2 sum p.g,  dE/dE = sum p,  dE/ds = 2 E_dd (lengths scaled by s),
//   dE/dK = -sum (|p_x| + |p_y|)  (K > 0).
//
// The tensor of r = (dx, dy, dz) is even or odd in dz, so for each |dz| a lane
// sums the disc of columns (dx, dy) around its own z once, into an even and an
// odd part, and the sites at z +- |dz| take them at the end through LDS: a
// third of the products of the sum over pairs.  The columns (dx, dy) and (dx,
// -dy) are folded as they are read; constants are folded at compile time.
// A workgroup owns rows * zl sites of a plane (zl: the whole row, or a cut of
// it with RC sites of halo at both ends) and walks along x in steps of NX: it
// takes the 2 RC + NX planes of a step through two halves of LDS, two more
// planes on their way from memory meanwhile; a plane is read once for all NX.
// 32 replicas of 48^3, cut-off 3: 136 us (245 us with the sum over pairs on
// staged 8^3 tiles), 48^3 with mixed lengths 14 us (18.5 us).  The products
// take 40 % of it; two waves a SIMD in step with a barrier a plane do not hide
// the LDS reads behind them (three x a step spill: 161 us; 256 threads, two
// workgroups a CU but more halo: 146 us; one plane ahead: 171 us).
// Per-workgroup partial sums of the energy parts and parameter derivatives go
// to `partials` (kEnergyParts per workgroup, reduced afterwards).
#pragma once
#include "sn_sweep_field.h"

namespace sn {

constexpr int kEnergyParts = 10;   // {E_dd, E_cage, E_field, E_K, dJ, dEx, dEy, dEz, ds, dK}
constexpr int kEnergyThreads = 512;
constexpr int kEnergyRegion = 2 * kEnergyThreads;   // largest staged plane: two sites a thread

// x of a step where the lattices fill the chip: their sums (6 RC + 6 doubles
// each) have to stay in registers.
constexpr int energy_wide(int rc, bool two_d) { return two_d || rc <= 2 ? 4 : 2; }

// One workgroup: rows y0.. (nrows of them) and sites z0.. of replica, x0..x0+nx-1
// (in steps of the kernel's NX).
struct EnergyBlock {
    int replica, x0, nx, y0, nrows, z0, zl, pad;
};

struct EnergyArgs {
    const double4 *lat;
    const RepDev *reps;
    const EnergyBlock *blocks;   // the launch's workgroups, grouped by replica
    double *grad;                // 3 per site (row rep.base - grad_origin + site) or null
    long long grad_origin;       // lattice row of grad's first row
    double *partials;            // kEnergyParts per workgroup
};

constexpr size_t energy_lds(bool two_d, bool mixed)
{
    const size_t stage = (size_t)2 * (mixed ? 6 : 3) * kEnergyRegion, exchange = two_d ? 0 : 2 * 6 * kEnergyThreads;
    return (stage > exchange ? stage : exchange) * sizeof(double);
}

// Disc sums of one site for |dz| = 0..HZ (h without the central column's dz = 0).
template <int RC, int HZ>
struct DiscSum {
    double even[3][HZ + 1], odd[3][HZ + 1], g[3];

    // Plane boundary: the sums are formed before the next plane is read.  The
    // scheduler otherwise runs the chains last and spills what they wait for.
    __device__ __forceinline__ void fence()
    {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            asm volatile("" : "+v"(g[c]));
#pragma unroll
            for (int k = 0; k <= HZ; k++) {
                asm volatile("" : "+v"(even[c][k]));
                if (k > 0) asm volatile("" : "+v"(odd[c][k]));
            }
        }
    }

    // columns (DX, +DY) and (DX, -DY): s their sum, d their difference
    template <int DX, int DY>
    __device__ __forceinline__ void add(const double s[3], const double d[3])
    {
        constexpr int H = cisqrt(RC * RC - DX * DX - DY * DY), K = H < HZ ? H : HZ;
        double along = 0.0;
        if constexpr (DX != 0) along = DX * s[0];
        if constexpr (DY != 0) along = DX != 0 ? fma((double)DY, d[1], along) : DY * d[1];
        static_for<(DX == 0 && DY == 0) ? 1 : 0, K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value, r2 = DX * DX + DY * DY + k * k;
            constexpr double r = csqrt((double)r2), w = 1.0 / (r * r * r), w3 = 3.0 * w / r2;
            even[0][k] = fma(w - w3 * (DX * DX), s[0], even[0][k]);
            even[1][k] = fma(w - w3 * (DY * DY), s[1], even[1][k]);
            even[2][k] = fma(w - w3 * (k * k), s[2], even[2][k]);
            if constexpr (DX != 0 && DY != 0) {
                const double xy = -w3 * (DX * DY);
                even[0][k] = fma(xy, d[1], even[0][k]);
                even[1][k] = fma(xy, d[0], even[1][k]);
            }
            if constexpr (k > 0) {
                if constexpr (DX != 0) odd[0][k] = fma(-w3 * (k * DX), s[2], odd[0][k]);
                if constexpr (DY != 0) odd[1][k] = fma(-w3 * (k * DY), d[2], odd[1][k]);
                if constexpr (DX != 0 || DY != 0) odd[2][k] = fma(-w3 * k, along, odd[2][k]);
            }
        });
    }
};

template <int RC, bool TWO_D, bool MIXED, int NX>
__global__ __launch_bounds__(kEnergyThreads) void energy_kernel(EnergyArgs ea)
{
    constexpr int HZ = TWO_D ? 0 : RC;
    constexpr int T = kEnergyThreads;
    constexpr int NL = kEnergyRegion / T;   // staged sites of a thread
    extern __shared__ double smem[];
    __shared__ double red[kEnergyParts][T / 64];
    const int tid = threadIdx.x;
    const int block = (int)xcd_block(blockIdx.x, gridDim.x);
    const EnergyBlock b = ea.blocks[block];
    const RepDev rep = ea.reps[b.replica];
    constexpr int M = kEnergyRegion;   // component stride: an immediate of the LDS instructions
    const int Z = rep.Z, zl = b.zl;
    const bool whole = TWO_D || zl == Z;
    const double4 *lat = ea.lat + rep.base;

    const int region = (b.nrows + 2 * RC) * zl;
    int at_plane[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int e = min(tid + i * T, region - 1);
        const int ry = e / zl, rz = e - ry * zl;
        at_plane[i] = wrap_once(b.y0 - RC + ry, rep.Y) * Z + (whole ? rz : wrap_once(b.z0 - HZ + rz, Z));
    }
    // x and y of a site share a 16-byte slot (one LDS instruction), z is apart
    auto put = [&](double *s, int e, double x, double y, double z) __attribute__((always_inline)) {
        ((double2 *)s)[e] = make_double2(x, y);
        s[2 * M + e] = z;
    };
    auto get = [&](const double *s, int e, double q[3]) __attribute__((always_inline)) {
        const double2 xy = ((const double2 *)s)[e];
        q[0] = xy.x; q[1] = xy.y; q[2] = s[2 * M + e];
    };
    // a half holds L p (p where lengths are uniform) and, for mixed lengths, p
    constexpr int kParts = MIXED ? 6 : 3;
    double4 v[2][NL];   // planes on their way, by parity
    auto load = [&](int x0, auto ic) __attribute__((always_inline)) {
        constexpr int I = decltype(ic)::value;
        // (twice: the last step of a short axis reaches beyond its second copy)
        const double4 *plane = lat + (long long)wrap_once(wrap_once(x0 - RC + I, rep.X), rep.X) * rep.Y * Z;
#pragma unroll
        for (int j = 0; j < NL; j++) v[I & 1][j] = plane[at_plane[j]];
    };
    auto store = [&](auto ic) __attribute__((always_inline)) {
        constexpr int I = decltype(ic)::value;
        double *s = smem + (I & 1) * kParts * M;
#pragma unroll
        for (int j = 0; j < NL; j++) {
            const int e = tid + j * T;
            const double4 &p = v[I & 1][j];
            const double f = MIXED ? p.w : 1.0;
            put(s, e, f * p.x, f * p.y, f * p.z);
            if (MIXED) put(s + 3 * M, e, p.x, p.y, p.z);
        }
    };

    const int row_of = tid / zl, zi = tid - row_of * zl;
    const bool mine = row_of < b.nrows && (whole || (zi >= HZ && zi < zl - HZ && b.z0 - HZ + zi < Z));
    const int row = row_of < b.nrows ? row_of : 0;
    const int at = (row + RC) * zl + zi;
    const int above = whole && zi + 1 == zl ? 1 - zl : 1, below = whole && zi == 0 ? zl - 1 : -1;

    const double J = rep.J, K = rep.K;
    const double Lh = MIXED ? 1.0 : rep.L0;   // h without the L_j factor when lengths are uniform
    double part[kEnergyParts];
#pragma unroll
    for (int c = 0; c < kEnergyParts; c++) part[c] = 0.0;
    const long long plane_sites = (long long)rep.Y * Z;
    const long long own = ((long long)b.y0 + row) * Z + (whole ? zi : b.z0 - HZ + zi);
    constexpr int P = 2 * RC + NX;   // planes of a step
    load(b.x0, std::integral_constant<int, 0>());
    load(b.x0, std::integral_constant<int, 1>());
    for (int x0 = b.x0; x0 < b.x0 + b.nx; x0 += NX) {
        // the next step's first planes load behind this one's last (after the
        // last step these again, unused: no branch between the planes)
        const bool more = x0 + NX < b.x0 + b.nx;
        const int x_next = more ? x0 + NX : x0;
        DiscSum<RC, HZ> S[NX];
#pragma unroll
        for (int o = 0; o < NX; o++) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                S[o].g[c] = 0.0;
#pragma unroll
                for (int k = 0; k <= HZ; k++) S[o].even[c][k] = S[o].odd[c][k] = 0.0;
            }
        }
        static_for<0, P - 1>([&](auto ic) __attribute__((always_inline)) {
            constexpr int I = decltype(ic)::value;
            store(ic);
            if constexpr (I + 2 < P) load(x0, std::integral_constant<int, I + 2>());
            else load(x_next, std::integral_constant<int, I & 1>());
            __syncthreads();
            const double *sm = smem + (I & 1) * kParts * M, *sp = MIXED ? sm + 3 * M : sm;
            static_for<0, RC>([&](auto yc) __attribute__((always_inline)) {
                constexpr int DY = decltype(yc)::value;
                // some output has (dx, DY) in its disc: the nearest dx decides
                constexpr int near = I < RC ? RC - I : I > RC + NX - 1 ? I - RC - NX + 1 : 0;
                if constexpr (near * near + DY * DY <= RC * RC) {
                    double s[3], d[3] = {0.0, 0.0, 0.0}, gs[3], q[3];
                    get(sm, at + DY * zl, s);
                    if constexpr (DY > 0) {
                        get(sm, at - DY * zl, q);
#pragma unroll
                        for (int c = 0; c < 3; c++) { d[c] = s[c] - q[c]; s[c] += q[c]; }
                    }
#pragma unroll
                    for (int c = 0; c < 3; c++) gs[c] = s[c];
                    if constexpr (MIXED && DY <= 1) {
                        get(sp, at + DY * zl, gs);
                        if constexpr (DY == 1) {
                            get(sp, at - DY * zl, q);
#pragma unroll
                            for (int c = 0; c < 3; c++) gs[c] += q[c];
                        }
                    }
                    static_for<0, NX - 1>([&](auto oc) __attribute__((always_inline)) {
                        constexpr int O = decltype(oc)::value, DX = I - RC - O;
                        if constexpr (DX * DX + DY * DY <= RC * RC) S[O].template add<DX, DY>(s, d);
                        if constexpr (DX * DX + DY * DY == 1) {
#pragma unroll
                            for (int c = 0; c < 3; c++) S[O].g[c] += gs[c];
                        }
                        if constexpr (!TWO_D && DX == 0 && DY == 0) {
                            double u[3];
                            get(sp, at + above, u);
                            get(sp, at + below, q);
#pragma unroll
                            for (int c = 0; c < 3; c++) S[O].g[c] += u[c] + q[c];
                        }
                    });
                }
            });
#pragma unroll
            for (int o = 0; o < NX; o++) S[o].fence();
        });

        // ---- h of every site, gradient and sums ----
        double4 p[NX];
#pragma unroll
        for (int o = 0; o < NX; o++)   // (an x beyond the lattice's last reads a site, uses nothing)
            p[o] = lat[min(x0 + o, rep.X - 1) * plane_sites + (mine ? own : 0)];
        if (!TWO_D) __syncthreads();   // the exchange reuses the planes' LDS
        int half = 0;                  // by halves, one barrier each
#pragma unroll
        for (int o = 0; o < NX; o++) {
            double h[3];
#pragma unroll
            for (int c = 0; c < 3; c++) h[c] = S[o].even[c][0];
            if constexpr (!TWO_D) {
                int up = zi, down = zi;
#pragma unroll
                for (int k = 1; k <= HZ; k++) {
                    // parts for the sites below and above by k
                    double2 *xy = (double2 *)(smem + half * 6 * T);
                    double *zz = (double *)(xy + 2 * T);
                    half ^= 1;
                    double dn[3], upw[3];
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        dn[c] = S[o].even[c][k] + S[o].odd[c][k];
                        upw[c] = S[o].even[c][k] - S[o].odd[c][k];
                    }
                    xy[tid] = make_double2(dn[0], dn[1]);
                    xy[T + tid] = make_double2(upw[0], upw[1]);
                    zz[tid] = dn[2];
                    zz[T + tid] = upw[2];
                    __syncthreads();
                    up = whole && up + 1 == zl ? 0 : up + 1;
                    down = whole && down == 0 ? zl - 1 : down - 1;
                    const int from_above = min(tid + (up - zi), T - 1), from_below = min(max(tid + (down - zi), 0), T - 1);
                    const double2 p0 = xy[from_above], p1 = xy[T + from_below];
                    h[0] += p0.x + p1.x;
                    h[1] += p0.y + p1.y;
                    h[2] += zz[from_above] + zz[T + from_below];
                }
            }
            if (mine && x0 + o < b.x0 + b.nx) {
                const double hx = Lh * h[0], hy = Lh * h[1], hz = Lh * h[2];
                const double *g = S[o].g;
                const double Li = MIXED ? p[o].w : rep.L0;
                const double ph = p[o].x * hx + p[o].y * hy + p[o].z * hz;
                const double pg = p[o].x * g[0] + p[o].y * g[1] + p[o].z * g[2];
                double gx = Li * hx - J * g[0] + rep.E[0];
                double gy = Li * hy - J * g[1] + rep.E[1];
                const double gz = Li * hz - J * g[2] + rep.E[2];
                const double ak = fabs(p[o].x) + fabs(p[o].y);
                if (K > 0.0) {
                    gx -= K * ((p[o].x > 0.0) - (p[o].x < 0.0));
                    gy -= K * ((p[o].y > 0.0) - (p[o].y < 0.0));
                }
                if (ea.grad) {
                    double *out = ea.grad + 3 * (rep.base - ea.grad_origin + (x0 + o) * plane_sites + own);
                    out[0] = gx; out[1] = gy; out[2] = gz;
                }
                part[0] += 0.5 * Li * ph;
                part[1] += -0.5 * J * pg;
                part[2] += p[o].x * rep.E[0] + p[o].y * rep.E[1] + p[o].z * rep.E[2];
                part[3] += K > 0.0 ? -K * ak : 0.0;
                part[4] += -0.5 * pg;
                part[5] += p[o].x; part[6] += p[o].y; part[7] += p[o].z;
                part[8] += Li * ph;
                part[9] += K > 0.0 ? -ak : 0.0;
            }
        }
        if (more) __syncthreads();   // the next planes go where this was read
    }

    // ---- workgroup partial sums: wave shuffles, then the waves through LDS ----
#pragma unroll
    for (int c = 0; c < kEnergyParts; c++) {
        double x = part[c];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
        if ((tid & 63) == 0) red[c][tid >> 6] = x;
    }
    __syncthreads();
    if (tid < kEnergyParts) {
        double x = 0.0;
        for (int w = 0; w < T / 64; w++) x += red[tid][w];
        ea.partials[(long long)block * kEnergyParts + tid] = x;
    }
}

}  // namespace sn
