// sn_stencil.h -- dipole_potential (src/starrynight-analysis.c:65-94) and
// dipole_electricfield (src/starrynight-analysis.c:393-457) at every site of a
// replica, FP64 (gfx950).
//
//   potential  sum over 0 < |r| <= 6 of L_j p_j . r / |r|^3
//   field      sum over 0 < |r| <= R of (3 n (n . p_j) - p_j) / |r|^3, then - p_i / 3
// j = i + r; the dz range runs even when Z == 1, where it wraps onto the plane.
//
// Both are, for each dz, a weighted sum over the disc of columns (dx, dy), and
// the weight knows only |dz|.  So a lane sums the disc around its own z once,
// for every |dz| into two registers (the part even and the part odd in dz;
// three of each for the field), with the columns (dx, dy) and (dx, -dy) folded
// first, and adds up the +-dz at the end from the lanes that own z + dz: a
// third of the products of the direct sum, no modulo, and 13 rows of 13 read
// where the direct sum reads 924 neighbours.  Rows of up to 64 sites are held
// whole, several to a wave if short; longer ones are cut into 64 lanes of
// which R at each end only give.
//
// A workgroup is 8 waves of rows at NX = 2 successive x (one for the widest
// fields, whose registers do not hold two): a plane is read from LDS once for
// both, and the next one loads meanwhile into the other half of LDS.
// 64^3: potential 28 us (399 us with 924 gathers a site), field of radius 4
// 34 us (125 us); half of it products, the rest waits on LDS and weights with
// two waves a SIMD (one x per workgroup, four waves: 30 and 31 us).
#pragma once
#include "sn_device.h"

namespace sn {

constexpr int kStencilThreads = 512;
constexpr int kPotentialR = 6;   // the reference's MAX in dipole_potential
constexpr int kFieldMaxR = 9;

// Sites of the largest staged plane: 8 waves of rows and R rows on either side.
__host__ __device__ constexpr int stencil_region(int R) { return kStencilThreads + 2 * R * 64; }
constexpr size_t stencil_lds(int R) { return 2 * 3 * (size_t)stencil_region(R) * sizeof(double); }
// Weights of (|dx|, |dy|): w = |r|^-3 for |dz| = 0..R, for the field then
// 3 w / |r|^2; 0 outside the ball, which has a row |dx| = R + 1 of zeros.
// They are read whole (a few wide scalar loads): a branch for each |dz| outside
// the ball saves a third of the products, but its loads then wait one by one
// (49 us against 28 us for the potential of a 64^3 lattice).
constexpr int stencil_row(int R, bool field) { return (field ? 2 : 1) * (R + 1); }
constexpr int stencil_weights(int R, bool field) { return (R + 2) * (R + 1) * stencil_row(R, field); }

struct StencilArgs {
    const double4 *lat;
    const RepDev *reps;
    const double *weights;
    double *out;
    int replica, ny, nz;     // workgroups along y and z
    int zl, rows, valid;     // sites of a row held by lanes, rows per wave, sites of a row per workgroup
};

// Sums of one site for |dz| = 0..R, parts even and odd in dz.
template <int R, bool FIELD>
struct StencilSum {
    static constexpr int C = FIELD ? 3 : 1;
    double even[C][R + 1], odd[C][R + 1];

    // s, d: sum and difference of the columns (dx, +dy) and (dx, -dy)
    __device__ __forceinline__ void add(const double *w, double dx, double dy, const double s[3], const double d[3])
    {
        const double along = dx * s[0] + dy * d[1];
        if constexpr (FIELD) {
            const double x = dx * along, y = dy * (dx * d[0] + dy * s[1]), xz = dx * s[2], yz = dy * d[2];
#pragma unroll
            for (int k = 0; k <= R; k++) {
                const double w1 = w[k], w3 = w[R + 1 + k];
                even[0][k] += w3 * x - w1 * s[0];
                even[1][k] += w3 * y - w1 * s[1];
                even[2][k] += w3 * ((double)(k * k) * s[2]) - w1 * s[2];
                odd[0][k] += w3 * xz;
                odd[1][k] += w3 * yz;
                odd[2][k] += w3 * along;
            }
        } else {
#pragma unroll
            for (int k = 0; k <= R; k++) {
                even[0][k] += w[k] * along;
                odd[0][k] += w[k] * s[2];
            }
        }
    }
};

template <int R, bool FIELD, int NX>
__global__ __launch_bounds__(kStencilThreads) void stencil_observable_kernel(StencilArgs sa)
{
    constexpr int M = stencil_region(R);
    constexpr int NL = (M + kStencilThreads - 1) / kStencilThreads;   // staged sites of a thread
    extern __shared__ double lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const RepDev &rep = sa.reps[sa.replica];
    const int X = rep.X, Y = rep.Y, Z = rep.Z, zl = sa.zl;
    const bool whole = Z <= 64;   // a row's lanes hold all of it
    const int block = (int)xcd_block(blockIdx.x, gridDim.x);
    const int z0 = block % sa.nz * sa.valid, q0 = block / sa.nz;
    const int y0 = q0 % sa.ny * (8 * sa.rows), x0 = q0 / sa.ny * NX;
    const int nrows = min(8 * sa.rows, Y - y0);
    const int sub = lane / zl, zi = lane - sub * zl;
    const int row = wave * sa.rows + sub;
    const bool own = sub < sa.rows && row < nrows;

    const int region = (nrows + 2 * R) * zl;
    int g[NL];   // site within its plane
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int e = min(tid + i * kStencilThreads, region - 1);
        const int ry = e / zl, rz = e - ry * zl;
        g[i] = wrap_any(y0 - R + ry, Y) * Z + wrap_any(whole ? rz : z0 - R + rz, Z);
    }
    const double4 *lat = sa.lat + rep.base;
    auto load = [&](int x, double4 v[NL]) __attribute__((always_inline)) {
        const double4 *plane = lat + (long long)wrap_any(x, X) * Y * Z;
#pragma unroll
        for (int i = 0; i < NL; i++) v[i] = plane[g[i]];
    };
    auto store = [&](double *s, const double4 v[NL]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int e = tid + i * kStencilThreads;
            if (e < region) {
                const double f = FIELD ? 1.0 : v[i].w;
                s[e] = f * v[i].x;
                s[e + M] = f * v[i].y;
                s[e + 2 * M] = f * v[i].z;
            }
        }
    };
    {
        double4 v[NL];
        load(x0 - R, v);
        store(lds, v);
    }
    __syncthreads();

    StencilSum<R, FIELD> S[NX] = {};
    const int at = ((own ? row : 0) + R) * zl + zi;
    constexpr int kPlanes = 2 * R + NX, kRow = stencil_row(R, FIELD);
    constexpr int kUnroll = R < 9 ? R + 1 : 1;   // the widest body exceeds what the compiler unrolls
#pragma unroll 1
    for (int i = 0; i < kPlanes; i++) {
        const bool next = i + 1 < kPlanes;
        double4 v[NL];
        if (next) load(x0 - R + i + 1, v);
        const double *p = lds + (i & 1) * 3 * M + at;
        const double *w[NX];
        int rest = -1;   // R^2 - dx^2 of the output nearer to the plane
        double dx[NX];
#pragma unroll
        for (int o = 0; o < NX; o++) {
            const int d = i - R - o;
            dx[o] = d;
            rest = max(rest, R * R - d * d);
            w[o] = sa.weights + abs(d) * ((R + 1) * kRow);
        }
#pragma unroll kUnroll
        for (int dy = 0; dy <= R; dy++) {
            if (dy * dy > rest) break;
            double wk[NX][kRow];
#pragma unroll
            for (int o = 0; o < NX; o++)
#pragma unroll
                for (int k = 0; k < kRow; k++) wk[o][k] = w[o][dy * kRow + k];
            double s[3], d[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double a = p[c * M + dy * zl], b = dy ? p[c * M - dy * zl] : 0.0;
                s[c] = a + b;
                d[c] = dy ? a - b : 0.0;
            }
#pragma unroll
            for (int o = 0; o < NX; o++) S[o].add(wk[o], dx[o], (double)dy, s, d);
        }
        if (next) store(lds + ((i + 1) & 1) * 3 * M, v);
        __syncthreads();
    }

    // sum over dz: the lane of z + dz holds its even and odd parts
    constexpr int C = StencilSum<R, FIELD>::C;
    int up = lane, down = lane, zu = zi, zd = zi;
    double e[NX][C];
#pragma unroll
    for (int o = 0; o < NX; o++)
#pragma unroll
        for (int c = 0; c < C; c++) e[o][c] = S[o].even[c][0];
#pragma unroll
    for (int k = 1; k <= R; k++) {
        up++; zu++; down--; zd--;
        if (whole && zu == zl) { zu = 0; up -= zl; }
        if (whole && zd < 0) { zd = zl - 1; down += zl; }
#pragma unroll
        for (int o = 0; o < NX; o++)
#pragma unroll
            for (int c = 0; c < C; c++) {
                const double ev = S[o].even[c][k], od = k * S[o].odd[c][k];
                e[o][c] += __shfl(ev + od, up & 63) + __shfl(ev - od, down & 63);
            }
    }
    const int z = whole ? zi : z0 - R + zi;
    if (!own || (!whole && (zi < R || zi >= 64 - R || z >= Z))) return;
#pragma unroll
    for (int o = 0; o < NX; o++) {
        if (x0 + o >= X) break;
        const long long s = ((long long)(x0 + o) * Y + (y0 + row)) * Z + z;
        if constexpr (FIELD) {
            const double4 a = lat[s];
            sa.out[3 * s] = e[o][0] - a.x / 3.0;
            sa.out[3 * s + 1] = e[o][1] - a.y / 3.0;
            sa.out[3 * s + 2] = e[o][2] - a.z / 3.0;
        } else {
            sa.out[s] = e[o][0];
        }
    }
}

// Rows of 64 lanes with R at each end only giving need R < 32; two x per
// workgroup hold 2 x 2 x C x (R + 1) sums, 168 registers at C = 3, R = 6.
constexpr int stencil_nx(int R, bool field) { return field && R > 6 ? 1 : 2; }

}  // namespace sn
