// sn_radial.h -- radial_order_parameter (src/starrynight-analysis.c:528-598) in FP64 (gfx950).
//
// Over every site i and every offset r with |r|^2 <= 80 (the dz range runs
// even when Z == 1, where it wraps onto the same plane, as in the reference):
//   FE[r^2]  += p_i.p_j,   AFE[r^2] += p_i.p_j - 3 (n.p_i)(n.p_j),  j = i + r
// with n = r/|r| (n = 0 at r = 0).
//
// A lane owns an offset column (dx, dy), not a site: +r and -r sum the same
// pairs, so half the plane's 249 columns are left, 125 of them, two waves.
// With u along (dx, dy) and v across it in the plane a column needs, for each
// |dz| = 0..8, only the sums over sites of u u', v v', z z' and +-(u z' + z u'):
// 5 FMAs a pair, held in registers from the first site to the last, and
// nothing is reduced before the end.  Walking along z the lane keeps its
// column's window z-8..z+8 in registers, one new site a step.  Columns are
// sorted by dx^2 + dy^2: the far half (>= 40) needs |dz| <= 6 only.
//
// A workgroup takes 4 y rows x up to 16 z (8 waves: a near and a far one per
// row, which share a SIMD) and walks a range of x, over a ring of ten planes
// in LDS: 20 x 32 sites each, the tenth loading while the nine of dx = 0..8
// are read.  The pair sums bound it: 64^3 takes 144 us (1593 us with a site per
// lane, 3071 gathers with three modulos each and 162 wave reductions).
#pragma once
#include <utility>
#include "sn_device.h"

namespace sn {

constexpr int kRadialBins = 81;
constexpr int kRadialH = 8;        // largest |dx|, |dy|, |dz|
constexpr int kRadialFar = 6;      // largest |dz| of the far columns
constexpr int kRadialCols = 128;   // 125 columns, near half first, padded with (0, 0)
constexpr int kRadialTY = 4, kRadialTZ = 16;
constexpr int kRadialThreads = 2 * 64 * kRadialTY;
constexpr int kRadialRegionY = kRadialTY + 2 * kRadialH, kRadialRegionZ = kRadialTZ + 2 * kRadialH;
// Row and plane strides spread a wave's 64 columns over the banks: 4.8 lanes
// on the fullest one on average, against 9 for unpadded planes.
constexpr int kRadialRow = kRadialRegionZ + 1, kRadialPlane = 680;
constexpr int kRadialSlots = kRadialH + 2;
constexpr int kRadialComponent = kRadialSlots * kRadialPlane;
constexpr int kRadialLds = 3 * kRadialComponent * (int)sizeof(double);
constexpr int kRadialSums = (kRadialH + 1) * kRadialCols;   // (|dz|, column)
static_assert(kRadialPlane >= kRadialRegionY * kRadialRow, "a plane's rows overlap the next plane");
static_assert(kRadialLds <= 160 * 1024, "ring of planes exceeds LDS");
static_assert(kRadialTY * kRadialSums * 2 * (int)sizeof(double) <= kRadialLds, "row sums exceed LDS");

struct RadialCol {
    double cx, cy;   // unit vector along (dx, dy); (1, 0) for the column of the site itself
    int dx, dy;
};

struct RadialArgs {
    const double4 *lat;
    const RepDev *reps;
    const RadialCol *cols;
    const unsigned short *entries;   // |dz| * kRadialCols + column, grouped by r^2
    const int *bin_start;            // kRadialBins + 1
    double *partials;                // 2 * kRadialBins per workgroup
    int replica, ny, nz, tz, cx;     // workgroups along y and z, sites along z and x of a workgroup
};

// Sums of a lane's column, index |dz|.
struct RadialSum {
    double uu[kRadialH + 1], vv[kRadialH + 1], zz[kRadialH + 1], uz[kRadialH + 1];
};

template <class Step, int... T>
__device__ __forceinline__ void radial_steps(Step &step, int n, std::integer_sequence<int, T...>)
{
    ((T < n ? step(std::integral_constant<int, T>()) : void()), ...);
}

// One row of n sites along z.  a: the row's first site; q: the column's site
// at dz = -DZ of it.  A step's loads are issued a step ahead.
template <int DZ>
__device__ __forceinline__ void radial_row(const double *a, const double *q, int n, double cx, double cy,
                                           RadialSum &S)
{
    constexpr int W = 2 * DZ + 1;
    double u[W], v[W], z[W];
#pragma unroll
    for (int i = 0; i < 2 * DZ; i++) {
        const double x = q[i], y = q[i + kRadialComponent];
        u[i] = cx * x + cy * y;
        v[i] = cx * y - cy * x;
        z[i] = q[i + 2 * kRadialComponent];
    }
    double qx = q[2 * DZ], qy = q[2 * DZ + kRadialComponent], qz = q[2 * DZ + 2 * kRadialComponent];
    double ax = a[0], ay = a[kRadialComponent], az = a[2 * kRadialComponent];
    // the window rotates through the registers: a step is compiled for each t
    auto step = [&](auto T) __attribute__((always_inline)) {
        constexpr int t = decltype(T)::value, C = kRadialComponent;
        constexpr int top = (t + 2 * DZ) % W, mid = (t + DZ) % W;
        u[top] = cx * qx + cy * qy;
        v[top] = cx * qy - cy * qx;
        z[top] = qz;
        const double ua = cx * ax + cy * ay, va = cx * ay - cy * ax, za = az;
        if (t + 1 < kRadialTZ) {
            qx = q[t + 1 + 2 * DZ]; qy = q[t + 1 + 2 * DZ + C]; qz = q[t + 1 + 2 * DZ + 2 * C];
            ax = a[t + 1]; ay = a[t + 1 + C]; az = a[t + 1 + 2 * C];
        }
        S.uu[0] += ua * u[mid];
        S.vv[0] += va * v[mid];
        S.zz[0] += za * z[mid];
#pragma unroll
        for (int k = 1; k <= DZ; k++) {
            const int p = (t + DZ + k) % W, m = (t + DZ - k) % W;
            S.uu[k] += ua * u[p];
            S.vv[k] += va * v[p];
            S.zz[k] += za * z[p];
            S.uz[k] += ua * z[p];
            S.uu[k] += ua * u[m];
            S.vv[k] += va * v[m];
            S.zz[k] += za * z[m];
            S.uz[k] -= ua * z[m];
            S.uz[k] += za * u[p];
            S.uz[k] -= za * u[m];
        }
    };
    radial_steps(step, n, std::make_integer_sequence<int, kRadialTZ>());
}

__global__ __launch_bounds__(kRadialThreads) void radial_order_kernel(RadialArgs ra)
{
    extern __shared__ double lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = wave % kRadialTY;
    const bool far = wave >= kRadialTY;
    const RepDev &rep = ra.reps[ra.replica];
    const int X = rep.X, Y = rep.Y, Z = rep.Z;
    const int block = (int)xcd_block(blockIdx.x, gridDim.x);
    const int z0 = block % ra.nz * ra.tz, q0 = block / ra.nz;
    const int y0 = q0 % ra.ny * kRadialTY, x0 = q0 / ra.ny * ra.cx;
    const int n = min(ra.tz, Z - z0);
    const int x1 = min(x0 + ra.cx, X);
    const RadialCol col = ra.cols[(far ? 64 : 0) + lane];

    // a plane is 640 sites: one per thread, and a second for the first 128
    constexpr int kPlaneSites = kRadialRegionY * kRadialRegionZ, kRest = kPlaneSites - kRadialThreads;
    static_assert(kRest > 0 && kRest <= kRadialThreads, "two sites of a plane per thread");
    const int py[2] = {tid / kRadialRegionZ, (tid + kRadialThreads) / kRadialRegionZ};
    const int pz = tid % kRadialRegionZ;
    const bool second = tid < kRest;
    const int gz = wrap_any(z0 - kRadialH + pz, Z);
    const double4 *lat = ra.lat + rep.base + gz;
    const long long g[2] = {(long long)wrap_any(y0 - kRadialH + py[0], Y) * Z,
                            (long long)wrap_any(y0 - kRadialH + (second ? py[1] : 0), Y) * Z};
    const int d[2] = {py[0] * kRadialRow + pz, py[1] * kRadialRow + pz};
    auto load = [&](int x, double4 v[2]) __attribute__((always_inline)) {
        const double4 *plane = lat + (long long)(x % X) * Y * Z;
        v[0] = plane[g[0]];
        v[1] = plane[g[1]];
    };
    auto store = [&](int slot, const double4 v[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (k == 0 || second) {
                double *s = lds + slot * kRadialPlane + d[k];
                s[0] = v[k].x;
                s[kRadialComponent] = v[k].y;
                s[2 * kRadialComponent] = v[k].z;
            }
    };
    static_assert((kRadialH + 1) % 3 == 0, "planes staged three at a time");
    for (int p = 0; p <= kRadialH; p += 3) {
        double4 v[3][2];
#pragma unroll
        for (int k = 0; k < 3; k++) load(x0 + p + k, v[k]);
#pragma unroll
        for (int k = 0; k < 3; k++) store(p + k, v[k]);
    }
    __syncthreads();

    RadialSum S = {};
    const bool work = y0 + row < Y;
    const int own = (kRadialH + row) * kRadialRow + kRadialH;
    const int other = own + col.dy * kRadialRow - (far ? kRadialFar : kRadialH);
    int s_own = 0, s_other = col.dx, s_new = kRadialH + 1;
    for (int x = x0; x < x1; x++) {
        const bool next = x + 1 < x1;
        double4 v[2];
        if (next) load(x + kRadialH + 1, v);
        if (work) {
            const double *a = lds + s_own * kRadialPlane + own, *q = lds + s_other * kRadialPlane + other;
            if (far) radial_row<kRadialFar>(a, q, n, col.cx, col.cy, S);
            else radial_row<kRadialH>(a, q, n, col.cx, col.cy, S);
        }
        if (next) store(s_new, v);
        __syncthreads();
        s_own = s_own + 1 == kRadialSlots ? 0 : s_own + 1;
        s_other = s_other + 1 == kRadialSlots ? 0 : s_other + 1;
        s_new = s_new + 1 == kRadialSlots ? 0 : s_new + 1;
    }

    // every column stands for itself and its mirror image, (0, 0) for itself
    const double rho2 = (double)(col.dx * col.dx + col.dy * col.dy);
    const double weight = rho2 > 0.0 ? 2.0 : 1.0;
#pragma unroll
    for (int k = 0; k <= kRadialH; k++) {
        const double d2 = rho2 + k * k;
        const double fe = weight * (S.uu[k] + S.vv[k] + S.zz[k]);
        const double rr = weight * (rho2 * S.uu[k] + sqrt(rho2) * k * S.uz[k] + (double)(k * k) * S.zz[k]);
        double *o = lds + 2 * (row * kRadialSums + k * kRadialCols + (far ? 64 : 0) + lane);
        o[0] = fe;
        o[1] = d2 > 0.0 ? fe - 3.0 * rr / d2 : fe;
    }
    __syncthreads();
    if (tid < 2 * kRadialBins) {
        const int b = tid >> 1, part = tid & 1;
        double s = 0.0;
        const int e1 = ra.bin_start[b + 1];
        for (int e = ra.bin_start[b]; e < e1; e++) {
            const double *o = lds + 2 * ra.entries[e] + part;
            double t = 0.0;
#pragma unroll
            for (int r = 0; r < kRadialTY; r++) t += o[2 * r * kRadialSums];
            s += t;
        }
        ra.partials[(long long)block * 2 * kRadialBins + tid] = s;
    }
}

}  // namespace sn
