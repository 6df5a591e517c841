// sn_torus.h -- whole-lattice sweep of small replicas in one workgroup (gfx950, FP64).
//
// A replica small enough for LDS (its x, y, z (, length) arrays at once) is
// swept by one workgroup, sweep after sweep, inside one launch: no tiles, no
// halo staging, no launch per coarse colour.  The sites are coloured by a
// sublattice that holds the replica's box vectors and whose shortest vector is
// longer than DipoleCutOff, so the sites of one colour are more than rc apart
// through the periodic boundary and update together; colours follow one
// another with a workgroup barrier.  The neighbours' LDS addresses (periodic
// wrap, the reference's % X, src/starrynight-montecarlo-core.c:97) come from a
// table of the replica's box, streamed from L2 three rounds ahead: forming them in
// the round took 66 of its instructions (25 x 25), after the barrier.
// Per site the arithmetic is the tile kernels': G lanes share a site, each
// lane takes NPL of the +-r pairs, one scalar per lane is reduced over the
// group, and the Metropolis threshold and proposal come from the same
// counter RNG draw of (seed, replica, sweep, site).
#pragma once
#include "sn_kernels.h"

namespace sn {

// One box size: where its tables start.
struct TorusBox {
    int sites_off;             // sites by colour (linear index), N of them
    int nrounds;               // of one sweep
    int chunk_off, nchunks;    // first round and first site of each run of proposals (nchunks + 1 of both)
    long long round_off;       // first of its lane records: R per lane and round
};

struct TorusArgs {
    double4 *lat;
    const RepDev *reps;
    const PairDev *pairs;      // padded with zero pairs to kPairSlots
    const int *box_of;         // R entries
    const TorusBox *boxes;
    const int *sites;          // per box (sites_off)
    // per box (round_off), round, site and lane, for the layout of the launch
    // (uniform or mixed lengths):
    const int2 *owns;          // LDS bytes of the lane's own component (with kLast, kIdle) and of its proposal's
    const int *nears;          // 2 NPL: LDS bytes of its neighbours, + and - of each pair
    const int *chunks;         // per box (chunk_off)
    const unsigned *sweep_ctr;
    unsigned long long *counters;  // 2 per replica: accepted, rejected (accumulated)
    int site_bytes;            // LDS bytes of the largest replica's sites
    int prop_cap;              // proposal slots (>= the largest colour): colours are drawn in
                               // runs of at most this many sites
};

// Flags in the low bits of an own component's LDS address: a colour's last
// round (it ends with the barrier), a group without a site.
constexpr int kLast = 1, kIdle = 2;

// LDS layout in blocks of 256 sites, so that a site's components lie at fixed
// distances from its address, which the reads take as immediate offsets (x, y
// and z arrays a runtime stride apart cost two adds per neighbour): x, y and z
// arrays of the block, or with mixed lengths (x, y) and (z, L) pairs.  The
// distances are odd multiples of 8 or 16 bytes, so that a site's components
// lie in different banks, and beyond the reach of a two-address read: blocks
// of 64 with 512 bytes between x and y, which the compiler reads as one
// read2st64 from one bank, ran 25 x 25 16% slower than the runtime strides.
__host__ __device__ inline int torus_address(int site, bool mixed)
{
    return (site >> 8) * (mixed ? 2 * 4112 : 3 * 2056) + (site & 255) * (mixed ? 16 : 8);
}
// of component c (x, y, z, L) relative to the site's address
__host__ __device__ inline int torus_component(int c, bool mixed)
{
    return mixed ? (c >> 1) * 4112 + (c & 1) * 8 : (c < 3 ? c : 2) * 2056;
}

// LDS at a byte address: the kernel has no static LDS (the host refuses an
// instance that has any), so its dynamic array, and with it torus_address,
// begins at 0.  (Through a pointer into the array
// every read of a table's address cost an add of that zero.)
typedef double lds_double2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ T lds_load(int address)
{
    return *(const __attribute__((address_space(3))) T *)(uintptr_t)(unsigned)address;
}
__device__ __forceinline__ void lds_store(int address, double v)
{
    *(__attribute__((address_space(3))) double *)(uintptr_t)(unsigned)address = v;
}

// R sites per group and round, of one colour: with one (colours that fit the
// groups) a round's latencies follow one another; two sites' reads, sums and
// reductions overlap (64 x 12^3 at DipoleCutOff 3, 54 sites a colour on 16
// groups, 10 sweeps: 643 -> 569 us).
template <int G, int NPL, bool MIXED, int BLK, int R>
__global__ __launch_bounds__(BLK) void torus_sweep_kernel(TorusArgs t, int nsweeps)
{
    static_assert(G * NPL <= kPairSlots, "the pair table covers every lane's slots");
    extern __shared__ __align__(16) double smem[];
    const int tid = threadIdx.x, r = blockIdx.x;
    const RepDev rep = t.reps[r];
    const TorusBox box = t.boxes[t.box_of[r]];
    const int N = rep.X * rep.Y * rep.Z;
    constexpr int YO = MIXED ? 8 : 2056, ZO = 4112;   // torus_component of y and z
    char *sites = (char *)smem;                               // torus_address, torus_component
    double *prop = (double *)(sites + t.site_bytes);          // px, py, pz and threshold of slot k at prop[4 k]
    int *s_chunk = (int *)(prop + 4 * t.prop_cap);
    unsigned *s_cnt = (unsigned *)(s_chunk + 2 * (box.nchunks + 1));   // (no static LDS: sites begin at address 0)
    unsigned short *s_site = (unsigned short *)(s_cnt + 2);   // sites by colour
    double4 *lat = t.lat + rep.base;

    // ---- the whole replica into LDS ----
    for (int i = tid; i < N; i += BLK) {
        const double4 v = lat[i];
        char *p = sites + torus_address(i, MIXED);
        if (MIXED) {
            *(double2 *)p = make_double2(v.x, v.y);
            *(double2 *)(p + ZO) = make_double2(v.z, v.w);
        } else {
            *(double *)p = v.x; *(double *)(p + YO) = v.y; *(double *)(p + ZO) = v.z;
        }
        s_site[i] = (unsigned short)t.sites[box.sites_off + i];
    }
    for (int i = tid; i < 2 * (box.nchunks + 1); i += BLK) s_chunk[i] = t.chunks[box.chunk_off + i];

    // ---- this lane's share of the +-r pairs ----
    const int part = tid % G;
    double nx[NPL], ny[NPL], nz[NPL], w[NPL], w3[NPL], nnf = 0.0;
#pragma unroll
    for (int m = 0; m < NPL; m++) {
        const PairDev p = t.pairs[part + m * G];
        nx[m] = p.nx; ny[m] = p.ny; nz[m] = p.nz; w[m] = p.w; w3[m] = -3.0 * p.w;
        // nearest-neighbour pairs come first in the table, so they sit in slot 0
        if (m == 0) nnf = p.nn ? 1.0 : 0.0;
    }
    const double rbeta = 1.0 / rep.beta;
    // the field term, the factors of uniform lengths and a site's own
    // components: see the tile sweep
    const double J = rep.J, K = rep.K;
    const double E0 = part == 0 ? rep.E[0] : 0.0, E1 = part == 0 ? rep.E[1] : 0.0, E2 = part == 0 ? rep.E[2] : 0.0;
    if constexpr (!MIXED) {
        const double LL = rep.L0 * rep.L0;
#pragma unroll
        for (int m = 0; m < NPL; m++) { w[m] *= LL; w3[m] *= LL; }
        w[0] -= nnf * J;
    }
    const double Kp = part < 2 ? K : 0.0;
    const bool writer = part < 3 && (MIXED || rep.L0 != 0.0);   // vacancies never move and are not counted
    unsigned nacc = 0, nvis = 0;   // accepted (on a group's first lane), visited
    if (tid < 2) s_cnt[tid] = 0;

    // ---- the round tables, three rounds ahead (a load issued one round ahead
    // is still on its way from L2 when the round begins) ----
    struct Near {
        int a[2 * NPL];   // + and - neighbour of each pair
    };
    struct Round {
        int2 own[R];
        Near n[R];
    };
    const int2 *owns = t.owns + box.round_off + tid;
    const Near *nears = (const Near *)t.nears + box.round_off + tid;
    Round q0, q1, q2;
    int ahead = 0;   // the round loaded next (the sweep's rounds repeat)
    auto fetch = [&](Round &q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            q.own[i] = owns[(long long)(ahead * R + i) * BLK];
            q.n[i] = nears[(long long)(ahead * R + i) * BLK];
        }
        ahead = ahead + 1 < box.nrounds ? ahead + 1 : 0;
    };
    fetch(q0);
    fetch(q1);
    fetch(q2);
    const unsigned sweep0 = t.sweep_ctr[r];
    __syncthreads();

    for (int s = 0; s < nsweeps; s++) {
        const unsigned sweep = sweep0 + (unsigned)s;
        for (int ch = 0; ch < box.nchunks; ch++) {
            // ---- proposals of a run of colours, two sites per lane at a time
            // (one where no lane of the wave has a second) ----
            const int p0 = s_chunk[2 * ch + 1], np = s_chunk[2 * ch + 3] - p0;
            auto store = [&](int k, double px, double py, double pz, double u) __attribute__((always_inline)) {
                ((double2 *)prop)[2 * k] = make_double2(px, py);
                ((double2 *)prop)[2 * k + 1] = make_double2(pz, metropolis_threshold(u, rep.beta, rbeta));
            };
            for (int i = tid; i < np; i += 2 * BLK) {
                const bool two = i + BLK < np;
                if (__any(two)) {
                    const uint32_t site[2] = {s_site[p0 + i], s_site[p0 + (two ? i + BLK : i)]};
                    double px[2], py[2], pz[2], u[2];
                    counter_draws<2>(rep.seed, (uint32_t)r, sweep, site, rep.constrain_to_x, px, py, pz, u);
                    store(i, px[0], py[0], pz[0], u[0]);
                    if (two) store(i + BLK, px[1], py[1], pz[1], u[1]);
                } else {
                    double px, py, pz, u;
                    counter_draw(rep.seed, (uint32_t)r, sweep, s_site[p0 + i], rep.constrain_to_x, px, py, pz, u);
                    store(i, px, py, pz, u);
                }
            }
            const int r0 = __builtin_amdgcn_readfirstlane(s_chunk[2 * ch]);
            const int r1 = __builtin_amdgcn_readfirstlane(s_chunk[2 * ch + 2]);
            __syncthreads();
            // ---- the run's rounds: every group decides its sites; a colour's
            // last round ends with the barrier (before it, rounds of a colour
            // are independent of each other) ----
            auto round = [&](const Round &q) __attribute__((always_inline)) {
                // one site: groups without one (whole DPP rows or quads) skip
                // the round.  Two: waves without any do; a group without one
                // runs on the site its entry names and drops the result, so
                // that both sites' instructions are one stream.
                if (R == 1 ? !(q.own[0].x & kIdle) : __any(!(q.own[0].x & kIdle))) {
                    double ax[R][NPL], ay[R][NPL], az[R][NPL], bx[R][NPL], by[R][NPL], bz[R][NPL], la[R][NPL], lb[R][NPL];
                    double pv[R], ov[R], dE[R], thr[R], Li[R];
                    auto pair_reads = [&](int i, int m) __attribute__((always_inline)) {
                        const int pa = q.n[i].a[2 * m], pb = q.n[i].a[2 * m + 1];
                        if (MIXED) {
                            const lds_double2 xya = lds_load<lds_double2>(pa), zla = lds_load<lds_double2>(pa + ZO);
                            const lds_double2 xyb = lds_load<lds_double2>(pb), zlb = lds_load<lds_double2>(pb + ZO);
                            ax[i][m] = xya.x; ay[i][m] = xya.y; az[i][m] = zla.x; la[i][m] = zla.y;
                            bx[i][m] = xyb.x; by[i][m] = xyb.y; bz[i][m] = zlb.x; lb[i][m] = zlb.y;
                        } else {
                            ax[i][m] = lds_load<double>(pa);
                            ay[i][m] = lds_load<double>(pa + YO);
                            az[i][m] = lds_load<double>(pa + ZO);
                            bx[i][m] = lds_load<double>(pb);
                            by[i][m] = lds_load<double>(pb + YO);
                            bz[i][m] = lds_load<double>(pb + ZO);
                        }
                        if (m + 1 == NPL) {
                            pv[i] = lds_load<double>(q.own[i].y);
                            ov[i] = lds_load<double>(q.own[i].x & ~7);
                        }
                    };
                    // two sites: reads run two pairs ahead of the sums (see the
                    // tile sweep; 64 x 12^3, 10 sweeps: 565 us, all reads
                    // first 617)
                    constexpr int AHEAD = R == 1 || R * NPL < 2 ? R * NPL : 2;
#pragma unroll
                    for (int k = 0; k < AHEAD; k++) pair_reads(k / NPL, k % NPL);
#pragma unroll
                    for (int i = 0; i < R; i++) {
                        double hx_, hy_, hz_, gx_, gy_, gz_;
#pragma unroll
                        for (int m = 0; m < NPL; m++) {
                            if (R > 1) asm volatile("" ::: "memory");
                            double mx, my, mz;
                            if (MIXED) {
                                mx = la[i][m] * ax[i][m] + lb[i][m] * bx[i][m];
                                my = la[i][m] * ay[i][m] + lb[i][m] * by[i][m];
                                mz = la[i][m] * az[i][m] + lb[i][m] * bz[i][m];
                                if (m == 0) {
                                    gx_ = nnf * (ax[i][0] + bx[i][0]); gy_ = nnf * (ay[i][0] + by[i][0]);
                                    gz_ = nnf * (az[i][0] + bz[i][0]);
                                }
                            } else {
                                mx = ax[i][m] + bx[i][m]; my = ay[i][m] + by[i][m]; mz = az[i][m] + bz[i][m];
                            }
                            const double f = w3[m] * (nx[m] * mx + ny[m] * my + nz[m] * mz);
                            hx_ = fma(f, nx[m], m == 0 ? (MIXED ? w[m] * mx : fma(w[m], mx, E0)) : fma(w[m], mx, hx_));
                            hy_ = fma(f, ny[m], m == 0 ? (MIXED ? w[m] * my : fma(w[m], my, E1)) : fma(w[m], my, hy_));
                            hz_ = fma(f, nz[m], m == 0 ? (MIXED ? w[m] * mz : fma(w[m], mz, E2)) : fma(w[m], mz, hz_));
                            if (R > 1) asm volatile("" : "+v"(hx_), "+v"(hy_), "+v"(hz_) : : "memory");
                            const int next = i * NPL + m + AHEAD;
                            if (next < R * NPL) pair_reads(next / NPL, next % NPL);
                        }
                        Li[i] = 1.0;
                        if (MIXED) {
                            Li[i] = lane_bcast<3, G>(ov[i]);
                            hx_ = fma(Li[i], hx_, fma(-J, gx_, E0)); hy_ = fma(Li[i], hy_, fma(-J, gy_, E1));
                            hz_ = fma(Li[i], hz_, fma(-J, gz_, E2));
                        }
                        const double d = pv[i] - ov[i];
                        dE[i] = lane_bcast<0, G>(d) * hx_ + lane_bcast<1, G>(d) * hy_ + lane_bcast<2, G>(d) * hz_;
                        if (K > 0.0) {
                            asm volatile("" ::: "memory");
                            dE[i] -= Kp * (fabs(pv[i]) - fabs(ov[i]));
                        }
                        thr[i] = lane_bcast<3, G>(pv[i]);
                    }
#pragma unroll
                    for (int i = 0; i < R; i++) {
                        dE[i] = group_sum_dpp<G>(dE[i]);
                        // (the fence keeps the exchanges above the branch, where every lane is on)
                        asm volatile("" : "+v"(dE[i]), "+v"(thr[i]), "+v"(Li[i]));
                    }
#pragma unroll
                    for (int i = 0; i < R; i++)
                        if (writer && (!MIXED || Li[i] != 0.0) && (R == 1 || !(q.own[i].x & kIdle))) {
                            nvis++;
                            if (dE[i] < thr[i]) {
                                lds_store(q.own[i].x & ~7, pv[i]);
                                nacc++;
                            }
                        }
                }
                if (__builtin_amdgcn_readfirstlane(q.own[0].x) & kLast) __syncthreads();
            };
            // (three copies of the round: rotating one register set into the
            // next would wait for the loads just issued)
            int rd = r0;
            for (; rd + 3 <= r1; rd += 3) {
                round(q0);
                fetch(q0);
                round(q1);
                fetch(q1);
                round(q2);
                fetch(q2);
            }
            for (; rd < r1; rd++) {
                round(q0);
                q0 = q1;
                q1 = q2;
                fetch(q2);
            }
        }
    }

    // ---- count, write back ----
    if (part == 0 && nvis) {
        if (nacc) atomicAdd(&s_cnt[0], nacc);
        atomicAdd(&s_cnt[1], nvis - nacc);
    }
    __syncthreads();
    if (tid < 2) atomicAdd(t.counters + 2 * r + tid, (unsigned long long)s_cnt[tid]);
    for (int i = tid; i < N; i += BLK) {
        const char *p = sites + torus_address(i, MIXED);
        double4 v;
        v.x = *(const double *)p;
        v.y = *(const double *)(p + YO);
        v.z = *(const double *)(p + ZO);
        v.w = MIXED ? *(const double *)(p + ZO + 8) : rep.L0;
        lat[i] = v;
    }
}

}  // namespace sn
