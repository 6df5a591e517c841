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
// table of the replica's box, streamed from L2 two rounds ahead: forming them in
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
    int entry_off, nrounds;    // NG step_entry's per round; rounds of one sweep
    int chunk_off, nchunks;    // first round and first site of each run of proposals (nchunks + 1 of both)
    int pad;
    long long near_off;        // 2 NPL shorts per lane and round
};

struct TorusArgs {
    double4 *lat;
    const RepDev *reps;
    const PairDev *pairs;      // padded with zero pairs to kPairSlots
    const int *box_of;         // R entries
    const TorusBox *boxes;
    const int *sites;          // per box (sites_off)
    const int *entries;        // per box (entry_off): site | slot << 13 by group, flags as step_entry
    const unsigned short *nears;   // per box (near_off): 8 x site index of the lane's neighbours, + and - of each pair
    const int *chunks;         // per box (chunk_off)
    const unsigned *sweep_ctr;
    unsigned long long *counters;  // 2 per replica: accepted, rejected (accumulated)
    int max_sites;             // stride of the staged arrays
    int prop_cap;              // proposal slots (>= the largest colour): colours are drawn in
                               // runs of at most this many sites
};

// Entry of a lane group: site and proposal slot have 13 bits each (a replica
// of at most kTorusMaxSites fits in LDS).
constexpr int kTorusMaxSites = 8191;
__host__ __device__ inline int torus_entry(int site, int slot, bool last, bool idle)
{
    return site | (slot << 13) | (last ? kStepBarrier : 0) | (idle ? kStepIdle : 0);
}

template <int G, int NPL, bool MIXED, int BLK>
__global__ __launch_bounds__(BLK) void torus_sweep_kernel(TorusArgs t, int nsweeps)
{
    static_assert(G * NPL <= kPairSlots, "the pair table covers every lane's slots");
    extern __shared__ __align__(16) double smem[];
    const int tid = threadIdx.x, r = blockIdx.x;
    const RepDev rep = t.reps[r];
    const TorusBox box = t.boxes[t.box_of[r]];
    const int N = rep.X * rep.Y * rep.Z;
    const int MS = t.max_sites, PS = t.prop_cap;
    // as the tile sweep: x, y and z arrays, or (x, y) and (z, L) pairs
    constexpr int ZS = MIXED ? 2 : 1;
    double *sx = smem;
    double *sy = MIXED ? sx + 1 : sx + MS;
    double *sz = sx + 2 * MS;
    double *prop = sx + (((MIXED ? 4 : 3) * MS + 1) & ~1);   // px, py, pz and threshold of slot k at prop[4 k]
    int *s_chunk = (int *)(prop + 4 * PS);
    double4 *lat = t.lat + rep.base;

    // ---- the whole replica into LDS ----
    for (int i = tid; i < N; i += BLK) {
        const double4 v = lat[i];
        if (MIXED) {
            ((double2 *)sx)[i] = make_double2(v.x, v.y);
            ((double2 *)sz)[i] = make_double2(v.z, v.w);
        } else {
            sx[i] = v.x; sy[i] = v.y; sz[i] = v.z;
        }
    }
    for (int i = tid; i < 2 * (box.nchunks + 1); i += BLK) s_chunk[i] = t.chunks[box.chunk_off + i];

    // ---- this lane's share of the +-r pairs ----
    const int part = tid % G, group = tid / G;
    constexpr int NG = BLK / G;
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
    const int comp = part & 3;
    double *own = MIXED ? sx + (comp >> 1) * 2 * MS + (comp & 1) : sx + (comp < 3 ? comp : 2) * MS;
    const double Kp = part < 2 ? K : 0.0;
    const bool writer = part < 3 && (MIXED || rep.L0 != 0.0);   // vacancies never move and are not counted
    unsigned nacc = 0, nvis = 0;   // accepted (on a group's first lane), visited
    __shared__ unsigned s_cnt[2];
    if (tid < 2) s_cnt[tid] = 0;

    // ---- the round tables, two rounds ahead of their use ----
    struct Near {
        unsigned ab[NPL];   // 8 x site of the pair's + neighbour, - neighbour << 16
    };
    const int *entries = t.entries + box.entry_off + group;
    const Near *nears = (const Near *)(t.nears + box.near_off) + tid;
    int e0, e1, e2;
    Near n0, n1, n2;
    int ahead = 0;   // the round loaded next (the sweep's rounds repeat)
    auto fetch = [&](int &e, Near &n) __attribute__((always_inline)) {
        e = entries[ahead * NG];
        n = nears[(long long)ahead * BLK];
        ahead = ahead + 1 < box.nrounds ? ahead + 1 : 0;
    };
    fetch(e0, n0);
    fetch(e1, n1);
    __syncthreads();

    for (int s = 0; s < nsweeps; s++) {
        const unsigned sweep = t.sweep_ctr[r] + (unsigned)s;
        for (int ch = 0; ch < box.nchunks; ch++) {
            // ---- proposals of a run of colours, two sites per lane at a time ----
            const int p0 = s_chunk[2 * ch + 1], np = s_chunk[2 * ch + 3] - p0;
            for (int i = tid; i < np; i += 2 * BLK) {
                const bool two = i + BLK < np;
                const uint32_t site[2] = {(uint32_t)t.sites[box.sites_off + p0 + i],
                                          (uint32_t)t.sites[box.sites_off + p0 + (two ? i + BLK : i)]};
                double px[2], py[2], pz[2], u[2];
                counter_draws<2>(rep.seed, (uint32_t)r, sweep, site, rep.constrain_to_x, px, py, pz, u);
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if (q == 0 || two) {
                        ((double2 *)prop)[2 * (i + q * BLK)] = make_double2(px[q], py[q]);
                        ((double2 *)prop)[2 * (i + q * BLK) + 1] =
                            make_double2(pz[q], metropolis_threshold(u[q], rep.beta, rbeta));
                    }
            }
            const int r0 = __builtin_amdgcn_readfirstlane(s_chunk[2 * ch]);
            const int r1 = __builtin_amdgcn_readfirstlane(s_chunk[2 * ch + 2]);
            __syncthreads();
            // ---- the run's rounds: every group decides one site; a colour's
            // last round ends with the barrier (before it, rounds of a colour
            // are independent of each other) ----
            for (int rd = r0; rd < r1; rd++) {
                fetch(e2, n2);
                if (e0 >= 0) {   // whole groups are active or not
                    const int si = e0 & 8191, pq = (e0 >> 13) & 8191;
                    double hx_, hy_, hz_, gx_, gy_, gz_;
                    double ax[NPL], ay[NPL], az[NPL], bx[NPL], by[NPL], bz[NPL], la[NPL], lb[NPL];
#pragma unroll
                    for (int m = 0; m < NPL; m++) {
                        const unsigned a8 = n0.ab[m] & 0xFFFF, b8 = n0.ab[m] >> 16;
                        if (MIXED) {
                            const char *pxy = (const char *)sx, *pzl = (const char *)sz;
                            const double2 pa = *(const double2 *)(pxy + 2 * a8), pb = *(const double2 *)(pxy + 2 * b8);
                            const double2 za = *(const double2 *)(pzl + 2 * a8), zb = *(const double2 *)(pzl + 2 * b8);
                            ax[m] = pa.x; ay[m] = pa.y; az[m] = za.x; la[m] = za.y;
                            bx[m] = pb.x; by[m] = pb.y; bz[m] = zb.x; lb[m] = zb.y;
                        } else {
                            ax[m] = *(const double *)((const char *)sx + a8);
                            ay[m] = *(const double *)((const char *)sy + a8);
                            az[m] = *(const double *)((const char *)sz + a8);
                            bx[m] = *(const double *)((const char *)sx + b8);
                            by[m] = *(const double *)((const char *)sy + b8);
                            bz[m] = *(const double *)((const char *)sz + b8);
                        }
                    }
                    const double pv = prop[4 * pq + comp], ov = own[ZS * si];
#pragma unroll
                    for (int m = 0; m < NPL; m++) {
                        double mx, my, mz;
                        if (MIXED) {
                            mx = la[m] * ax[m] + lb[m] * bx[m];
                            my = la[m] * ay[m] + lb[m] * by[m];
                            mz = la[m] * az[m] + lb[m] * bz[m];
                            if (m == 0) {
                                gx_ = nnf * (ax[0] + bx[0]); gy_ = nnf * (ay[0] + by[0]); gz_ = nnf * (az[0] + bz[0]);
                            }
                        } else {
                            mx = ax[m] + bx[m]; my = ay[m] + by[m]; mz = az[m] + bz[m];
                        }
                        const double f = w3[m] * (nx[m] * mx + ny[m] * my + nz[m] * mz);
                        hx_ = fma(f, nx[m], m == 0 ? (MIXED ? w[m] * mx : fma(w[m], mx, E0)) : fma(w[m], mx, hx_));
                        hy_ = fma(f, ny[m], m == 0 ? (MIXED ? w[m] * my : fma(w[m], my, E1)) : fma(w[m], my, hy_));
                        hz_ = fma(f, nz[m], m == 0 ? (MIXED ? w[m] * mz : fma(w[m], mz, E2)) : fma(w[m], mz, hz_));
                    }
                    double Li = 1.0;
                    if (MIXED) {
                        Li = lane_bcast<3, G>(ov);
                        hx_ = fma(Li, hx_, fma(-J, gx_, E0)); hy_ = fma(Li, hy_, fma(-J, gy_, E1));
                        hz_ = fma(Li, hz_, fma(-J, gz_, E2));
                    }
                    const double d = pv - ov;
                    double dE = lane_bcast<0, G>(d) * hx_ + lane_bcast<1, G>(d) * hy_ + lane_bcast<2, G>(d) * hz_;
                    if (K > 0.0) {
                        asm volatile("" ::: "memory");
                        dE -= Kp * (fabs(pv) - fabs(ov));
                    }
                    dE = group_sum_dpp<G>(dE);
                    // (the fence keeps the exchange above the branch, where lane 3 is on)
                    double thr = lane_bcast<3, G>(pv);
                    asm volatile("" : "+v"(thr), "+v"(Li));
                    if (writer && Li != 0.0) {
                        nvis++;
                        if (dE < thr) {
                            own[ZS * si] = pv;
                            nacc++;
                        }
                    }
                }
                if (__builtin_amdgcn_readfirstlane(e0) & kStepBarrier) __syncthreads();
                e0 = e1; n0 = n1;
                e1 = e2; n1 = n2;
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
        double4 v;
        v.x = sx[ZS * i]; v.y = sy[ZS * i]; v.z = sz[ZS * i];
        v.w = MIXED ? sz[2 * i + 1] : rep.L0;
        lat[i] = v;
    }
}

}  // namespace sn
