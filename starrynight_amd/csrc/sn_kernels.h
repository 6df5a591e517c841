// sn_kernels.h -- HIP kernels of the Metropolis dipole-lattice path (gfx950).
//
// All arithmetic is IEEE double.  The dipolar part of site_energy
// (src/starrynight-montecarlo-core.c:91-117) is evaluated as a local field:
//   dE_dd = L_i (p' - p) . h_i,   h_i = sum_r L_j (p_j - 3 n (n . p_j)) / d^3,
// which is the reference's per-neighbour expression with the common factor
// (p' - p) pulled out (it is linear in the proposal), and the cage term as
//   dE_cage = -J (p' - p) . g_i,  g_i = sum_{|r|=1} p_j.
#pragma once
#include "sn_device.h"

namespace sn {

constexpr int kBlock = 256;   // threads per workgroup of the tile sweep
constexpr int kPairSlots = 512;   // largest lanes x pairs per lane of a gather instance

struct SweepArgs {
    double4 *lat;
    const RepDev *reps;
    const TileDev *tiles;
    const ShapeDev *shapes;
    const PairDev *pairs;      // padded with zero pairs to kPairSlots
    const unsigned *sweep_ctr;
    unsigned long long *counters;  // 2 per tile: accepted, rejected (accumulated over sweeps)
    const int *sites;         // per shape (TileDev.sites_off): tile sites by fine colour, packed lx | ly << 10 | lz << 20
    const int *gsteps;        // per shape (TileDev.gstep_off): per step BLK / G entries (step_entry), an idle row, then
                              // the first step and the first site of each proposal chunk (nchunks + 1 of both)
    int npairs;               // read by no kernel, but the arguments behind it stay where they are: without it tiles
                              // of mixed lengths ran 2% faster, some of uniform lengths 1% slower
    int rc, two_d, max_region;
    int prop_stride;          // proposal slots per chunk (<= kBlock)
};

// Entry of a lane group in the step table: the site's region index, its slot
// in the chunk's proposals, a flag on a colour's last step (it ends with the
// barrier), and the sign bit for a group without a site.
constexpr int kStepBarrier = 1 << 30, kStepIdle = (int)0x80000000u;
__host__ __device__ inline int step_entry(int ri, int slot, bool last, bool idle)
{
    return ri | (slot << 16) | (last ? kStepBarrier : 0) | (idle ? kStepIdle : 0);
}

// DPP lane exchange of a double (two 32-bit moves); CTRL is a dpp_ctrl code.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v)
{
    // every control used here permutes lanes within a row, so each lane has a
    // source and no old value is needed
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, true);
    hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// Lane C of the aligned quad (G < 16) or of the row of 16 lanes (G >= 16, one
// instruction) in every lane of it.
template <int C, int G>
__device__ __forceinline__ double lane_bcast(double v)
{
    if constexpr (G >= 16) return __builtin_amdgcn_update_dpp(v, v, 0x150 + C, 0xF, 0xF, true);
    else return dpp_f64<C * 0x55>(v);
}

// v + v[lane ^ 16] (ROWS = 16) or v + v[lane ^ 32] (ROWS = 32) in every lane,
// by gfx950's v_permlane16_swap / v_permlane32_swap on both halves of the
// double: the two results of a swap hold the even and the odd row of each
// row pair (no LDS round trip, unlike ds_swizzle or ds_bpermute).  The sum is
// the same in both lanes of a pair, bit for bit (addition commutes).
template <int ROWS>
__device__ __forceinline__ double pair_sum_f64(double v)
{
    const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    if constexpr (ROWS == 16) {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    }
}

// Sum over aligned groups of G lanes, result in every lane of the group:
// butterfly of row_mirror (i <-> 15-i), row_half_mirror (i <-> 7-i) and
// quad permutations xor 2, xor 1, plus row-pair swaps for G >= 32 (lane xor
// 16) and G = 64 (lane xor 32).
template <int G>
__device__ __forceinline__ double group_sum_dpp(double v)
{
    static_assert(G == 1 || G == 2 || G == 4 || G == 8 || G == 16 || G == 32 || G == 64, "G is a power of two <= 64");
    if (G >= 64) v = pair_sum_f64<32>(v);
    if (G >= 32) v = pair_sum_f64<16>(v);
    if (G >= 16) v += dpp_f64<0x140>(v);
    if (G >= 8) v += dpp_f64<0x141>(v);
    if (G >= 4) v += dpp_f64<0x4E>(v);
    if (G >= 2) v += dpp_f64<0xB1>(v);
    return v;
}

// -3 w n of a lane's pairs (present only where the kernel keeps it)
template <int N, bool ON> struct PairTerm { double x[N], y[N], z[N]; };
template <int N> struct PairTerm<N, false> {};

// One workgroup updates one tile: stage tile + halo in LDS, draw the
// proposals of all tile sites, run the fine colours one after another (G lanes
// share one site's neighbour sum, NPL +-r pairs per lane), write the tile back.
//
// BLK threads per workgroup (256 or 512); proposals are drawn in chunks of at
// most prop_stride (<= kBlock) sites.  The staged x, y, z arrays are read by
// separate instructions: a read2 of x and y at a stride that is a multiple of
// the bank cycle puts both halves in one bank (measured: 2.9 conflict cycles
// per LDS instruction against 1.3, and 9% slower at 8^3 tiles).
// MRC > 0 fixes the stride of the staged arrays at compile time (the launch's
// max_region must equal it, and its prop_stride kBlock): the y and z reads then
// take immediate LDS offsets from the x address instead of an address add each
// (measured 2% at 8^3 tiles).
template <int G, int NPL, bool MIXED, int BLK, int MRC = 0>
__global__ __launch_bounds__(BLK) void tile_sweep_kernel(SweepArgs a, int first_tile, int ntiles)
{
    static_assert(G * NPL <= kPairSlots, "the pair table covers every lane's slots");
    extern __shared__ __align__(16) double smem[];
    const int tid = threadIdx.x;
    const int b = blockIdx.x;
    // Consecutive tiles (spatial neighbours sharing halo sites) go to the same
    // XCD: the hardware deals workgroups to the 8 XCDs round-robin.
    const int t = (ntiles % 8 == 0) ? (b % 8) * (ntiles / 8) + b / 8 : b;
    const TileDev tile = a.tiles[first_tile + t];
    const int hx = a.rc, hy = a.rc, hz = a.two_d ? 0 : a.rc;
    const int tx = tile.size & 1023, ty = (tile.size >> 10) & 1023, tz = tile.size >> 20;
    const int RX = tx + 2 * hx, RY = ty + 2 * hy, RZ = tz + 2 * hz;
    const int RZs = gather_zstride(RZ);                    // z stride in LDS (>= RZ)

    const int MR = MRC > 0 ? MRC : a.max_region;          // stride of the staged arrays
    // Uniform lengths: x, y and z arrays (the fixed-stride instances reach y
    // and z by immediate offsets from the x address).  Mixed lengths: (x, y)
    // pairs and (z, L) pairs, so two 16-byte reads bring a neighbour's
    // dipole and length (measured at DipoleCutOff 4, half vacant: three
    // 8-byte reads and a length read 2.49e9, (z, L) pairs 2.68e9, both pairs
    // 2.81e9 site-updates/s; the uniform instances lost 2% with (x, y) pairs).
    constexpr int ZS = MIXED ? 2 : 1;                      // doubles per site in the x, y and z arrays
    double *sx = smem;                                     // x of site i at sx[ZS * i]
    double *sy = MIXED ? sx + 1 : sx + MR;                 // y of site i at sy[ZS * i]
    double *sz = sx + 2 * MR;                              // z of site i at sz[ZS * i]
    double *sl = sz + 1;                                   // L of site i at sl[2 * i] (MIXED only)
    // proposals: px, py, pz and threshold of slot k at prop[4 k]
    double *prop = sx + (((MIXED ? 4 : 3) * MR + 1) & ~1);
    const int PS = MRC > 0 ? kBlock : a.prop_stride;        // (fixed-stride launches draw chunks of kBlock)
    int *s_gstep = (int *)(prop + 4 * PS);                 // step table and chunk table
    constexpr int SW = BLK / G;                            // entries per step

    const RepDev rep = a.reps[tile.replica];
    const unsigned sweep = a.sweep_ctr[tile.replica];
    const long long tile_base = ((long long)tile.x0 * tile.Y + tile.y0) * tile.Z + tile.z0;

    const double rbeta = 1.0 / rep.beta;
    auto global_site = [&](int xyz) __attribute__((always_inline)) {   // of packed tile coordinates
        const int lx = xyz & 1023, ly = (xyz >> 10) & 1023, lz = xyz >> 20;
        return (uint32_t)(tile_base + ((long long)lx * tile.Y + ly) * tile.Z + lz);
    };
    // This lane's proposal slot in chunk ch (512 threads: alternate halves of
    // the workgroup, so the first two chunks are drawn side by side)
    auto slot_of = [&](int ch) __attribute__((always_inline)) { return tid - (BLK > kBlock ? (ch & 1) * kBlock : 0); };
    const int k0 = slot_of(0), k1 = slot_of(1);
    const int n0 = tile.first_chunks & 0xFFFF, n1 = tile.first_chunks >> 16;
    const bool draw0 = k0 < n0, draw1 = k1 >= 0 && k1 < n1;   // (k0 is never negative)
    int xyz0 = draw0 ? a.sites[tile.sites_off + k0] : 0;
    int xyz1 = draw1 ? a.sites[tile.sites_off + n0 + k1] : 0;
    // the step table's first entries, on their way to LDS
    constexpr int NT = 4;
    const int nstep = (tile.gsteps_n + 1) * SW + 2 * (tile.nchunks + 1);
    int tab[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) tab[k] = tid + k * BLK < nstep ? a.gsteps[tile.gstep_off + tid + k * BLK] : 0;

    // ---- this lane's share of the neighbour pairs, held in registers ----
    const int part = tid % G;
    const int group = tid / G;
    int dl[NPL];
    double nx[NPL], ny[NPL], nz[NPL], w[NPL], w3[NPL], nnf = 0.0;
#pragma unroll
    for (int m = 0; m < NPL; m++) {
        const PairDev p = a.pairs[part + m * G];   // (padded with zero pairs to every G x NPL)
        dl[m] = (p.dx * RY + p.dy) * RZs + p.dz;
        nx[m] = p.nx; ny[m] = p.ny; nz[m] = p.nz; w[m] = p.w; w3[m] = -3.0 * p.w;
        // nearest-neighbour pairs come first in the table, so they sit in slot 0
        if (m == 0) nnf = p.nn ? 1.0 : 0.0;
    }
    // ---- load tile + halo (periodic wrap).  A lane keeps its (y, z) and walks
    // the x planes, so a load's address costs an add (stepping every lane
    // through the region's mixed radix cost 65 instructions a load).  A launch
    // finds the L2 empty and these loads take microseconds: NV of them per lane
    // (all of a fixed-stride tile's 14 planes) are issued before anything
    // waits, behind the few loads that the draws below need (loads return in
    // order), and unconditionally (past the last plane: the last one again), so
    // that the wait for the earlier loads can count them ----
    constexpr int NV = MRC > 0 ? 14 : 8;
    const double4 *lat = a.lat + tile.base;
    const int rows = RY * RZ;
    const int per = rows < BLK ? BLK / rows : 1;   // planes loaded by one pass of the workgroup
    double4 v[NV];
    struct Row {
        int px, lds;        // first plane; region index of plane 0
        const double4 *src; // plane 0 of the lattice
        bool on;
    };
    // the lane's row in sub-pass s (planes of more than BLK rows take several)
    auto row_of = [&](int s) __attribute__((always_inline)) {
        Row r;
        const int q = tid + s * BLK;
        r.px = q / rows;
        const int k = min(q - r.px * rows, rows - 1), iy = k / RZ, iz = k - iy * RZ;
        r.on = per > 1 ? r.px < per : q < rows;
        if (per == 1) r.px = 0;
        r.lds = iy * RZs + iz;
        r.src = lat + (long long)wrap_once(tile.y0 - hy + iy, tile.Y) * tile.Z + wrap_once(tile.z0 - hz + iz, tile.Z);
        return r;
    };
    auto load_planes = [&](const Row &r, int x) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int ix = min(x + k * per + r.px, RX - 1);
            v[k] = r.src[(long long)(wrap_once(tile.x0 - hx + ix, tile.X) * (tile.Y * tile.Z))];
        }
    };
    Row row = row_of(0);
    load_planes(row, 0);

    // The first two chunks' proposals are drawn while the tile's loads are in
    // flight (the fence keeps the loads above them); the second chunk's wait in
    // registers for their slots.
    double2 nxy, nzt;
    asm volatile("" : "+v"(xyz0), "+v"(xyz1) : : "memory");
#pragma unroll
    for (int k = 0; k < NT; k++)
        if (tid + k * BLK < nstep) s_gstep[tid + k * BLK] = tab[k];
    {
        // 256 threads: both sites of a lane together; 512: one each
        constexpr int ND = BLK > kBlock ? 1 : 2;
        uint32_t site[ND];
        double px[ND], py[ND], pz[ND], u[ND];
        site[0] = global_site(ND == 1 && draw1 ? xyz1 : xyz0);
        site[ND - 1] = ND == 1 ? site[0] : global_site(xyz1);
        if (draw0 || draw1) counter_draws<ND>(rep.seed, (uint32_t)tile.replica, sweep, site, rep.constrain_to_x, px, py, pz, u);
        if (draw0) {
            ((double2 *)prop)[2 * k0] = make_double2(px[0], py[0]);
            ((double2 *)prop)[2 * k0 + 1] = make_double2(pz[0], metropolis_threshold(u[0], rep.beta, rbeta));
        }
        if (draw1) {
            nxy = make_double2(px[ND - 1], py[ND - 1]);
            nzt = make_double2(pz[ND - 1], metropolis_threshold(u[ND - 1], rep.beta, rbeta));
        }
    }
    for (int i = tid + NT * BLK; i < nstep; i += BLK) s_gstep[i] = a.gsteps[tile.gstep_off + i];

    // ---- staged sites into LDS ----
    for (int sub = 0;;) {
        for (int x = 0;;) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int ix = x + k * per + row.px;
                if (row.on && ix < RX) {
                    const int i = ix * (RY * RZs) + row.lds;
                    if (MIXED) {
                        ((double2 *)sx)[i] = make_double2(v[k].x, v[k].y);
                        ((double2 *)sz)[i] = make_double2(v[k].z, v[k].w);
                    } else {
                        sx[i] = v[k].x; sy[i] = v[k].y; sz[i] = v[k].z;
                    }
                }
            }
            x += NV * per;
            if (x >= RX) break;
            load_planes(row, x);
        }
        if (++sub * BLK >= rows) break;
        row = row_of(sub);
        load_planes(row, 0);
    }

    // TN: t = -3 w n per pair in registers, one multiply fewer per pair for
    // three more registers.  Only the fixed-stride instances take it: their
    // LDS (>= 66 KB) allows two workgroups per CU, so up to 256 VGPRs cost no
    // occupancy, while smaller tiles run three workgroups per CU (<= 168).
    constexpr bool TN = MRC > 0;
    // the field term, and with it K's, ride on the group's first lane
    const double J = rep.J, K = rep.K;
    const double E0 = part == 0 ? rep.E[0] : 0.0, E1 = part == 0 ? rep.E[1] : 0.0, E2 = part == 0 ? rep.E[2] : 0.0;
    // A site's own data, one component a lane: lane c of each quad reads p'_c
    // and p_c (c < 3), lane 3 the threshold and (mixed lengths) the length, and
    // hands its difference to the others by DPP: two LDS reads a step instead
    // of the seven doubles every lane needs; an accepted site's components are
    // written by three lanes at once.
    const int comp = part & 3;
    double *own = MIXED ? sx + (comp >> 1) * 2 * MR + (comp & 1) : sx + (comp < 3 ? comp : 2) * MR;
    const double Kp = part < 2 ? K : 0.0;
    // Uniform lengths: L0^2 and the cage strain ride on the weights, w' = L0^2 w
    // (- J for nearest neighbours), so no separate g is accumulated.  Mixed
    // lengths keep g (L_j sits inside h).
    if constexpr (!MIXED) {
        const double LL = rep.L0 * rep.L0;
#pragma unroll
        for (int m = 0; m < NPL; m++) { w[m] *= LL; w3[m] *= LL; }
        w[0] -= nnf * J;
    }
    PairTerm<NPL, TN> t3;
    if constexpr (TN) {
#pragma unroll
        for (int m = 0; m < NPL; m++) { t3.x[m] = w3[m] * nx[m]; t3.y[m] = w3[m] * ny[m]; t3.z[m] = w3[m] * nz[m]; }
    }
    const bool writer = part < 3 && (MIXED || rep.L0 != 0.0);   // vacancies never move and are not counted
    unsigned nacc = 0, nvis = 0;   // accepted (on a group's first lane), visited
    __shared__ unsigned s_cnt[2];
    if (tid < 2) s_cnt[tid] = 0;
    // the pair registers are loaded by now: waiting for them here keeps the
    // waits out of the step loop
#pragma unroll
    for (int m = 0; m < NPL; m++) asm volatile("" : "+v"(dl[m]), "+v"(nx[m]), "+v"(ny[m]), "+v"(nz[m]), "+v"(w[m]));
    __syncthreads();
    if (MIXED) {
        // vacant sites (length 0) leave the tile's step table: the reference
        // returns from MC_move for them before drawing or counting
        // (src/starrynight-montecarlo-core.c:163).  Each step's remaining
        // sites then move to its first lane groups (one lane per step), so
        // whole waves skip the step.  Measured on 128^3 DipoleCutOff 4, half
        // vacant, 512 threads: 1.89e9 -> 2.29e9 (dropping) -> 2.43e9 (packing)
        // site-updates/s.  Packing a colour's sites across its steps instead
        // measured 2.36e9.
        for (int i = tid; i < tile.gsteps_n * SW; i += BLK)
            if (sl[2 * (s_gstep[i] & 0xFFFF)] == 0.0) s_gstep[i] |= kStepIdle;
        __syncthreads();
        for (int st_ = tid; st_ < tile.gsteps_n; st_ += BLK) {
            int *row = s_gstep + st_ * SW;
            const int idle = row[0] | kStepIdle;   // with the row's barrier flag
            int k = 0;
            for (int g = 0; g < SW; g++) {
                const int e_ = row[g];
                if (e_ >= 0) row[k++] = e_;
            }
            for (; k < SW; k++) row[k] = idle;
        }
        __syncthreads();
    }

    const int *chunk = s_gstep + (tile.gsteps_n + 1) * SW;
    for (int ch = 0; ch < tile.nchunks; ch++) {
        const int st0 = __builtin_amdgcn_readfirstlane(chunk[2 * ch]);
        const int st1 = __builtin_amdgcn_readfirstlane(chunk[2 * ch + 2]);
        if (ch > 0) {
            // the proposals drawn ahead take the slots (the last step of a
            // chunk ended with the barrier), then the following chunk's are drawn
            const int s0 = chunk[2 * ch + 1], s1 = chunk[2 * ch + 3], k = slot_of(ch);
            if (k >= 0 && k < s1 - s0) {
                ((double2 *)prop)[2 * k] = nxy;
                ((double2 *)prop)[2 * k + 1] = nzt;
            }
            if (ch + 1 < tile.nchunks) {
                const int s2 = chunk[2 * ch + 5], kn = slot_of(ch + 1);
                if (kn >= 0 && kn < s2 - s1) {
                    double u;
                    counter_draw(rep.seed, (uint32_t)tile.replica, sweep, global_site(a.sites[tile.sites_off + s1 + kn]),
                                 rep.constrain_to_x, nxy.x, nxy.y, nzt.x, u);
                    nzt.y = metropolis_threshold(u, rep.beta, rbeta);
                }
            }
            __syncthreads();
        }
        // this chunk's steps: every group decides one site per step; a step
        // holds sites of one colour and a colour's last step ends with the
        // barrier.  The next step's entry loads with this step's data (the LDS
        // table has one spare row, whose value is never used).
        int e = s_gstep[st0 * SW + group];
        for (int st = st0; st < st1; st++) {
            // a group without a site this step (a short colour) skips the step:
            // its lanes issue no LDS reads (the group's lanes are whole DPP rows,
            // so the reduction of the active groups is unaffected)
            const int e_next = s_gstep[(st + 1) * SW + group];
            if (e >= 0) {
                const int ri = e & 0xFFFF, pq = (e >> 16) & 0xFF;
                double hx_, hy_, hz_, gx_, gy_, gz_;
                double ax[NPL], ay[NPL], az[NPL], bx[NPL], by[NPL], bz[NPL], la[NPL], lb[NPL];
                double pv, ov;
                const double *cx = sx + ri, *cy = sy + ri, *cz = sz + ri;
                const double2 *cxy = (const double2 *)sx + ri, *czl = (const double2 *)sz + ri;
                auto pair_reads = [&](int m) __attribute__((always_inline)) {
                    if (MIXED) {
                        const double2 pa = cxy[dl[m]], pb = cxy[-dl[m]];
                        const double2 za = czl[dl[m]], zb = czl[-dl[m]];
                        ax[m] = pa.x; ay[m] = pa.y; az[m] = za.x; la[m] = za.y;
                        bx[m] = pb.x; by[m] = pb.y; bz[m] = zb.x; lb[m] = zb.y;
                    } else {
                        ax[m] = cx[dl[m]]; ay[m] = cy[dl[m]]; az[m] = cz[dl[m]];
                        bx[m] = cx[-dl[m]]; by[m] = cy[-dl[m]]; bz[m] = cz[-dl[m]];
                    }
                };
                auto site_reads = [&]() __attribute__((always_inline)) {
                    pv = prop[4 * pq + comp];
                    ov = own[ZS * ri];
                };
                // The reads run AHEAD pairs ahead of the sums: a wave's wait
                // names at most 15 outstanding LDS reads, so with all of a
                // step's reads issued at once the first sums waited for half of
                // them (64^3: 10.51 -> 10.35 ms per 50 sweeps)
                constexpr int AHEAD = NPL < 3 ? NPL : 3;
#pragma unroll
                for (int m = 0; m < AHEAD; m++) pair_reads(m);
                if (NPL == AHEAD) site_reads();
#pragma unroll
                for (int m = 0; m < NPL; m++) {
                    asm volatile("" ::: "memory");
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
                    const double s = nx[m] * mx + ny[m] * my + nz[m] * mz;
                    // the first pair starts the sums (no adds of +0.0); each
                    // component is two dependent FMAs
                    double tx, ty, tz, f;
                    if constexpr (TN) { tx = t3.x[m]; ty = t3.y[m]; tz = t3.z[m]; f = s; }
                    else { tx = nx[m]; ty = ny[m]; tz = nz[m]; f = w3[m] * s; }
                    hx_ = fma(f, tx, m == 0 ? (MIXED ? w[m] * mx : fma(w[m], mx, E0)) : fma(w[m], mx, hx_));
                    hy_ = fma(f, ty, m == 0 ? (MIXED ? w[m] * my : fma(w[m], my, E1)) : fma(w[m], my, hy_));
                    hz_ = fma(f, tz, m == 0 ? (MIXED ? w[m] * mz : fma(w[m], mz, E2)) : fma(w[m], mz, hz_));
                    asm volatile("" : "+v"(hx_), "+v"(hy_), "+v"(hz_) : : "memory");
                    if (m + AHEAD < NPL) pair_reads(m + AHEAD);
                    if (m + AHEAD + 1 == NPL) site_reads();
                }
                if (MIXED) {
                    const double Li = lane_bcast<3, G>(ov);
                    hx_ = fma(Li, hx_, fma(-J, gx_, E0)); hy_ = fma(Li, hy_, fma(-J, gy_, E1));
                    hz_ = fma(Li, hz_, fma(-J, gz_, E2));
                }
                const double d = pv - ov;
                double dE = lane_bcast<0, G>(d) * hx_ + lane_bcast<1, G>(d) * hy_ + lane_bcast<2, G>(d) * hz_;
                if (K > 0.0) {   // (kept a branch: three instructions in every step otherwise)
                    asm volatile("" ::: "memory");
                    dE -= Kp * (fabs(pv) - fabs(ov));
                }
                dE = group_sum_dpp<G>(dE);
                // (the fence keeps the exchange above the branch, where lane 3 is on)
                double thr = lane_bcast<3, G>(pv);
                asm volatile("" : "+v"(thr));
                nvis++;
                if (writer && dE < thr) {
                    own[ZS * ri] = pv;
                    nacc++;
                }
            }
            if (__builtin_amdgcn_readfirstlane(e) & kStepBarrier) __syncthreads();
            e = e_next;
        }
    }

    // ---- counters: this tile's own slot (one workgroup per tile per launch;
    // adds without a return value, before the tile's stores, so that nothing
    // waits for the old count or for the stores) ----
    if (part == 0 && nvis && writer) {
        if (nacc) atomicAdd(&s_cnt[0], nacc);
        atomicAdd(&s_cnt[1], nvis - nacc);
    }
    __syncthreads();
    if (tid < 2) atomicAdd(a.counters + 2 * (first_tile + t) + tid, (unsigned long long)s_cnt[tid]);

    // ---- write the tile back ----
    double4 *out = a.lat + tile.base;
    {
        const int trows = ty * tz, tper = trows < BLK ? BLK / trows : 1;
        for (int q = tid; q < (trows < BLK ? tper * trows : trows); q += BLK) {
            const int px = q / trows, k = q - px * trows, ly = k / tz, lz = k - ly * tz;
            for (int lx = px; lx < tx; lx += tper) {
                const int ri = ((lx + hx) * RY + (ly + hy)) * RZs + (lz + hz);
                double4 o;
                o.x = sx[ZS * ri]; o.y = sy[ZS * ri]; o.z = sz[ZS * ri];
                o.w = MIXED ? sl[2 * ri] : rep.L0;
                out[tile_base + ((long long)lx * tile.Y + ly) * tile.Z + lz] = o;
            }
        }
    }
}

}  // namespace sn
