// gi_kernels.hip -- HIP kernels of the Giant-Impact step loop for gfx950.
//
// The reference evaluates the Greenspan Fe/Si force in one all-pairs kernel
// whose inner loop branches on material, distance and receding
// (getForcesCollisionSingleGPU, Code/ImpactCode/impactAddTime.cu:245-377).
// Here the same force is produced by three passes:
//
//   1. all pairs, branch free: sum_j (G mi mj) dp / r^3 with a hardware rsq,
//      in one of two forms chosen per simulation by the tuning table:
//      k_gravity (one-sided: i-particles in registers, R per lane,
//      j-particles through wave-uniform scalar loads, Kahan-folded float
//      tiles, one j-chunk per wavefront, partial sums to a slot buffer), or
//      the mutual pass (k_mutual_pad, k_mutual, k_mutual_sum: each pair
//      evaluated once for both particles, per-particle compensated sums).
//   2. the contact grid -- a spatial hash of cells of size 1 (the element
//      diameter) built by counting sort (k_grid_*).
//   3. k_finish   -- per particle: its all-pairs sum plus, for every pair
//      with r < 1 found through the grid, the reference's exact piecewise
//      contact force minus what pass 1 added for that pair.  When every
//      simulation takes the mutual pass, the same correction is computed by
//      k_contact_corr beside pass 1 (it needs only the grid) and added by
//      k_mutual_sum.
//
// Only pairs with r < 1 can differ from gravity (impactAddTime.cu:300,320,349),
// so the sum equals the reference's force up to float rounding, and the
// contact branch decisions are made with the reference's own arithmetic.
#include "gi_device.h"

#include <type_traits>

namespace gi {

// ---------------------------------------------------------------------------
// Pass 1: all-pairs gravity (and the potential variant for the energy check)
// ---------------------------------------------------------------------------

__device__ __forceinline__ void kahan_add(float& sum, float& comp, float v) {
    float y = v - comp;
    float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
}

// R: i-particles per lane.  T: j per float tile between Kahan folds.
// POT: accumulate sum_j 1/r (self excluded) instead of sum_j dp/r^3.
// V: how r^-3 is formed (0: rsq cubed, 1: rsq times rcp).
template <int R, int T, bool POT, int V>
__global__ __launch_bounds__(256) void k_gravity(const float4* __restrict__ pos,
                                                 const GravTask* __restrict__ tasks, int ntasks,
                                                 const SimDesc* __restrict__ sims,
                                                 float4* __restrict__ partial) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    if (w >= ntasks) return;
    const GravTask t = tasks[w];
    const int start = sims[t.sim].start;
    const int fe_end = sims[t.sim].fe_end;
    const int end = sims[t.sim].end;
    const int pbase = sims[t.sim].partial_base;
    const float gFeFe = sims[t.sim].law.GMassFeFe;
    const float gFeSi = sims[t.sim].law.GMassFeSi;

    float xi[R], yi[R], zi[R];
    float ax[R], ay[R], az[R], cx[R], cy[R], cz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int i = t.i0 + r * 64 + lane;
        int ic = i < end ? i : end - 1;
        float4 p = pos[ic];
        xi[r] = p.x;
        yi[r] = p.y;
        zi[r] = p.z;
        ax[r] = ay[r] = az[r] = 0.0f;
        cx[r] = cy[r] = cz[r] = 0.0f;
    }

    for (int jb = t.j0; jb < t.j1; jb += T) {
        const int je = min(jb + T, t.j1);
        float tx[R], ty[R], tz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) tx[r] = ty[r] = tz[r] = 0.0f;
#pragma unroll 4
        for (int j = jb; j < je; ++j) {
            const float4 pj = pos[j];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float dx = pj.x - xi[r];
                float dy = pj.y - yi[r];
                float dz = pj.z - zi[r];
                if constexpr (!POT) {
                    float s = inv_r3<V>(fast_r2(dx, dy, dz));
                    tx[r] = __builtin_fmaf(s, dx, tx[r]);
                    ty[r] = __builtin_fmaf(s, dy, ty[r]);
                    tz[r] = __builtin_fmaf(s, dz, tz[r]);
                } else {
                    float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    float ri = r2 > 0.0f ? __builtin_amdgcn_rsqf(r2) : 0.0f;
                    tx[r] += ri;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            kahan_add(ax[r], cx[r], tx[r]);
            if constexpr (!POT) {
                kahan_add(ay[r], cy[r], ty[r]);
                kahan_add(az[r], cz[r], tz[r]);
            }
        }
    }

    const int n = end - start;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int i = t.i0 + r * 64 + lane;
        if (i < end) {
            const bool ife = i < fe_end;
            const float g = t.jfe ? (ife ? gFeFe : gFeSi) : (ife ? gFeSi : 1.0f);
            float4 o;
            o.x = (ax[r] - cx[r]) * g;
            o.y = (ay[r] - cy[r]) * g;
            o.z = (az[r] - cz[r]) * g;
            o.w = 0.0f;
            partial[pbase + t.chunk * n + (i - start)] = o;
        }
    }
}

// sim_of: for each particle its simulation index (particle ranges are given
// by sims[]); computed by a binary search over the sorted starts.
__device__ __forceinline__ int find_sim(const SimDesc* __restrict__ sims, int nsims, int i) {
    int lo = 0, hi = nsims - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sims[mid].start <= i)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// Pass 1, mutual form: each pair evaluated once, applied to both particles
// ---------------------------------------------------------------------------
//
// The pair term (G mi mj) dp / r^3 is odd in dp and r^2 is even, so the term
// j receives from i is exactly the negation of the one i receives from j.
// A wavefront holds a row of 64*R particles in registers (R per lane) and
// streams 64-particle blocks j of the same simulation that lie beyond the
// row.  Each lane holds the force accumulator of one j of the block; after
// every step the accumulators rotate by one lane (DPP wave_ror), so in 64
// steps every lane has met every j of the block and each j has collected the
// terms of all 64*R row particles.  The positions stay put in wave-private
// LDS and each step reads the one its lane's accumulator now belongs to.
// Per pair: 15 VALU ops including one rsq plus 3/R lane rotations, for two
// interactions, against 12 ops per interaction one-sided.  Measured on
// gfx950: rotating the positions with DPP as well is 6% slower (the
// rotation sits on every step's dependency chain); accumulating the j-side
// terms with LDS float adds instead of rotating is about 5x slower.
//
// Simulations are copied into a padded layout (iron then silicate, each
// rounded up to whole rows with ghosts far away) so that every row and every
// 64-block is of one material and the gravity product is one factor per task.
// The row against itself ("diag" task) takes each of its pairs once too (a
// one-sided form at R = 8 made the 64-simulation batched step 1.5% slower).
// Outputs: per task an i-side slot (an (x, y, z) record per place of the
// row) and per (row, j-block) a j-side slab entry (an (x, y, z) record per
// j), so that k_mutual_sum reads 768 contiguous bytes per wavefront and
// entry; k_mutual_sum adds them in
// compensated float sums in a fixed order.  Both sides accumulate in plain
// float: a j-side entry sums
// 64*R terms, an i-side slot at most one chunk (<= 4096 j, the planner's
// cap), so the rounding error stays at a few 1e-6 of the sum of the terms'
// magnitudes; leaving out tile sums and compensation keeps the register
// count low enough for five (k_mutual) or six (k_mutual_grp) wavefronts per
// SIMD at R = 8.

__device__ __forceinline__ float rotate_lanes(float v) {
    // wave_ror:1 -- lane l reads lane l-1 (mod 64).
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x13C, 0xF, 0xF, false));
}

// Orders this wavefront's LDS accesses before and after (its lanes exchange
// data through LDS).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Offset (in entries, per plane) of row `row`'s part of a simulation's
// j-side slab: rows before it hold gn - (r+1)*B entries each.
__host__ __device__ __forceinline__ long long jside_row_offset(int row, int gn, int B) {
    return (long long)row * gn - (long long)B * row * (row + 1) / 2;
}

// What group g of WB places adds to a place's entry offset over that of
// group 0: SumBlock::jfirst + 3 times this is the place's record.
__host__ __device__ __forceinline__ long long sum_group_offset(int g, int gn, long long WB) {
    return (long long)g * gn - WB * g * (g + 1) / 2 - WB * g;
}

constexpr int kMutualWaves = 4;  // wavefronts per block of k_mutual

// One wavefront's task t of simulation sd (P: its padded positions, q: the
// wavefront's 128 float4 of LDS): a row against itself (t.diag) or against
// j beyond the row, whose j-side sums go to J (one (x, y, z) record per
// entry, entry j - (t.row + 1) * B); the row's i-side sums go to slot t.slot
// (one (x, y, z) record per place of the row).  POT: x only.
template <int R, bool POT>
__device__ __forceinline__ void mutual_wave_task(const MutualTask& t, const SimDesc& sd,
                                                 const float4* __restrict__ P, float4* __restrict__ q,
                                                 float* __restrict__ iside, float* __restrict__ J, int lane) {
    constexpr int B = 64 * R;
    const int ib = t.row * B;
    const bool ife = ib < sd.gfe;
    const float g = t.jfe ? (ife ? sd.law.GMassFeFe : sd.law.GMassFeSi) : (ife ? sd.law.GMassFeSi : 1.0f);

    float xi[R], yi[R], zi[R];
    float ax[R], ay[R], az[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float4 p = P[ib + r * 64 + lane];
        xi[r] = p.x;
        yi[r] = p.y;
        zi[r] = p.z;
        ax[r] = ay[r] = az[r] = 0.0f;
    }

    // The block's positions, twice, in wave-private LDS: q[m] holds
    // j_((127 - m) mod 64), so step k reads q[63 - lane + k] =
    // j_((lane - k) mod 64) -- the j whose accumulator lane `lane` holds
    // after k rotations -- at the immediate offset 16 k.
    if (t.diag) {
        // The row against itself, each pair once: its 64-blocks m holding a
        // real particle against the row's sub-blocks r < m (both sides, as
        // below), and against sub-block m itself over rotations 1..32 (lanes
        // 0..31 only at 32): every pair of the block exactly once, the self
        // pair never.  The j-side sums return to their lanes after 64
        // rotations and belong to sub-block m's particles.  A task takes the
        // blocks m of [j0, j1) (the planner may cut a row's diagonal in
        // pieces of about equal work, each with its own slot).
        const int m0 = (t.j0 - ib) >> 6, m1 = (t.j1 - ib) >> 6;
        for (int m = m0; m < m1; ++m) {
            const float4 own = P[ib + m * 64 + lane];
            wave_lds_sync();  // the previous block's reads are done
            q[63 - lane] = own;
            q[127 - lane] = own;
            wave_lds_sync();
            float xj = own.x, yj = own.y, zj = own.z;
            const float4* __restrict__ qb = q + (63 - lane);
            float fx = 0.0f, fy = 0.0f, fz = 0.0f;
#pragma unroll 4
            for (int k = 0; k < 64; ++k) {
                const float4 pn = qb[k + 1 < 64 ? k + 1 : 63];  // next step's j
                const bool self_on = (k >= 1 && k < 32) || (k == 32 && lane < 32);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (r > m || (r == m && !self_on)) continue;
                    const float dx = xj - xi[r];
                    const float dy = yj - yi[r];
                    const float dz = zj - zi[r];
                    if constexpr (!POT) {
                        const float s = fast_inv_r3(fast_r2(dx, dy, dz));
                        ax[r] = __builtin_fmaf(s, dx, ax[r]);
                        ay[r] = __builtin_fmaf(s, dy, ay[r]);
                        az[r] = __builtin_fmaf(s, dz, az[r]);
                        fx = __builtin_fmaf(s, dx, fx);
                        fy = __builtin_fmaf(s, dy, fy);
                        fz = __builtin_fmaf(s, dz, fz);
                    } else {
                        const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                        const float ri = (r2 > 0.0f && r2 < kGhostR2) ? __builtin_amdgcn_rsqf(r2) : 0.0f;
                        ax[r] += ri;
                        fx += ri;
                    }
                }
                xj = pn.x;
                yj = pn.y;
                zj = pn.z;
                fx = rotate_lanes(fx);
                if constexpr (!POT) {
                    fy = rotate_lanes(fy);
                    fz = rotate_lanes(fz);
                }
            }
            // The force on j is the negated sum; the potential is symmetric.
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r == m) {
                    if constexpr (!POT) {
                        ax[r] -= fx;
                        ay[r] -= fy;
                        az[r] -= fz;
                    } else {
                        ax[r] += fx;
                    }
                }
        }
    } else {
        const int first = (t.row + 1) * B;  // first j of the row's slab
        float4 nx = P[t.j0 + lane];
        for (int J0 = t.j0; J0 < t.j1; J0 += 64) {
            float xj = nx.x, yj = nx.y, zj = nx.z;
            wave_lds_sync();  // the previous block's reads are done
            q[63 - lane] = nx;
            q[127 - lane] = nx;
            wave_lds_sync();
            // next block's positions, in flight during this block
            nx = P[(J0 + 64 < t.j1 ? J0 + 64 : J0) + lane];
            const float4* __restrict__ qb = q + (63 - lane);
            float fx = 0.0f, fy = 0.0f, fz = 0.0f;
            // unroll 16: 1-2% faster than 8 at 14k-98k particles (measured)
#pragma unroll 16
            for (int k = 0; k < 64; ++k) {
                const float4 pn = qb[k + 1 < 64 ? k + 1 : 63];  // next step's j
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float dx = xj - xi[r];
                    const float dy = yj - yi[r];
                    const float dz = zj - zi[r];
                    if constexpr (!POT) {
                        const float s = fast_inv_r3(fast_r2(dx, dy, dz));
                        ax[r] = __builtin_fmaf(s, dx, ax[r]);
                        ay[r] = __builtin_fmaf(s, dy, ay[r]);
                        az[r] = __builtin_fmaf(s, dz, az[r]);
                        fx = __builtin_fmaf(s, dx, fx);
                        fy = __builtin_fmaf(s, dy, fy);
                        fz = __builtin_fmaf(s, dz, fz);
                    } else {
                        const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                        const float ri = (r2 > 0.0f && r2 < kGhostR2) ? __builtin_amdgcn_rsqf(r2) : 0.0f;
                        ax[r] += ri;
                        fx += ri;
                    }
                }
                xj = pn.x;
                yj = pn.y;
                zj = pn.z;
                fx = rotate_lanes(fx);
                if constexpr (!POT) {
                    fy = rotate_lanes(fy);
                    fz = rotate_lanes(fz);
                }
            }
            // After 64 rotations lane l holds j = J0 + l again.  The force on
            // j is the negated sum (dp points from j to the row particle);
            // the potential is symmetric.
            const long long o = (long long)(J0 - first) + lane;
            if constexpr (!POT) {
                J[3 * o] = -fx * g;
                J[3 * o + 1] = -fy * g;
                J[3 * o + 2] = -fz * g;
            } else {
                J[3 * o] = fx * g;
            }
        }
    }

    float* __restrict__ I = iside + (size_t)t.slot * (3 * B);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        I[3 * (r * 64 + lane)] = ax[r] * g;
        if constexpr (!POT) {
            I[3 * (r * 64 + lane) + 1] = ay[r] * g;
            I[3 * (r * 64 + lane) + 2] = az[r] * g;
        }
    }
}

template <int R, bool POT>
__global__ __launch_bounds__(64 * kMutualWaves) void k_mutual(const float4* __restrict__ gpos,
                                                              const MutualTask* __restrict__ tasks,
                                                              int ntasks, const SimDesc* __restrict__ sims,
                                                              float* __restrict__ iside,
                                                              float* __restrict__ jside) {
    constexpr int B = 64 * R;
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * kMutualWaves + wv);
    if (w >= ntasks) return;
    const MutualTask t = tasks[w];
    const SimDesc& sd = sims[t.sim];
    __shared__ float4 lq[kMutualWaves][128];
    float* __restrict__ J = jside + sd.jbase + 3 * jside_row_offset(t.row, sd.gn, B);
    mutual_wave_task<R, POT>(t, sd, gpos + sd.gbase, lq[wv], iside, J, lane);
}

// ---------------------------------------------------------------------------
// Pass 1, mutual form with row groups: the j-side sums of kMutualWaves rows
// added in LDS before they are written
// ---------------------------------------------------------------------------
//
// In k_mutual every (row, 64-block) pair leaves a j-side slab entry, so the
// slab holds ~N^2 / (128 R) floats per component -- more than the whole pass
// writes otherwise.  Here a workgroup's W = kMutualWaves wavefronts hold W
// consecutive rows (a group) and stream the same j-blocks beyond the group:
// the block's positions sit once in LDS for all of them, and after each block
// the W j-side sums (each times its own row's gravity product) are added in a
// fixed order and written as one entry per (group, block), a W-th of the
// entries.  Pairs inside a group (a row against itself and against the later
// rows of its group) are single-wavefront row tasks as in k_mutual, packed W
// to a workgroup, whose j-side sums go to a small per-row slab.
constexpr int kGroupRows = kMutualWaves;

template <int R, bool POT>
__device__ __forceinline__ void mutual_group_task(const GroupTask& gt, const SimDesc& sd,
                                                  const RowDesc* __restrict__ rows, const float4* __restrict__ P,
                                                  float* __restrict__ iside, float* __restrict__ jside, int wv,
                                                  int lane, float4 (*__restrict__ sq)[128],
                                                  float (*__restrict__ red)[3][kGroupRows][64]) {
    constexpr int B = 64 * R;
    constexpr int W = kGroupRows;
    const int nrows = sd.gn / B;
    const int row = gt.group * W + wv;
    const bool live = row < nrows;  // wave-uniform
    const int ib = row * B;
    const bool ife = ib < sd.gfe;
    const float g = !live ? 0.0f
                          : gt.jfe ? (ife ? sd.law.GMassFeFe : sd.law.GMassFeSi) : (ife ? sd.law.GMassFeSi : 1.0f);
    float xi[R], yi[R], zi[R];
    float ax[R], ay[R], az[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float4 p = live ? P[ib + r * 64 + lane] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        xi[r] = p.x;
        yi[r] = p.y;
        zi[r] = p.z;
        ax[r] = ay[r] = az[r] = 0.0f;
    }
    const int gend = min((gt.group + 1) * W, nrows) * B;  // first j of the group's slab
    float* __restrict__ J = jside + sd.jbase + 3 * jside_row_offset(gt.group, sd.gn, W * B);
    // Each wavefront stages a quarter of every block: lanes 0..15 of wave wv
    // own j = 16 wv + lane, stored twice as k_mutual lays a block out.
    const int jl = wv * 16 + (lane & 15);
    const bool stager = lane < 16;
    float4 nx = stager ? P[gt.j0 + jl] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (stager) {
        sq[0][63 - jl] = nx;
        sq[0][127 - jl] = nx;
    }
    __syncthreads();
    int buf = 0;
    for (int J0 = gt.j0; J0 < gt.j1; J0 += 64) {
        const bool more = J0 + 64 < gt.j1;
        if (more && stager) nx = P[J0 + 64 + jl];  // the next block's quarter, in flight
        float fx = 0.0f, fy = 0.0f, fz = 0.0f;
        if (live) {
            const float4* __restrict__ qb = sq[buf] + (63 - lane);
            const float4 c0 = qb[0];
            float xj = c0.x, yj = c0.y, zj = c0.z;
            // unroll 2: 1.7% faster than 8 at N = 262,144 and 2% on the
            // batched step; 4 and 16 in between, 1 slower (measured)
#pragma unroll 2
            for (int k = 0; k < 64; ++k) {
                const float4 pn = qb[k + 1 < 64 ? k + 1 : 63];  // next step's j
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float dx = xj - xi[r];
                    const float dy = yj - yi[r];
                    const float dz = zj - zi[r];
                    if constexpr (!POT) {
                        const float s = fast_inv_r3(fast_r2(dx, dy, dz));
                        ax[r] = __builtin_fmaf(s, dx, ax[r]);
                        ay[r] = __builtin_fmaf(s, dy, ay[r]);
                        az[r] = __builtin_fmaf(s, dz, az[r]);
                        fx = __builtin_fmaf(s, dx, fx);
                        fy = __builtin_fmaf(s, dy, fy);
                        fz = __builtin_fmaf(s, dz, fz);
                    } else {
                        const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                        const float ri = (r2 > 0.0f && r2 < kGhostR2) ? __builtin_amdgcn_rsqf(r2) : 0.0f;
                        ax[r] += ri;
                        fx += ri;
                    }
                }
                xj = pn.x;
                yj = pn.y;
                zj = pn.z;
                fx = rotate_lanes(fx);
                if constexpr (!POT) {
                    fy = rotate_lanes(fy);
                    fz = rotate_lanes(fz);
                }
            }
        }
        // This wavefront's j-side sums, times its own gravity product (the
        // force on j is the negated sum; the potential is symmetric).
        if constexpr (!POT) {
            red[buf][0][wv][lane] = -fx * g;
            red[buf][1][wv][lane] = -fy * g;
            red[buf][2][wv][lane] = -fz * g;
        } else {
            red[buf][0][wv][lane] = fx * g;
        }
        if (more && stager) {
            sq[buf ^ 1][63 - jl] = nx;
            sq[buf ^ 1][127 - jl] = nx;
        }
        __syncthreads();
        // wavefront c adds component c over the group's rows in row order
        if (wv < (POT ? 1 : 3)) {
            float a = red[buf][wv][0][lane];
#pragma unroll
            for (int w = 1; w < W; ++w) a += red[buf][wv][w][lane];
            J[3 * ((J0 - gend) + lane) + wv] = a;
        }
        buf ^= 1;
    }
    if (live) {
        float* __restrict__ I = iside + (size_t)(rows[sd.row0 + row].slot0 + gt.piece) * (3 * B);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            I[3 * (r * 64 + lane)] = ax[r] * g;
            if constexpr (!POT) {
                I[3 * (r * 64 + lane) + 1] = ay[r] * g;
                I[3 * (r * 64 + lane) + 2] = az[r] * g;
            }
        }
    }
}

// Six wavefronts per SIMD (at most 80 VGPRs; R = 8 needs a few more
// unconstrained, and the compiler spills two or three values outside the
// inner loop): 2.5% faster at N = 262,144 than five.
template <int R, bool POT>
__global__ __launch_bounds__(64 * kMutualWaves) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_mutual_grp(
    const float4* __restrict__ gpos, const GroupTask* __restrict__ gtasks, int ntasks,
    const MutualTask* __restrict__ rtasks, const SimDesc* __restrict__ sims, const RowDesc* __restrict__ rows,
    float* __restrict__ iside, float* __restrict__ jside, float* __restrict__ jintra) {
    constexpr int B = 64 * R;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if ((int)blockIdx.x >= ntasks) return;
    const GroupTask gt = gtasks[blockIdx.x];
    __shared__ float4 lq[kMutualWaves][128];
    __shared__ float red[2][3][kGroupRows][64];
    if (gt.kind == 1) {
        const MutualTask t = rtasks[gt.rtask0 + wv];
        if (t.j1 <= t.j0) return;  // a filler of the last workgroup
        const SimDesc& sd = sims[t.sim];
        float* __restrict__ J = jintra + sd.jibase + 3LL * (kGroupRows - 1) * B * t.row;
        mutual_wave_task<R, POT>(t, sd, gpos + sd.gbase, lq[wv], iside, J, lane);
        return;
    }
    const SimDesc& sd = sims[gt.sim];
    mutual_group_task<R, POT>(gt, sd, rows, gpos + sd.gbase, iside, jside, wv, lane,
                              reinterpret_cast<float4(*)[128]>(&lq[0][0]), red);
}

// Binary search of the simulation owning padded slot q (sims ordered by gbase).
__device__ __forceinline__ int find_gsim(const SimDesc* __restrict__ sims, int nsims, int q) {
    int lo = 0, hi = nsims - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sims[mid].gbase <= q)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Padded layout of the mutual pass: per simulation, iron [0, gfe) then
// silicate [gfe, gn); slots past a segment's particles are ghosts.
__global__ void k_mutual_pad(const float4* __restrict__ pos, int gtot, const SimDesc* __restrict__ sims,
                             int nsims, float4* __restrict__ gpos) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= gtot) return;
    const SimDesc& sd = sims[find_gsim(sims, nsims, q)];
    const int u = q - sd.gbase;
    int src = -1;
    if (u < sd.gfe) {
        if (u < sd.fe_end - sd.start) src = sd.start + u;
    } else if (u - sd.gfe < sd.end - sd.fe_end) {
        src = sd.fe_end + (u - sd.gfe);
    }
    gpos[q] = src >= 0 ? pos[src] : make_float4(kGhostCoord, kGhostCoord, kGhostCoord, 0.0f);
}

// Per particle: the i-side slots of its row and the j-side entries of every
// earlier row (k_mutual), or of every earlier group and the earlier rows of
// its own group (k_mutual_grp, groups of W rows), added in compensated
// float sums (CompSum) in a fixed order.  A workgroup takes 64 padded
// places of one row (a SumBlock; the host lists the blocks holding a real
// particle, heaviest rows first), so the loop bounds are uniform.  Four
// wavefronts per block: wavefront w adds the w-th quarter of each particle's
// slots and slab entries (one particle per lane, so the loads stay
// coalesced), and the quarters are added in LDS in a fixed order -- four
// times the loads in flight of one thread per particle.
// With corr (the contact corrections of k_contact_corr), the correction plus
// the sum rounded to float goes to force.xyz -- k_finish's arithmetic --
// and, with mpos / mvel, the particle then takes the move's step (k_move's,
// k_move_collision's or k_move_damped_separate's arithmetic) with mv; with
// gpos, the moved position also goes to its padded place, so that the next
// step of the same run needs no k_mutual_pad (two separate bodies of 15,000
// particles: 148.3 us a step with a move kernel and a padded copy of their
// own, 142.6 fused; one simulation of 21,000, whose move was fused before,
// 115 and 114).  Without corr, the sum goes to gsum for k_finish /
// k_finish_potential.
// Bound by the entries' bytes: 102 us at N = 262,144 (5.1 TB/s), 28 us at
// 65,536.  Below, where a few loads in turn are all of it, one load of the
// workgroup's descriptor instead of three in turn and the particle's state
// asked for before the entries: 6.2 us -> 5.0 at N = 13,255.  Two or sixteen
// entries in flight, or eight or sixteen wavefronts per block: the same
// within 5% at every size.
constexpr int kSumSplit = 4;

// Move constants of a move fused into k_mutual_sum: one set for the call, or
// each SimDesc's own (the batched engine), or the damped move's with its
// borders (k_move_damped_separate).
enum SumMoveKind { kMoveOne = 0, kMovePerSim = 1, kMoveDamped = 2 };
struct SumMove {
    float dt, dt_over_mass_fe, dt_over_mass_si;
    int kind;
    int b1, b2, b3;
    float damp1, damp2;
};

// A wavefront's part of a particle's entries (its quarters of the slots, of
// the earlier groups' slab entries and of the earlier rows of its group, one
// after the other) are one list: the loads of kSumBatch entries are issued
// before their additions, whatever list they are of, and so are those of the
// entries left over, so a list costs one round trip to memory per kSumBatch
// entries.  The additions keep their order.
constexpr int kSumBatch = 8;

// Entries k .. k + M - 1: at(k)'s record holds lane 0's (x, y, z), lane l's
// is 3 l further, so a wavefront reads 768 contiguous bytes per entry.  POT:
// x only.
template <int M, bool POT, typename At>
__device__ __forceinline__ void add_entries(int k, int lane, At at, CompSum& sx, CompSum& sy, CompSum& sz) {
    float vx[M], vy[M], vz[M];
#pragma unroll
    for (int u = 0; u < M; ++u) {
        const float* e = at(k + u) + 3 * lane;
        vx[u] = e[0];
        if constexpr (!POT) {
            vy[u] = e[1];
            vz[u] = e[2];
        }
    }
#pragma unroll
    for (int u = 0; u < M; ++u) {
        sx.add(vx[u]);
        if constexpr (!POT) {
            sy.add(vy[u]);
            sz.add(vz[u]);
        }
    }
}

template <bool POT>
__global__ __launch_bounds__(64 * kSumSplit) void k_mutual_sum(const SumBlock* __restrict__ blocks,
                                                              const SimDesc* __restrict__ sims, int B, int W,
                                                              const float* __restrict__ iside,
                                                              const float* __restrict__ jside,
                                                              const float* __restrict__ jintra,
                                                              float4* __restrict__ gsum,
                                                              const float* __restrict__ corr, int ntot,
                                                              float4* __restrict__ force,
                                                              float4* __restrict__ mpos,
                                                              float4* __restrict__ mvel,
                                                              float4* __restrict__ gpos, SumMove mv) {
    __shared__ float red[3][2][kSumSplit][64];  // per component: sum and compensation of each quarter
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: the addresses below stay scalar
    const SumBlock blk = blocks[blockIdx.x];
    const bool real = lane < blk.nreal;
    const int i = blk.i0 + lane;
    // what the last step needs, on its way beside the entries
    float2 rx = {}, ry = {}, rz = {};
    float4 v = {}, p = {};
    if (w == 0 && real && corr) {
        const float2* rec = reinterpret_cast<const float2*>(corr + 6 * (size_t)i);
        rx = rec[0];
        ry = rec[1];
        rz = rec[2];
        if (mpos) {
            v = mvel[i];
            p = mpos[i];
        }
    }
    CompSum sx, sy, sz;
    sx.zero();
    sy.zero();
    sz.zero();
    const int sl0 = blk.nslot * w / kSumSplit, gr0 = blk.group * w / kSumSplit, in0 = blk.in_group * w / kSumSplit;
    const int nsl = blk.nslot * (w + 1) / kSumSplit - sl0;
    const int nsg = nsl + blk.group * (w + 1) / kSumSplit - gr0;
    const int n = nsg + blk.in_group * (w + 1) / kSumSplit - in0;
    const float* const slots = iside + (size_t)(blk.slot0 + sl0) * (3 * B) + 3 * (blk.q0 % B);
    const float* const groups = jside + blk.jfirst;
    const long long istep = 3 * ((long long)(W - 1) * B - B);
    const float* const inner = jintra + blk.ifirst + istep * in0;
    // the record of entry k for lane 0 (wavefront-uniform); lane l's is 3 l further
    auto at = [&](int k) {
        const float* const a0 = slots + (size_t)k * (3 * B);
        const float* const a1 = groups + 3 * sum_group_offset(gr0 + k - nsl, blk.gn, (long long)W * B);
        const float* const a2 = inner + istep * (k - nsg);
        const float* const a12 = k < nsg ? a1 : a2;
        return k < nsl ? a0 : a12;
    };
    if (real) {
        int k = 0;
        for (; k + kSumBatch <= n; k += kSumBatch) add_entries<kSumBatch, POT>(k, lane, at, sx, sy, sz);
        switch (n - k) {
            case 7: add_entries<7, POT>(k, lane, at, sx, sy, sz); break;
            case 6: add_entries<6, POT>(k, lane, at, sx, sy, sz); break;
            case 5: add_entries<5, POT>(k, lane, at, sx, sy, sz); break;
            case 4: add_entries<4, POT>(k, lane, at, sx, sy, sz); break;
            case 3: add_entries<3, POT>(k, lane, at, sx, sy, sz); break;
            case 2: add_entries<2, POT>(k, lane, at, sx, sy, sz); break;
            case 1: add_entries<1, POT>(k, lane, at, sx, sy, sz); break;
            default: break;
        }
    }
    red[0][0][w][lane] = sx.s;
    red[0][1][w][lane] = sx.c;
    red[1][0][w][lane] = sy.s;
    red[1][1][w][lane] = sy.c;
    red[2][0][w][lane] = sz.s;
    red[2][1][w][lane] = sz.c;
    __syncthreads();
    if (w == 0 && real) {
        // the quarters in order; their compensations join the total's
        CompSum ax, ay, az;
        ax.zero();
        ay.zero();
        az.zero();
#pragma unroll
        for (int k = 0; k < kSumSplit; ++k) {
            ax.add(red[0][0][k][lane]);
            ax.c += red[0][1][k][lane];
            ay.add(red[1][0][k][lane]);
            ay.c += red[1][1][k][lane];
            az.add(red[2][0][k][lane]);
            az.c += red[2][1][k][lane];
        }
        if (corr) {
            // k_finish's arithmetic: the correction's (sum, compensation)
            // pair plus the all-pairs sum rounded to float, rounded once
            CompSum cx{rx.x, rx.y}, cy{ry.x, ry.y}, cz{rz.x, rz.y};
            cx.add(ax.value());
            cy.add(ay.value());
            cz.add(az.value());
            const float fx = cx.value(), fy = cy.value(), fz = cz.value();
            force[i].x = fx;
            force[i].y = fy;
            force[i].z = fz;
            if (mpos) {
                const SimDesc& sd = sims[blk.sim];
                const bool own = mv.kind == kMovePerSim;
                const float dt = own ? sd.dt : mv.dt;
                const float dtm_fe = own ? sd.dt_over_mass_fe : mv.dt_over_mass_fe;
                const float dtm_si = own ? sd.dt_over_mass_si : mv.dt_over_mass_si;
                if (mv.kind == kMoveDamped) {
                    const bool second = mv.b3 <= i || mv.b2 <= i;
                    const bool si = mv.b3 <= i || (mv.b2 > i && mv.b1 <= i);
                    const float temp = si ? dtm_si : dtm_fe, damp = second ? mv.damp2 : mv.damp1;
                    v.x += (fx - damp * v.x) * temp;
                    v.y += (fy - damp * v.y) * temp;
                    v.z += (fz - damp * v.z) * temp;
                } else {
                    const float temp = blk.iron ? dtm_fe : dtm_si;
                    v.x += fx * temp;
                    v.y += fy * temp;
                    v.z += fz * temp;
                }
                p.x += v.x * dt;
                p.y += v.y * dt;
                p.z += v.z * dt;
                mvel[i] = v;
                mpos[i] = p;
                if (gpos) gpos[sd.gbase + blk.q0 + lane] = p;
            }
        } else {
            gsum[i] = make_float4(ax.value(), ay.value(), az.value(), 0.0f);
        }
    }
}

// ---------------------------------------------------------------------------
// Pass 2: spatial hash of unit cells (counting sort, deterministic buckets)
// ---------------------------------------------------------------------------

__global__ void k_fill_int(int* __restrict__ a, int n, int v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// The grid takes five launches (it can be the critical path beside the pair
// kernel of a mid-size plan, where each launch of a chain is 5 us): the
// buckets' counts with each particle's place of arrival in its bucket; the
// scan of every 1,024 counts, which leaves them at zero for the next grid;
// the scan of the block totals; the particles at their places; and each
// particle at its rank by id among its bucket's, with its position and
// velocity.  (Cleared, counted, scanned in three launches, scattered, sorted
// a bucket per lane and gathered took eight; the block totals summed by every
// workgroup of k_grid_place for itself took its 256 lanes and their barriers
// 50 us beside a running pair kernel.)
__global__ void k_grid_count(const float4* __restrict__ pos, int ntot, const SimDesc* __restrict__ sims,
                             int nsims, int* __restrict__ counts, int2* __restrict__ place) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntot) return;
    const SimDesc& sd = sims[find_sim(sims, nsims, i)];
    float4 p = pos[i];
    unsigned h = cell_bucket(sd.hbase, sd.hmask, cell_coord(p.x), cell_coord(p.y), cell_coord(p.z));
    place[i] = make_int2((int)h, atomicAdd(&counts[h], 1));
}

// Exclusive scan of in[0..m) into out[0..m], 1024 elements per block; CLEAR
// leaves in[] at zero.
template <bool CLEAR>
__global__ __launch_bounds__(256) void k_scan_blocks(int* __restrict__ in, int m, int* __restrict__ out,
                                                     int* __restrict__ block_sums) {
    __shared__ int sh[256];
    const int base = blockIdx.x * 1024 + threadIdx.x * 4;
    int v[4];
    int local = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = (base + k < m) ? in[base + k] : 0;
        if (CLEAR && base + k < m) in[base + k] = 0;
        local += v[k];
    }
    sh[threadIdx.x] = local;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        int add = threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += add;
        __syncthreads();
    }
    int run = sh[threadIdx.x] - local;  // exclusive prefix of this thread
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (base + k < m) out[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 255) block_sums[blockIdx.x] = sh[255];
}

// Exclusive scan of the block sums in one workgroup of kScanTopThreads
// threads, 16 sums each (nb <= 4096).  The workgroup is kept to one
// wavefront per SIMD: it runs on a side stream beside the pair kernel, and a
// 1,024-thread workgroup (four wavefronts on every SIMD of one CU) waited
// for a CU to drain for most of the pair kernel's run.
constexpr int kScanTopThreads = 256;
__global__ __launch_bounds__(kScanTopThreads) void k_scan_top(int* __restrict__ block_sums, int nb,
                                                              int* __restrict__ total_out) {
    constexpr int T = kScanTopThreads, E = 4096 / kScanTopThreads;
    __shared__ int sh[T];
    const int base = threadIdx.x * E;
    int v[E];
    int local = 0;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        v[k] = (base + k < nb) ? block_sums[base + k] : 0;
        local += v[k];
    }
    sh[threadIdx.x] = local;
    __syncthreads();
    for (int off = 1; off < T; off <<= 1) {
        int add = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += add;
        __syncthreads();
    }
    int run = sh[threadIdx.x] - local;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        if (base + k < nb) block_sums[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == T - 1) *total_out = sh[T - 1];
}

__global__ void k_scan_add(int* __restrict__ out, int m, const int* __restrict__ block_sums) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) out[i] += block_sums[i >> 10];
}

// The bucket offsets of the whole grid (starts[0..m)) and the particle ids at
// their places of arrival (slots), from the scan's blocks (lstarts,
// block_sums): buckets and particles are dealt out over one grid.
__global__ void k_grid_place(int ntot, int m, const int* __restrict__ lstarts, const int* __restrict__ block_sums,
                             const int2* __restrict__ place, int* __restrict__ starts, int* __restrict__ slots) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) starts[t] = lstarts[t] + block_sums[t >> 10];
    if (t < ntot) {
        const int2 p = place[t];
        slots[lstarts[p.x] + block_sums[p.x >> 10] + p.y] = t;
    }
}

// Each particle at its rank by id among its bucket's particles, so that the
// contact sums run in a fixed order, with its position and velocity: the
// contact pass reads the particles of a cell from consecutive memory.
__global__ void k_grid_rank(int ntot, const int* __restrict__ slots, const int2* __restrict__ place,
                            const int* __restrict__ starts, const float4* __restrict__ pos,
                            const float4* __restrict__ vel, int* __restrict__ sorted, float4* __restrict__ spos,
                            float4* __restrict__ svel) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntot) return;
    const int i = slots[t];
    const int h = place[i].x;
    const int s = starts[h], e = starts[h + 1];
    int at = s;
    for (int k = s; k < e; ++k) at += slots[k] < i;
    sorted[at] = i;
    spos[at] = pos[i];
    if (svel) svel[at] = vel[i];
}

// ---------------------------------------------------------------------------
// Pass 3: chunk sums + exact contact correction
// ---------------------------------------------------------------------------

// The contact correction of a particle, for every pair with r < 1 found
// through the grid: the reference's exact contact term minus what the
// all-pairs pass added for that pair.  Contact terms are rounded exactly as
// the reference rounds them (float products of a float magnitude); each
// term and each gravity term subtracted goes into a compensated float sum,
// so cancellation between large contact forces adds no summation error.
//
// The 27-cell walk is a chain of dependent loads (bucket bounds, then each
// candidate).  It is cut into the nine rows of three cells (oz, oy) =
// (r / 3 - 1, r % 3 - 1), r = 0..8; each row is summed from zero (cells in x
// order, candidates in bucket order) and the nine row sums are added in row
// order.  LANES = 9 walks the rows of a particle on nine lanes at once (seven
// particles per wavefront, the row sums added through LDS): a chain a ninth
// as long, for plans too small to hide the walk behind the all-pairs pass.
// LANES = 1 walks them in turn on one lane.  The arithmetic is the same, so
// the two forms give bitwise the same corrections.  No candidate's cell is
// looked at: a bucket may hold particles of other cells, but the 27 cells
// have 27 buckets (a simulation has at least 4 x 4 x 4), a pair with r < 1
// lies in adjacent cells (coordinates a unit apart or more round to a
// difference of one or more), and so it is met in one bucket alone.  A simulation's buckets
// hold only its own particles, and the particle itself sits at position t,
// so a candidate's index is loaded only for a pair in contact.
constexpr int kCellRows = 9;
constexpr int kContactWaves = 4;  // wavefronts per workgroup

__device__ __forceinline__ void contact_row(const SimDesc& sd, int t, int i, int row,
                                            const int* __restrict__ starts, const int* __restrict__ sorted,
                                            const float4* __restrict__ spos, const float4* __restrict__ svel,
                                            int variant, CompSum& ex, CompSum& ey, CompSum& ez) {
    const float4 pi = spos[t];
    const float4 vi = svel[t];
    const int ccx = cell_coord(pi.x), ccy = cell_coord(pi.y), ccz = cell_coord(pi.z);
    const bool ife = i < sd.fe_end;
    const int qy = ccy + row % 3 - 1, qz = ccz + row / 3 - 1;
    int b0[3], b1[3];
#pragma unroll
    for (int ox = 0; ox < 3; ++ox) {
        const unsigned h = cell_bucket(sd.hbase, sd.hmask, ccx + ox - 1, qy, qz);
        b0[ox] = starts[h];
        b1[ox] = starts[h + 1];
    }
#pragma unroll
    for (int ox = 0; ox < 3; ++ox) {
        for (int k = b0[ox]; k < b1[ox]; ++k) {
            const float4 pj = spos[k];
            if (k == t) continue;  // i itself
            const float dpx = pj.x - pi.x;
            const float dpy = pj.y - pi.y;
            const float dpz = pj.z - pi.z;
            const float r2 = dpx * dpx + dpy * dpy + dpz * dpz;
            if (1.0f <= r2) continue;  // then sqrtf(r2) >= 1 too: the root only for candidates that may touch
            const float r = sqrtf(r2);
            if (1.0f <= r) continue;
            const float invr = 1.0f / r;
            const int j = sorted[k];
            const int test = (int)ife + (int)(j < sd.fe_end);
            const float4 vj = svel[k];
            const float dvx = vj.x - vi.x, dvy = vj.y - vi.y, dvz = vj.z - vi.z;
            const float dot = dpx * dvx + dpy * dvy + dpz * dvz;
            const float fm = contact_pair_mag(sd.law, test, r, r2, dot);
            // The contact term minus what pass 1 added for this pair (for
            // r < 1 a bounded placeholder: |sf dp| < g), one addition each.
            const float g = gravity_product(sd.law, test);
            const float sf = g * inv_r3_variant(variant, fast_r2(dpx, dpy, dpz));
            ex.add(fm * dpx * invr - sf * dpx);
            ey.add(fm * dpy * invr - sf * dpy);
            ez.add(fm * dpz * invr - sf * dpz);
        }
    }
}

// Particles per wavefront of the contact walk.
template <int LANES>
__host__ __device__ constexpr int contact_per_wave() {
    return LANES == 1 ? 64 : 64 / LANES;
}

// Workgroups of k_finish / k_contact_corr for ntot particles.
template <int LANES>
__host__ __device__ constexpr int contact_blocks(int ntot) {
    return (ntot + kContactWaves * contact_per_wave<LANES>() - 1) / (kContactWaves * contact_per_wave<LANES>());
}

// The lane's particle (bucket position t, index i, simulation s; t = -1 for
// none) and, on the lane that owns the result (`lead`), its correction.
struct ContactLane {
    int t, i, s;
    bool lead;
    CompSum ex, ey, ez;  // the correction as an unrounded (sum, compensation) pair
};

template <int LANES>
__device__ __forceinline__ ContactLane contact_correction(int ntot, const SimDesc* __restrict__ sims, int nsims,
                                                          const int* __restrict__ starts,
                                                          const int* __restrict__ sorted,
                                                          const float4* __restrict__ spos,
                                                          const float4* __restrict__ svel, int variant) {
    static_assert(LANES == 1 || LANES == kCellRows, "one lane per particle or one per cell row");
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int slot = lane / LANES;  // LANES = 9: 0..6, and 7 for the idle lane 63
    const int row = LANES == 1 ? 0 : lane % LANES;
    ContactLane c;
    c.t = slot < contact_per_wave<LANES>()
              ? (blockIdx.x * kContactWaves + w) * contact_per_wave<LANES>() + slot
              : -1;
    if (c.t >= ntot) c.t = -1;
    c.i = c.t >= 0 ? sorted[c.t] : 0;
    c.s = c.t >= 0 ? find_sim(sims, nsims, c.i) : 0;
    const bool live = c.t >= 0 && sims[c.s].active;
    // each row summed from zero, then the nine rows' (sum, compensation)
    // pairs added in row order (the same arithmetic on one lane or nine)
    c.ex.zero();
    c.ey.zero();
    c.ez.zero();
    if constexpr (LANES == 1) {
        c.lead = live;
        if (live)
            for (int r = 0; r < kCellRows; ++r) {
                CompSum rx, ry, rz;
                rx.zero();
                ry.zero();
                rz.zero();
                contact_row(sims[c.s], c.t, c.i, r, starts, sorted, spos, svel, variant, rx, ry, rz);
                c.ex.add_sum(rx);
                c.ey.add_sum(ry);
                c.ez.add_sum(rz);
            }
    } else {
        __shared__ float part[kContactWaves][6][64];
        CompSum rx, ry, rz;
        rx.zero();
        ry.zero();
        rz.zero();
        if (live) contact_row(sims[c.s], c.t, c.i, row, starts, sorted, spos, svel, variant, rx, ry, rz);
        part[w][0][lane] = rx.s;
        part[w][1][lane] = rx.c;
        part[w][2][lane] = ry.s;
        part[w][3][lane] = ry.c;
        part[w][4][lane] = rz.s;
        part[w][5][lane] = rz.c;
        __syncthreads();
        c.lead = live && row == 0;
        if (c.lead) {
#pragma unroll
            for (int r = 0; r < kCellRows; ++r) {
                c.ex.add(part[w][0][lane + r]);
                c.ex.c += part[w][1][lane + r];
                c.ey.add(part[w][2][lane + r]);
                c.ey.c += part[w][3][lane + r];
                c.ez.add(part[w][4][lane + r]);
                c.ez.c += part[w][5][lane + r];
            }
        }
    }
    return c;
}

// Threads walk the particles in bucket (Morton) order: the lanes of a
// wavefront look up the same and adjacent cells.
template <int LANES>
__global__ __launch_bounds__(64 * kContactWaves) void k_finish(float4* __restrict__ force, int ntot,
                                                               const SimDesc* __restrict__ sims, int nsims,
                                                               const float4* __restrict__ partial,
                                                               const float4* __restrict__ gsum,
                                                               const int* __restrict__ starts,
                                                               const int* __restrict__ sorted,
                                                               const float4* __restrict__ spos,
                                                               const float4* __restrict__ svel, int variant) {
    const ContactLane c = contact_correction<LANES>(ntot, sims, nsims, starts, sorted, spos, svel, variant);
    if (!c.lead) return;
    const SimDesc& sd = sims[c.s];
    const int i = c.i;
    const int n = sd.end - sd.start;
    // the correction's pair plus the all-pairs sums, rounded once
    CompSum fx = c.ex, fy = c.ey, fz = c.ez;
    if (gsum && sd.gn > 0) {
        // mutual pass: already summed per particle
        const float4 gs = gsum[i];
        fx.add(gs.x);
        fy.add(gs.y);
        fz.add(gs.z);
    } else {
        for (int ch = 0; ch < sd.nchunk; ++ch) {
            float4 p = partial[sd.partial_base + ch * n + (i - sd.start)];
            fx.add(p.x);
            fy.add(p.y);
            fz.add(p.z);
        }
    }
    force[i].x = fx.value();
    force[i].y = fy.value();
    force[i].z = fz.value();
}

// The contact corrections alone, into corr (per particle, by index, one
// 24-byte record: the (sum, compensation) pairs of x, y and z -- the lanes
// walk in bucket order, so one record per lane keeps each store to one or
// two cache lines), for plans whose simulations all take the mutual pass:
// it needs only the grid, so it runs beside the all-pairs pass, and
// k_mutual_sum adds it to the sums -- the same arithmetic as k_finish.
template <int LANES>
__global__ __launch_bounds__(64 * kContactWaves) void k_contact_corr(int ntot, const SimDesc* __restrict__ sims,
                                                                     int nsims, const int* __restrict__ starts,
                                                                     const int* __restrict__ sorted,
                                                                     const float4* __restrict__ spos,
                                                                     const float4* __restrict__ svel, int variant,
                                                                     float* __restrict__ corr) {
    const ContactLane c = contact_correction<LANES>(ntot, sims, nsims, starts, sorted, spos, svel, variant);
    if (!c.lead) return;
    float2* rec = reinterpret_cast<float2*>(corr + 6 * (size_t)c.i);
    rec[0] = make_float2(c.ex.s, c.ex.c);
    rec[1] = make_float2(c.ey.s, c.ey.c);
    rec[2] = make_float2(c.ez.s, c.ez.c);
}

// ---------------------------------------------------------------------------
// Direct pass: the whole force of a small simulation in one launch
// ---------------------------------------------------------------------------
//
// For small N the three passes above are bound by their dozen launches, not by
// arithmetic.  k_direct computes the same force in one.  A workgroup holds
// kDirectI i-particles, their positions wave-uniform (scalar registers); its
// wavefronts deal out the simulation's 64-blocks of j, a j per lane, so that a
// block's positions are one coalesced load for 64 kDirectI pairs and a step
// is kDirectI independent chains.  (With the lanes over i and the j's
// broadcast to them, each 64 pairs took a 16-byte load per lane: 16 cycles of
// a CU's load path, which bounded the kernel: a step of N = 2,048, 4,096,
// 8,192 and 11,000 took 12.0, 20.1, 49.7 and 116 us, and takes 7.8, 12.7,
// 29.7 and 50.8.)  It is bound by vector issue, 16 instructions per 64 pairs,
// at the large end (11,000: 70% of the issue rate) and by the chain of loads,
// step, contact terms and sums at the small end.  A wavefront's j are of one
// material (the wavefronts are divided between the iron and the silicate j),
// so the gravity product is one factor per wavefront and i.  Every pair takes
// the all-pairs pass's branch-free gravity term into a float sum per lane and
// i, of at most kDirectFold terms; four lanes' sums are added in float, all
// beyond in FP64.
//
// Pairs with r^2 < 1 are listed as they are met, in j order, one list per
// wavefront; a full list and at the end what is left is worked off a pair per
// lane: the exact contact term minus the gravity term, with the arithmetic of
// k_finish, added in FP64.  The wavefronts' sums are added in FP64 in a fixed
// order and rounded once, so the result depends on the simulation alone.
// (64 lanes folded in float and the contact terms of a batch too, with
// compensated sums between: the whole error, which v_rsq sets, was 1.0 to
// 1.9% larger in contact states and up to 0.15% in others, N = 300 to 12,288,
// than with every sum compensated; as it is, within 0.1% of that.  FP64 costs
// 0.2 us a call up to N = 2,048 and 2.5 to 4% above.)
//
// Eight wavefronts per workgroup, so that another has room beside the running
// ones: a call takes 5.7, 7.0, 10.4 and 19.3 us at N = 1,024, 2,048, 3,072 and
// 6,000 (before the FP64 sums 5.5, 6.8, 9.9 and 18.5, and with 16 wavefronts
// 5.8, 6.7, 11.7 and 23.5; four were slower up to 8,192 and even above).
constexpr int kDirectI = 8;
constexpr int kDirectForceWaves = 8;
// r^2 (with FMAs and kSelfEps) of every pair whose exactly rounded r is below
// 1 lies below this: the margin covers the few ulps between the two forms.
constexpr float kDirectContactR2 = 1.0001f;
// 64-blocks a wavefront's float sums run over.
constexpr int kDirectFold = 64;

// The move of a step fused into the direct pass (MOVE = 1:
// moveBodiesCollisionSingleGPU, impactAddTime.cu:379-394; MOVE = 2:
// moveBodiesDampedSeperate, generateTargetImpactor.cu:628-664), with the
// same arithmetic as k_move_collision / k_move_damped_separate.  The new
// state goes to other arrays (pout, vout): the pass still reads the old
// positions of every particle.  MOVE = 1 reads b1 as NFe.
struct FusedMove {
    float4* pout;
    float4* vout;
    float dt, dt_over_mass_fe, dt_over_mass_si;
    int b1, b2, b3;
    float damp1, damp2;
};

template <int CTRL>
__device__ __forceinline__ float lane_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double lane_dpp(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true));
}
// The lower 32 lanes get x of themselves plus x of lane + 32, the upper 32 y of
// lane - 32 plus y of themselves; for SPAN = 16, of each pair of rows of lanes.
template <int SPAN>
__device__ __forceinline__ double halves_sum(double x, double y) {
    if constexpr (SPAN == 32) {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false, false);
        return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
    } else {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(x), __double2loint(y), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(x), __double2hiint(y), false, false);
        return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
    }
}
// lanes with `hi` keep y and send x to their partner, the others keep x
template <int CTRL>
__device__ __forceinline__ float lane_fold(float x, float y, bool hi) {
    const float keep = hi ? y : x, send = hi ? x : y;
    return keep + lane_dpp<CTRL>(send);
}
// x[k] summed over the 16 lanes of each row of lanes; lane p of the row gets
// the sum of x[p & 7].  Four lanes' sums are added in float, then FP64.
__device__ __forceinline__ double row_sums8(const float (&x)[8], int p) {
    float a[4], b[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = lane_fold<0x141>(x[k], x[k + 4], p & 4);  // lane p with 7 - p of its half row
#pragma unroll
    for (int k = 0; k < 2; ++k) b[k] = lane_fold<0x4E>(a[k], a[k + 2], p & 2);  // with p ^ 2
    const bool hi = p & 1;
    const double c = (double)(hi ? b[1] : b[0]) + (double)lane_dpp<0xB1>(hi ? b[0] : b[1]);  // with p ^ 1
    return c + lane_dpp<0x128>(c);                                                           // with p ^ 8
}
// The four rows' x, y and z added: row 0 gets x, row 1 y, row 2 z.
__device__ __forceinline__ double rows_sum_xyz(double x, double y, double z) {
    return halves_sum<16>(halves_sum<32>(x, z), halves_sum<32>(y, 0.0));
}

// x summed over the lanes 8 p + k of each k, on every lane.
__device__ __forceinline__ double eighths_sum(double x) {
    x += lane_dpp<0x128>(x);
    x = halves_sum<16>(x, x);
    return halves_sum<32>(x, x);
}

// Four float4 records in one load.
typedef float Float16 __attribute__((ext_vector_type(16), aligned(16)));

template <int MOVE>
__global__ __launch_bounds__(64 * kDirectForceWaves) void k_direct(const float4* __restrict__ pos,
                                                   const float4* __restrict__ vel,
                                                   const DirectBlock* __restrict__ blocks, int per_log2,
                                                   const SimDesc* __restrict__ sims, float4* __restrict__ force,
                                                   FusedMove mv) {
    constexpr int W = kDirectForceWaves;
    static_assert(W == 8, "a wavefront's eight lanes per particle add the wavefronts' sums");
    constexpr int IB = kDirectI;
    constexpr int kWorkOff = 128;             // listed pairs that are worked off before the next step
    constexpr int kList = kWorkOff + 64 * IB;  // and what one step can add
    __shared__ double grav[W][4 * 16];    // per wavefront: row c, lane p -> component c of i p
    __shared__ double contact[W][3][IB];
    __shared__ int list[W][kList];        // i << 24 | j
    __shared__ float4 term[W][64];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const DirectBlock blk = blocks[blockIdx.x >> per_log2];
    const int i0 = blk.i0 + IB * (blockIdx.x & ((1u << per_log2) - 1u));
    const int start = blk.start, fe_end = blk.fe_end, end = blk.end;
    const SimDesc& sd = sims[blk.sim];
    if (i0 >= end) return;
    // the wavefronts that take iron j: their share of the 64-blocks
    const int wf = blk.iron_waves;
    const bool jfe = wv < wf;
    const int je = jfe ? fe_end : end;
    const int stride = 64 * (jfe ? wf : W - wf);
    int jb = jfe ? start + 64 * wv : fe_end + 64 * (wv - wf);  // the step's 64-block
    float4 nx = pos[min(jb + lane, end - 1)];
    // Of every workgroup but a simulation's last, one run of records in two
    // scalar loads: eight queue behind those of the CU's other wavefronts.
    // N = 4,096: 12.4 us a call, 11.4 so; 11,000: 50.7 and 49.2, with nothing
    // divided and the results' operands asked for before the barrier.
    float xi[IB], yi[IB], zi[IB];
    if (i0 + IB <= end) {
        const Float16* __restrict__ run = reinterpret_cast<const Float16*>(pos + i0);
        const Float16 a = run[0], b = run[1];
#pragma unroll
        for (int k = 0; k < IB; ++k) {
            xi[k] = k < 4 ? a[4 * (k & 3)] : b[4 * (k & 3)];
            yi[k] = k < 4 ? a[4 * (k & 3) + 1] : b[4 * (k & 3) + 1];
            zi[k] = k < 4 ? a[4 * (k & 3) + 2] : b[4 * (k & 3) + 2];
        }
    } else {
#pragma unroll
        for (int k = 0; k < IB; ++k) {
            const float4 p = pos[min(i0 + k, end - 1)];
            xi[k] = p.x;
            yi[k] = p.y;
            zi[k] = p.z;
        }
    }
    float ax[IB], ay[IB], az[IB];
#pragma unroll
    for (int k = 0; k < IB; ++k) ax[k] = ay[k] = az[k] = 0.0f;
    double gsum = 0.0;                     // the folded tiles: row c, lane p -> component c of i p
    double cx = 0.0, cy = 0.0, cz = 0.0;  // lane 8 p + k: contact terms of i k
    int listed = 0;
    int jt = min(je, jb + kDirectFold * stride);  // the tile's end
    for (;;) {
        while (jb < jt && listed <= kWorkOff) {
            float4 pj = nx;
            const int j0 = jb;
            jb += stride;
            nx = pos[min(jb + lane, end - 1)];
            if (j0 + lane >= je) pj.x = pj.y = pj.z = kGhostCoord;  // past the segment: no force, no contact
            unsigned long long near[IB], any = 0;
#pragma unroll
            for (int k = 0; k < IB; ++k) {
                const float dx = pj.x - xi[k];
                const float dy = pj.y - yi[k];
                const float dz = pj.z - zi[k];
                const float r2 = fast_r2(dx, dy, dz);
                const float s = fast_inv_r3(r2);
                ax[k] = __builtin_fmaf(s, dx, ax[k]);
                ay[k] = __builtin_fmaf(s, dy, ay[k]);
                az[k] = __builtin_fmaf(s, dz, az[k]);
                near[k] = __ballot(r2 < kDirectContactR2);
                any |= near[k];
            }
            // the sums before the branch: sunk past it, their operands cost 32 registers
#pragma unroll
            for (int k = 0; k < IB; ++k) asm volatile("" : "+v"(ax[k]), "+v"(ay[k]), "+v"(az[k]));
            if (!any) continue;
#pragma unroll
            for (int k = 0; k < IB; ++k) {
                // not the pair of i k with itself, where this block holds it
                const int own = i0 + k - j0;
                unsigned long long m = near[k];
                if (own >= 0 && own < 64 && i0 + k < je) m &= ~(1ull << own);
                if (m == 0 || i0 + k >= end) continue;
                if (m >> lane & 1)
                    list[wv][listed + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                        k << 24 | (j0 + lane);
                listed += __popcll(m);
            }
        }
        // The listed pairs: the exact contact term minus the gravity term
        // s dp the sums took for it (k_finish's test and arithmetic), a pair
        // per lane, then added per i in list order.
        // the law read here: hoisted out, its registers spill the loop's
        const SimDesc* lp = sims + blk.sim;
        asm volatile("" : "+s"(lp));
        const PairLaw& law = lp->law;
        for (int e0 = 0; e0 < listed; e0 += 64) {
            const int cnt = min(64, listed - e0);
            wave_lds_sync();
            float4 t = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(-1));
            if (lane < cnt) {
                const int e = list[wv][e0 + lane];
                const int k = e >> 24, jj = e & 0xffffff;
                const float4 pi = pos[i0 + k], pj = pos[jj];
                const float4 vi = vel[i0 + k], vj = vel[jj];
                const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
                const float r2 = dx * dx + dy * dy + dz * dz;
                const float r = sqrtf(r2);
                if (r < 1.0f) {
                    const float invr = 1.0f / r;
                    const float dvx = vj.x - vi.x, dvy = vj.y - vi.y, dvz = vj.z - vi.z;
                    const float dot = dx * dvx + dy * dvy + dz * dvz;
                    const int test = (int)(i0 + k < fe_end) + (int)jfe;
                    const float fm = contact_pair_mag(law, test, r, r2, dot);
                    const float sf = gravity_product(law, test) * fast_inv_r3(fast_r2(dx, dy, dz));
                    t = make_float4(fm * dx * invr - sf * dx, fm * dy * invr - sf * dy, fm * dz * invr - sf * dz,
                                    __int_as_float(k));
                }
            }
            term[wv][lane] = t;
            wave_lds_sync();
            // Lane 8 p + k takes the terms of i k among every eighth term of
            // the batch.  (All 64 terms looked at by each of eight lanes took
            // 1 us a batch: a step of N = 1,024 in contact 9.3 us, 7.0 so, of
            // 8,192 33.5 and 29.6.)
#pragma unroll 4
            for (int u = 0; u < 8; ++u) {
                const float4 o = term[wv][8 * u + (lane >> 3)];
                const bool mine = __float_as_int(o.w) == (lane & 7);
                cx += (double)(mine ? o.x : 0.0f);
                cy += (double)(mine ? o.y : 0.0f);
                cz += (double)(mine ? o.z : 0.0f);
            }
        }
        listed = 0;
        if (jb < jt) continue;
        gsum += rows_sum_xyz(row_sums8(ax, lane & 15), row_sums8(ay, lane & 15), row_sums8(az, lane & 15));
        if (jb >= je) break;
        jt = min(je, jb + kDirectFold * stride);
#pragma unroll
        for (int k = 0; k < IB; ++k) ax[k] = ay[k] = az[k] = 0.0f;
    }
    grav[wv][lane] = gsum;
    cx = eighths_sum(cx);
    cy = eighths_sum(cy);
    cz = eighths_sum(cz);
    if (lane < IB) {
        contact[wv][0][lane] = cx;
        contact[wv][1][lane] = cy;
        contact[wv][2][lane] = cz;
    }
    // Wavefront c < 3 adds component c: lane w * 8 + k takes the sums of i k
    // of wavefront w, then the eight lanes of an i are added.  The move's
    // components are independent; wavefront 3 carries .w over.  What this
    // reads is asked for before the others are waited for.
    const int k = lane & 7, w = lane >> 3;
    const int i = i0 + k;
    float g = 0.0f, v = 0.0f, p = 0.0f;
    if (wv < 3) g = gravity_product(sd.law, (int)(i < fe_end) + (int)(w < wf));
    if constexpr (MOVE != 0)
        if (wv < 4 && i < end) {
            v = reinterpret_cast<const float*>(vel + i)[wv];
            p = reinterpret_cast<const float*>(pos + i)[wv];
        }
    __syncthreads();
    if (wv > 3) return;
    if (wv == 3) {
        if constexpr (MOVE != 0)
            if (lane < IB && i < end) {
                mv.pout[i].w = p;
                mv.vout[i].w = v;
            }
        return;
    }
    const double sum = eighths_sum((double)g * grav[w][16 * wv + k] + contact[w][wv][k]);
    if (lane >= IB || i >= end) return;
    const float f = (float)sum;
    reinterpret_cast<float*>(force + i)[wv] = f;
    if constexpr (MOVE != 0) {
        float temp, damp = 0.0f;
        if constexpr (MOVE == 1) {
            temp = i < mv.b1 ? mv.dt_over_mass_fe : mv.dt_over_mass_si;
        } else if (mv.b3 <= i) {
            temp = mv.dt_over_mass_si;
            damp = mv.damp2;
        } else if (mv.b2 <= i) {
            temp = mv.dt_over_mass_fe;
            damp = mv.damp2;
        } else if (mv.b1 <= i) {
            temp = mv.dt_over_mass_si;
            damp = mv.damp1;
        } else {
            temp = mv.dt_over_mass_fe;
            damp = mv.damp1;
        }
        if constexpr (MOVE == 1)
            v += f * temp;
        else
            v += (f - damp * v) * temp;
        p += v * mv.dt;
        reinterpret_cast<float*>(mv.vout + i)[wv] = v;
        reinterpret_cast<float*>(mv.pout + i)[wv] = p;
    }
}

// The per-particle potential of k_finish_potential in one launch, for the
// energy reduction (FP64 sums).  A workgroup holds 64 / S i-particles, S lanes
// each, and its kDirectWaves * S lanes per particle ("j-streams") share the
// simulation's j-range: each segment (iron j, then silicate j) is cut into
// groups of four j dealt out in turn (stream k takes groups k, k + 16 S, ...),
// summed in float tiles of kDirectTile j.
constexpr int kDirectWaves = 16;
constexpr int kDirectTile = 256;  // j per float tile

template <int S>
__global__ __launch_bounds__(64 * kDirectWaves) void k_direct_potential(const float4* __restrict__ pos,
                                                                        const DirectBlock* __restrict__ blocks,
                                                                        const SimDesc* __restrict__ sims,
                                                                        double* __restrict__ pe) {
    static_assert(S == 1 || S == 2 || S == 4 || S == 8, "lanes per particle");
    constexpr int IB = 64 / S;             // i-particles per workgroup
    constexpr int NS = kDirectWaves * S;   // j-streams per particle
    constexpr int TG = kDirectTile / 4;    // groups per stream per float tile
    __shared__ double red[kDirectWaves][64];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int stream = wv * S + lane / IB;  // wave-uniform when S == 1
    const DirectBlock b = blocks[blockIdx.x];
    const int start = sims[b.sim].start, fe_end = sims[b.sim].fe_end, end = sims[b.sim].end;
    const PairLaw law = sims[b.sim].law;
    const int i = b.i0 + lane % IB;
    const bool live = i < end;
    const int ic = live ? i : end - 1;
    const float4 pi = pos[ic];
    const bool ife = ic < fe_end;
    double sum = 0.0;  // this stream's gravity plus contact corrections
    for (int seg = 0; seg < 2; ++seg) {
        const bool jfe = seg == 0;  // iron j first, then silicate j
        const int a = jfe ? start : fe_end;
        const int e = jfe ? fe_end : end;
        const int ngroups = (e - a + 3) / 4;
        if (stream >= ngroups) continue;
        const int test = (int)ife + (int)jfe;
        const float g = gravity_product(law, test);
        double u = 0.0, c = 0.0;
        // k_finish_potential's term of a pair in contact
        auto contact = [&](int j, const float4 pj, float s) {
            const double ddx = (double)pj.x - pi.x, ddy = (double)pj.y - pi.y, ddz = (double)pj.z - pi.z;
            const double r = sqrt(ddx * ddx + ddy * ddy + ddz * ddz);
            if (r < 1.0 && j != i) {
                const double G = gravity_product(law, test);
                const double K = approach_k(law, test);
                const double exact = G * (r - 2.0) + (K / 3.0) * (r - 1.0) * (r - 1.0) * (r + 2.0);
                c += exact + G * (double)s;
            }
        };
        // this stream's groups, TG of them per float tile
        for (int g0 = stream; g0 < ngroups; g0 += NS * TG) {
            const int g1 = min(g0 + NS * TG, ngroups);
            float tx = 0.0f;
            auto pair = [&](const float4 q, float& s, bool& near) {
                const float dx = q.x - pi.x;
                const float dy = q.y - pi.y;
                const float dz = q.z - pi.z;
                const float r2f = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                s = r2f > 0.0f ? __builtin_amdgcn_rsqf(r2f) : 0.0f;
                tx += s;
                near |= r2f < kDirectContactR2;
            };
            // The next group's loads are in flight while this one is computed
            // (indices clamped into the segment; a partial last group only
            // takes its first e - j pairs).
            float4 q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = pos[min(a + 4 * g0 + k, e - 1)];
            for (int grp = g0; grp < g1; grp += NS) {
                const int j = a + 4 * grp;
                const int jn = grp + NS < g1 ? j + 4 * NS : j;
                float4 nq[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) nq[k] = pos[min(jn + k, e - 1)];
                float s[4];
                bool near = false;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (j + k < e) pair(q[k], s[k], near);
                if (near) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (j + k < e) contact(j + k, q[k], s[k]);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = nq[k];
            }
            u += (double)tx;
        }
        sum += -(double)g * u + c;
    }
    red[wv][lane] = sum;
    __syncthreads();
    if (wv == 0 && lane < IB && live) {
        double f = 0.0;
#pragma unroll
        for (int w = 0; w < kDirectWaves; ++w)
#pragma unroll
            for (int q = 0; q < S; ++q) f += red[w][q * IB + lane];
        pe[i] = 0.5 * f;
    }
}

// ---------------------------------------------------------------------------
// Move kernels
// ---------------------------------------------------------------------------

// moveBodiesCollisionSingleGPU (impactAddTime.cu:379-394), generalised to
// packed simulations.  No contraction: v + f*t and x + v*dt round as written.
__global__ void k_move(float4* __restrict__ pos, float4* __restrict__ vel,
                       const float4* __restrict__ force, int ntot, const SimDesc* __restrict__ sims,
                       int nsims) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntot) return;
    const SimDesc& sd = sims[nsims == 1 ? 0 : find_sim(sims, nsims, i)];
    if (!sd.active) return;
    const float temp = i < sd.fe_end ? sd.dt_over_mass_fe : sd.dt_over_mass_si;
    float4 v = vel[i];
    float4 p = pos[i];
    const float4 f = force[i];
    v.x += f.x * temp;
    v.y += f.y * temp;
    v.z += f.z * temp;
    p.x += v.x * sd.dt;
    p.y += v.y * sd.dt;
    p.z += v.z * sd.dt;
    vel[i] = v;
    pos[i] = p;
}

// moveBodiesCollisionSingleGPU with its constants by value (the drop-in path).
__global__ void k_move_collision(float4* __restrict__ pos, float4* __restrict__ vel,
                                 const float4* __restrict__ force, int n, float dt,
                                 float dt_over_mass_fe, float dt_over_mass_si, int nfe) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float temp = i < nfe ? dt_over_mass_fe : dt_over_mass_si;
    float4 v = vel[i];
    float4 p = pos[i];
    const float4 f = force[i];
    v.x += f.x * temp;
    v.y += f.y * temp;
    v.z += f.z * temp;
    p.x += v.x * dt;
    p.y += v.y * dt;
    p.z += v.z * dt;
    vel[i] = v;
    pos[i] = p;
}

// moveBodiesDampedSeperate (generateTargetImpactor.cu:628-664).
__global__ void k_move_damped_separate(float4* __restrict__ pos, float4* __restrict__ vel,
                                       const float4* __restrict__ force, int n, float dt,
                                       float dt_over_mass_fe, float dt_over_mass_si, int b1, int b2,
                                       int b3, float damp1, float damp2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float temp, damp;
    if (b3 <= i) {
        temp = dt_over_mass_si;
        damp = damp2;
    } else if (b2 <= i) {
        temp = dt_over_mass_fe;
        damp = damp2;
    } else if (b1 <= i) {
        temp = dt_over_mass_si;
        damp = damp1;
    } else {
        temp = dt_over_mass_fe;
        damp = damp1;
    }
    float4 v = vel[i];
    float4 p = pos[i];
    const float4 f = force[i];
    v.x += (f.x - damp * v.x) * temp;
    v.y += (f.y - damp * v.y) * temp;
    v.z += (f.z - damp * v.z) * temp;
    p.x += v.x * dt;
    p.y += v.y * dt;
    p.z += v.z * dt;
    vel[i] = v;
    pos[i] = p;
}

// ---------------------------------------------------------------------------
// FP64 reductions: mass moments, momentum, angular momentum, energy
// ---------------------------------------------------------------------------

// Per-particle potential: -(1/2) * (sum of the chunk partials of 1/r scaled
// by G mi mj) plus, for pairs with r < 1, half the difference between the
// exact contact potential and the gravity term pass 1 added.  FP64 output.
__global__ __launch_bounds__(256) void k_finish_potential(int ntot, const SimDesc* __restrict__ sims,
                                                          int nsims,
                                                          const float4* __restrict__ partial,
                                                          const float4* __restrict__ gsum,
                                                          const int* __restrict__ starts,
                                                          const int* __restrict__ sorted,
                                                          const float4* __restrict__ spos,
                                                          double* __restrict__ pe) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntot) return;
    const int i = sorted[t];
    const int s = find_sim(sims, nsims, i);
    const SimDesc& sd = sims[s];
    const int n = sd.end - sd.start;
    double phi = 0.0;
    if (gsum && sd.gn > 0)
        phi = (double)gsum[i].x;
    else
        for (int c = 0; c < sd.nchunk; ++c) phi += (double)partial[sd.partial_base + c * n + (i - sd.start)].x;
    double u = -phi;
    const float4 pi = spos[t];
    const int ccx = cell_coord(pi.x), ccy = cell_coord(pi.y), ccz = cell_coord(pi.z);
    const bool ife = i < sd.fe_end;
    for (int oz = -1; oz <= 1; ++oz)
        for (int oy = -1; oy <= 1; ++oy)
            for (int ox = -1; ox <= 1; ++ox) {
                const int qx = ccx + ox, qy = ccy + oy, qz = ccz + oz;
                const unsigned h = cell_bucket(sd.hbase, sd.hmask, qx, qy, qz);
                for (int k = starts[h]; k < starts[h + 1]; ++k) {
                    const float4 pj = spos[k];
                    if (cell_coord(pj.x) != qx || cell_coord(pj.y) != qy || cell_coord(pj.z) != qz)
                        continue;
                    const int j = sorted[k];
                    if (j == i || j < sd.start || j >= sd.end) continue;
                    const double dx = (double)pj.x - pi.x, dy = (double)pj.y - pi.y,
                                 dz = (double)pj.z - pi.z;
                    const double r = sqrt(dx * dx + dy * dy + dz * dz);
                    if (r >= 1.0) continue;
                    const int test = (int)ife + (int)(j < sd.fe_end);
                    const double G = gravity_product(sd.law, test);
                    const double K = approach_k(sd.law, test);
                    const double exact = G * (r - 2.0) + (K / 3.0) * (r - 1.0) * (r - 1.0) * (r + 2.0);
                    const float fx = pj.x - pi.x, fy = pj.y - pi.y, fz = pj.z - pi.z;
                    const float r2f = __builtin_fmaf(fz, fz, __builtin_fmaf(fy, fy, fx * fx));
                    const double fast = -G * (double)__builtin_amdgcn_rsqf(r2f);
                    u += exact - fast;
                }
            }
    pe[i] = 0.5 * u;
}

// Block partial sums of the 14 FP64 moments of the particles of one
// simulation: M, M x (3), M v (3), sum m x cross v (3), kinetic, potential,
// sum m |x|^2 (unused by callers, kept for the rigid-body test), count.
constexpr int kMoments = 14;

__global__ __launch_bounds__(256) void k_moments(const float4* __restrict__ pos,
                                                 const float4* __restrict__ vel,
                                                 const double* __restrict__ pe,
                                                 const int* __restrict__ block_sim,
                                                 const int* __restrict__ block_first,
                                                 const SimDesc* __restrict__ sims,
                                                 double mass_fe_override, double mass_si_override,
                                                 double* __restrict__ out) {
    __shared__ double sh[kMoments][256];
    const int s = block_sim[blockIdx.x];
    const int i = block_first[blockIdx.x] + threadIdx.x;
    const SimDesc& sd = sims[s];
    double v[kMoments];
#pragma unroll
    for (int k = 0; k < kMoments; ++k) v[k] = 0.0;
    if (i < sd.end) {
        double m;
        if (mass_fe_override > 0.0)
            m = i < sd.fe_end ? mass_fe_override : mass_si_override;
        else
            m = i < sd.fe_end ? (double)sd.law.GMassFeSi : 1.0;
        const float4 p = pos[i];
        const float4 u = vel[i];
        const double x = p.x, y = p.y, z = p.z, a = u.x, b = u.y, c = u.z;
        v[0] = m;
        v[1] = m * x;
        v[2] = m * y;
        v[3] = m * z;
        v[4] = m * a;
        v[5] = m * b;
        v[6] = m * c;
        v[7] = m * (y * c - z * b);
        v[8] = m * (z * a - x * c);
        v[9] = m * (x * b - y * a);
        v[10] = 0.5 * m * (a * a + b * b + c * c);
        v[11] = pe ? pe[i] : 0.0;
        v[12] = m * (x * x + y * y + z * z);
        v[13] = 1.0;
    }
#pragma unroll
    for (int k = 0; k < kMoments; ++k) sh[k][threadIdx.x] = v[k];
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
#pragma unroll
            for (int k = 0; k < kMoments; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x < kMoments) out[blockIdx.x * kMoments + threadIdx.x] = sh[threadIdx.x][0];
}

// Sum the block moments of each simulation in block order (one thread per
// simulation) and, for the recenter, turn them into the shift to apply.
__global__ void k_moments_final(const double* __restrict__ blocks, const int* __restrict__ sim_first_block,
                                int nsims, double* __restrict__ sums) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsims) return;
    double acc[kMoments];
#pragma unroll
    for (int k = 0; k < kMoments; ++k) acc[k] = 0.0;
    for (int b = sim_first_block[s]; b < sim_first_block[s + 1]; ++b)
#pragma unroll
        for (int k = 0; k < kMoments; ++k) acc[k] += blocks[b * kMoments + k];
#pragma unroll
    for (int k = 0; k < kMoments; ++k) sums[s * kMoments + k] = acc[k];
}

// FP64 mass moments of particles [0, n) (iron for i < nfe): per block
// {M, M x, M y, M z, M vx, M vy, M vz}, summed by k_moments_one_final.
constexpr int kMoments1 = 7;

__global__ __launch_bounds__(256) void k_moments_one(const float4* __restrict__ pos,
                                                     const float4* __restrict__ vel, int n, int nfe,
                                                     double mass_fe, double mass_si,
                                                     double* __restrict__ out) {
    __shared__ double sh[kMoments1][256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    double v[kMoments1];
#pragma unroll
    for (int k = 0; k < kMoments1; ++k) v[k] = 0.0;
    if (i < n) {
        const double m = i < nfe ? mass_fe : mass_si;
        const float4 p = pos[i];
        const float4 u = vel[i];
        v[0] = m;
        v[1] = m * p.x;
        v[2] = m * p.y;
        v[3] = m * p.z;
        v[4] = m * u.x;
        v[5] = m * u.y;
        v[6] = m * u.z;
    }
#pragma unroll
    for (int k = 0; k < kMoments1; ++k) sh[k][threadIdx.x] = v[k];
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
#pragma unroll
            for (int k = 0; k < kMoments1; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x < kMoments1) out[blockIdx.x * kMoments1 + threadIdx.x] = sh[threadIdx.x][0];
}

// One block: column k summed over the nb block rows in block order.
__global__ void k_moments_one_final(const double* __restrict__ blocks, int nb, double* __restrict__ sums) {
    const int k = threadIdx.x;
    if (k >= kMoments1) return;
    double acc = 0.0;
    for (int b = 0; b < nb; ++b) acc += blocks[b * kMoments1 + k];
    sums[k] = acc;
}

// Recenter (impactAddTime.cu:433-455) with the means taken in FP64 on the
// device: positions += target_com - com, velocities += target_vel - mean_vel.
__global__ void k_recenter_apply(float4* __restrict__ pos, float4* __restrict__ vel, int n,
                                 const double* __restrict__ sums, double tcx, double tcy, double tcz,
                                 double tvx, double tvy, double tvz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double M = sums[0];
    const float sx = (float)(tcx - sums[1] / M);
    const float sy = (float)(tcy - sums[2] / M);
    const float sz = (float)(tcz - sums[3] / M);
    const float ux = (float)(tvx - sums[4] / M);
    const float uy = (float)(tvy - sums[5] / M);
    const float uz = (float)(tvz - sums[6] / M);
    float4 p = pos[i];
    float4 v = vel[i];
    p.x += sx;
    p.y += sy;
    p.z += sz;
    v.x += ux;
    v.y += uy;
    v.z += uz;
    pos[i] = p;
    vel[i] = v;
}

// The reference's own recenter (impactAddTime.cu:433-455), float for float.
// getMassCollision(0) / getCenterOfMassCollision(0) /
// getLinearVelocityCollision(0) (impactBasicFunctions.h:219-230,268-297,
// 388-417) accumulate in float on the host, particle by particle in index
// order: acc = float(double(acc) + double(x) * m) with m the double element
// mass (iron for i < nfe), and the mass the same way with x = 1.  Each of
// those seven sums ("chains") is n dependent roundings.
//
// Taken one after another they cost 52 ns each on the device (3.4 ms at
// N = 65,536).  They need not be: a step a -> float(double(a) + t) commutes
// with a shift d of a whenever d is a multiple of two float ulps of the
// binade the step's sum lies in and neither the sum nor the shifted sum
// leaves that binade (then both roundings, to double and to float, act on
// the same grid, and d keeps the parity that ties look at).  So a run of
// steps can be taken from a guessed start g, and holds for the true start a
// too if d = a - g is such a multiple for the run's largest binade and |d| is
// smaller than every sum's distance from its binade's ends: its end is then
// the guess's end plus d, exactly.
//   k_rc_window_sums   FP64 sums of windows of the chain;
//   k_rc_bounds        cuts the chain in each window where the FP64 prefix is
//                      largest (the coarsest grid there, so few residues of
//                      the start matter) and guesses the start from it;
//   k_rc_runs          every run from 16 starts, one float ulp apart (they
//                      cover every residue up to 8 ulps), with its largest
//                      binade and least distance; then a workgroup's 16 runs
//                      joined from its first run's 16 starts;
//   k_rc_join          one wavefront per chain: the joined groups in order
//                      from the true start; where the conditions do not
//                      hold, run by run, and a run that does not hold is
//                      taken step by step.  No result depends on a guess: a
//                      guess only decides which way it is reached.
// Joining looks at all 16 starts at once, one per lane of a row, and takes the
// first that holds: 24 groups of an impact state's 448 go run by run instead
// of the 27 where only the start picked by the difference was tried, nothing
// is looked up by it, and the groups' own joins, 11 us in the chains' seven
// workgroups, run side by side.  What it compares is worked out beforehand, a
// candidate per lane (0.24 us a group or run before).
// Bound by the join's chain of dependent FP64 operations.  The impact states
// need 0 to 14 of 1,024 runs of a chain step by step.  N = 65,536, eight
// impact states: 75 to 140 us a call, 93 on average (sums 5 us, bounds 16,
// runs 17, join 25 to 95, apply 5; 119 with an element per load of all 16
// lanes and the candidates worked out as they are met, 137 with the groups
// joined in the chains' own workgroups and one start tried) against 3,404
// step by step; windows of 128 took 10% longer.  A system at rest that has just
// been recentred, whose sums cross zero, takes 290.
constexpr int kRcChains = 7;
constexpr int kRcStarts = 16;
constexpr int kRcGroup = 16;     // runs per group
constexpr int kRcMaxRuns = 1024;
constexpr float kRcRoom = 1.0e30f;  // no step yet
constexpr int kRcMaxGroups = kRcMaxRuns / kRcGroup;
static_assert(kRcStarts == 16 && kRcGroup == 16, "a workgroup of 256 holds a group's runs; a row of lanes a run's starts");

// A run from one start: its end, the least distance of a sum from its
// binade's ends (negative: never shift this run) and the largest binade.
struct __align__(16) RcRun {
    float end;
    int binade;
    float room;
    int pad;
};

// Scratch of one recenter over runs of `window` particles.
struct RcWork {
    double* sums;   // [kRcChains][nwin]
    int* bound;     // [kRcChains][nwin + 1]
    float* guess;   // [kRcChains][nwin]
    RcRun* runs;    // [kRcChains][nwin][kRcStarts]
    RcRun* groups;  // [kRcChains][ngroups][kRcStarts]: kRcGroup runs joined; binade -1: they do not hold
    float* total;   // [kRcChains]
    int window, nwin, ngroups;
};

// Term k of chain c: x, y, z, vx, vy, vz, 1 times the element's mass.
__device__ __forceinline__ float rc_value(const float4* __restrict__ pos, const float4* __restrict__ vel, int c,
                                          int k) {
    if (c == 6) return 1.0f;
    return reinterpret_cast<const float*>(c < 3 ? pos : vel)[4 * (size_t)k + (c < 3 ? c : c - 3)];
}

__device__ __forceinline__ void rc_terms(const float4* __restrict__ pos, const float4* __restrict__ vel, int k,
                                         double m, double (&t)[kRcChains]) {
    const float4 p = pos[k], v = vel[k];
    t[0] = (double)p.x * m;
    t[1] = (double)p.y * m;
    t[2] = (double)p.z * m;
    t[3] = (double)v.x * m;
    t[4] = (double)v.y * m;
    t[5] = (double)v.z * m;
    t[6] = m;
}

constexpr int kRcWindowWaves = 4;  // windows per workgroup, a wavefront each

// End of window w (also where the particle count is near the int range's end).
__device__ __forceinline__ int rc_window_end(const RcWork& wk, int w, int n) {
    return (int)min((long long)(w + 1) * wk.window, (long long)n);
}

__global__ __launch_bounds__(64 * kRcWindowWaves) void k_rc_window_sums(const float4* __restrict__ pos,
                                                                       const float4* __restrict__ vel, int n,
                                                                       int nfe, double mass_fe, double mass_si,
                                                                       RcWork wk) {
    const int lane = threadIdx.x & 63;
    const int w = blockIdx.x * kRcWindowWaves + (threadIdx.x >> 6);
    if (w >= wk.nwin) return;
    double s[kRcChains] = {};
    const int e = rc_window_end(wk, w, n);
    for (long long k = (long long)w * wk.window + lane; k < e; k += 64) {
        double t[kRcChains];
        rc_terms(pos, vel, (int)k, k < nfe ? mass_fe : mass_si, t);
#pragma unroll
        for (int c = 0; c < kRcChains; ++c) s[c] += t[c];
    }
#pragma unroll
    for (int c = 0; c < kRcChains; ++c) {
#pragma unroll
        for (int m = 32; m; m >>= 1) s[c] += __shfl_xor(s[c], m);
        if (lane == c) wk.sums[c * wk.nwin + w] = s[c];
    }
}

__global__ __launch_bounds__(64 * kRcWindowWaves) void k_rc_bounds(const float4* __restrict__ pos,
                                                                  const float4* __restrict__ vel, int n, int nfe,
                                                                  double mass_fe, double mass_si, RcWork wk) {
    const int lane = threadIdx.x & 63;
    const int w = blockIdx.x * kRcWindowWaves + (threadIdx.x >> 6);
    if (w >= wk.nwin) return;
    // the prefix before the window
    double p[kRcChains] = {};
    for (int k = lane; k < w; k += 64 * 4) {
        double v[4][kRcChains];  // four round trips to memory in one
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int c = 0; c < kRcChains; ++c) v[u][c] = wk.sums[c * wk.nwin + min(k + 64 * u, w - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int c = 0; c < kRcChains; ++c) p[c] += k + 64 * u < w ? v[u][c] : 0.0;
    }
    // this lane's share of the window: consecutive elements
    const int per = wk.window / 64;
    const int end = rc_window_end(wk, w, n);
    const int k0 = (int)min((long long)w * wk.window + lane * per, (long long)end), k1 = min((long long)k0 + per, (long long)end);
    double own[kRcChains] = {};
    for (int k = k0; k < k1; ++k) {
        double t[kRcChains];
        rc_terms(pos, vel, k, k < nfe ? mass_fe : mass_si, t);
#pragma unroll
        for (int c = 0; c < kRcChains; ++c) own[c] += t[c];
    }
#pragma unroll
    for (int c = 0; c < kRcChains; ++c) {
#pragma unroll
        for (int m = 32; m; m >>= 1) p[c] += __shfl_xor(p[c], m);
        double before = own[c];
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const double o = __shfl_up(before, m);
            if (lane >= m) before += o;
        }
        p[c] += before - own[c];
    }
    // the place of the largest prefix in the window
    double best[kRcChains], at[kRcChains];
    int place[kRcChains];
#pragma unroll
    for (int c = 0; c < kRcChains; ++c) {
        best[c] = -1.0;
        at[c] = 0.0;
        place[c] = 0x7fffffff;
    }
    for (int k = k0; k < k1; ++k) {
        double t[kRcChains];
        rc_terms(pos, vel, k, k < nfe ? mass_fe : mass_si, t);
#pragma unroll
        for (int c = 0; c < kRcChains; ++c) {
            p[c] += t[c];
            if (fabs(p[c]) > best[c]) {
                best[c] = fabs(p[c]);
                at[c] = p[c];
                place[c] = k + 1;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < kRcChains; ++c) {
#pragma unroll
        for (int m = 32; m; m >>= 1) {
            const double ob = __shfl_xor(best[c], m), oa = __shfl_xor(at[c], m);
            const int op = __shfl_xor(place[c], m);
            if (ob > best[c] || (ob == best[c] && op < place[c])) {
                best[c] = ob;
                at[c] = oa;
                place[c] = op;
            }
        }
        if (lane == 0) {
            int* __restrict__ bound = wk.bound + c * (wk.nwin + 1);
            float* __restrict__ guess = wk.guess + c * wk.nwin;
            if (w == 0) {
                bound[0] = 0;
                guess[0] = 0.0f;
            }
            const bool last = w + 1 == wk.nwin;
            // a window of NaNs has no largest prefix: cut at its end
            bound[w + 1] = last ? n : (best[c] >= 0.0 ? place[c] : end);
            if (!last) guess[w + 1] = (float)at[c];
        }
    }
}

// Start j of a run guessed to begin at g: j float ulps of g's binade above g.
__device__ __forceinline__ double rc_ulp(float g) {
    const int e = (int)((__float_as_uint(g) >> 23) & 0xff);
    // zero, denormal, infinite and NaN guesses have no ulp to step by
    return e == 0 || e == 255 ? 0.0 : __longlong_as_double((long long)(e - 127 - 23 + 1023) << 52);
}
__device__ __forceinline__ float rc_start(float g, int j) { return (float)((double)g + (double)j * rc_ulp(g)); }

// One step with term t: the sum's rounding to float, its binade
// and its distance from the binade's ends, rounded down to the sum's 21
// leading bits.  A zero term changes nothing from any start.
__device__ __forceinline__ void rc_step(float& a, double t, int& binade, float& room) {
    const double s = (double)a + t;
    const int hi = __double2hiint(s) & 0x7fffffff;
    const int e = hi >> 20;
    const int m = hi & 0xfffff;
    float r = __builtin_amdgcn_ldexpf((float)min(m, 0xfffff - m), e - 1023 - 20);
    // well inside the float range only (not infinite or NaN)
    if ((unsigned)(e - (1023 - 80)) > 160u) r = -1.0f;
    if (t != 0.0) {
        binade = max(binade, e);
        room = fminf(room, r);
    }
    a = (float)s;
}

// A run (or group) from one start as a join asks for it, worked out beforehand
// in FP64.  A group that does not hold starts at NaN; one whose terms are all
// zero takes any shift.
struct RcCand {
    double start, end, room, pairs;  // pairs: shifts in pairs of ulps of the largest binade, over the shift
};
__device__ __forceinline__ RcCand rc_cand(const RcRun& r, float start) {
    RcCand q{(double)start, (double)r.end, (double)r.room, __builtin_amdgcn_ldexp(1.0, 1023 + 22 - r.binade)};
    if (r.binade == 0) {
        q.room = __builtin_inf();
        q.pairs = 0.0;
    } else if (r.binade < 0) {
        q.start = __builtin_nan("");
    }
    return q;
}
// Whether it holds for the true start a, a float, and the difference d of the
// two starts: then a's end is the float q.end + d.
__device__ __forceinline__ bool rc_holds(double a, const RcCand& q, double& d) {
    d = a - q.start;
    const double k = d * q.pairs;
    const bool shift = (fabs(d) < q.room) & (k == rint(k));
    return (a - d == q.start) & (shift | (d == 0.0));
}

// Lane j of a row of 16 holds a run's (or group's) start j and what it led
// to: the lowest lane of the row it holds for, or -1.  All rows of the
// wavefront take part.
__device__ __forceinline__ int rc_pick(bool holds, int lane) {
    const unsigned m = (unsigned)(__ballot(holds) >> (lane & 48)) & 0xffffu;
    return m ? (lane & 48) + __builtin_ctz(m) : -1;
}

// Sixteen steps from U on, step u with lane u's term of each row of 16 lanes.
template <int U = 0>
__device__ __forceinline__ void rc_steps16(RcRun& r, double t) {
    if constexpr (U < 16) {
        rc_step(r.end,
                __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(t), 0x150 + U, 0xF, 0xF, true),
                                 __builtin_amdgcn_mov_dpp(__double2loint(t), 0x150 + U, 0xF, 0xF, true)),
                r.binade, r.room);
        rc_steps16<U + 1>(r, t);
    }
}

// One workgroup per group of a chain: the group's runs from their starts, a
// run and start per lane (a run's elements 16 at a time, one load per lane of
// its row, four such loads in flight), then the runs joined from each of the group's
// starts, a row of lanes per start.
__global__ __launch_bounds__(256) void k_rc_runs(const float4* __restrict__ pos, const float4* __restrict__ vel,
                                                 int nfe, double mass_fe, double mass_si, RcWork wk) {
    __shared__ RcCand run[kRcGroup][kRcStarts];
    __shared__ int binade[kRcGroup][kRcStarts];
    const int c = blockIdx.x / wk.ngroups, g = blockIdx.x % wk.ngroups;
    const int row = threadIdx.x / kRcStarts, j = threadIdx.x % kRcStarts, lane = threadIdx.x & 63;
    const int s0 = g * kRcGroup, ns = min(kRcGroup, wk.nwin - s0);
    if (row < ns) {
        const int s = s0 + row;
        const int* __restrict__ bound = wk.bound + c * (wk.nwin + 1);
        const int b = bound[s], e = bound[s + 1];
        const float gs = wk.guess[c * wk.nwin + s];
        RcRun r{rc_start(gs, j), 0, kRcRoom, 0};
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = rc_value(pos, vel, c, min(b + 16 * u + j, e - 1));
        for (int k = b; k < e; k += 64) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = k + 16 * u + j;
                // past the run's end: -0 leaves every sum as it is
                const double t = i < e ? (double)x[u] * (i < nfe ? mass_fe : mass_si) : -0.0;
                x[u] = rc_value(pos, vel, c, min(i + 64, e - 1));
                rc_steps16(r, t);
            }
        }
        wk.runs[((size_t)c * wk.nwin + s) * kRcStarts + j] = r;
        run[row][j] = rc_cand(r, rc_start(gs, j));
        binade[row][j] = r.binade;
    }
    __syncthreads();
    RcRun x{(float)run[0][row].start, 0, kRcRoom, 0};
    for (int s = 0; s < ns; ++s) {
        const RcCand q = run[s][j];
        double d;
        const int at = rc_pick(rc_holds((double)x.end, q, d), lane);
        const int from = max(at, 0);
        // rounded down: the least factor below 1 takes more than the
        // subtraction's and the conversion's rounding
        const float room = (float)((q.room - fabs(d)) * (1.0 - 0x1p-20));
        x.end = __shfl((float)(q.end + d), from);
        x.room = fminf(x.room, __shfl(room, from));
        x.binade = x.binade < 0 || at < 0 ? -1 : max(x.binade, binade[s][from & 15]);
    }
    if (j == 0) wk.groups[((size_t)c * wk.ngroups + g) * kRcStarts + row] = x;
}

// Chain c from a on over the elements [k0, e), step by step, by one wavefront:
// 64 terms at a time through its 64 doubles of LDS.
__device__ __forceinline__ double rc_chain(const float4* __restrict__ pos, const float4* __restrict__ vel, int c,
                                           int k0, int e, int nfe, double mass_fe, double mass_si, double a,
                                           double* __restrict__ terms) {
    const int lane = threadIdx.x & 63;
    for (; k0 < e; k0 += 64) {
        wave_lds_sync();
        const int k = min(k0 + lane, e - 1);
        // past the end: -0 leaves every sum as it is
        terms[lane] = k0 + lane < e ? (double)rc_value(pos, vel, c, k) * (k < nfe ? mass_fe : mass_si) : -0.0;
        wave_lds_sync();
#pragma unroll 8
        for (int u = 0; u < 64; ++u) a = (double)(float)(a + terms[u]);
    }
    return a;
}

// All of a chain step by step, for so few particles that the four launches of
// the runs cost more than they save.  N = 40, 256, 512, 1,024, 1,536 and
// 2,048: 8, 8, 12, 19, 27 and 35 us a call and by runs 24, 31, 35, 39, 39 and
// 45 (bodies in motion: 2,048 40 and 40, 3,000 54 and 43); all seven chains on
// one wavefront 9, 17, 31, 57, 84 and 110.
constexpr int kRcStepsMaxN = 2048;
__global__ __launch_bounds__(64) void k_rc_steps(const float4* __restrict__ pos, const float4* __restrict__ vel, int n,
                                                 int nfe, double mass_fe, double mass_si, float* __restrict__ total) {
    __shared__ double terms[64];
    const double a = rc_chain(pos, vel, blockIdx.x, 0, n, nfe, mass_fe, mass_si, 0.0, terms);
    if (threadIdx.x == 0) total[blockIdx.x] = (float)a;
}

__global__ __launch_bounds__(256) void k_rc_join(const float4* __restrict__ pos, const float4* __restrict__ vel,
                                                 int nfe, double mass_fe, double mass_si, RcWork wk) {
    __shared__ RcCand group[kRcMaxGroups][kRcStarts];
    __shared__ RcCand one[kRcGroup][kRcStarts];  // the runs of a group that does not hold
    __shared__ float guess[kRcMaxRuns];
    __shared__ double terms[64];
    const int c = blockIdx.x;
    const RcRun* __restrict__ runs = wk.runs + (size_t)c * wk.nwin * kRcStarts;
    const int ngroups = wk.ngroups;
    for (int s = threadIdx.x; s < wk.nwin; s += 256) guess[s] = wk.guess[c * wk.nwin + s];
    __syncthreads();
    for (int k = threadIdx.x; k < ngroups * kRcStarts; k += 256) {
        const int g = k / kRcStarts, j = k % kRcStarts;
        group[g][j] = rc_cand(wk.groups[(size_t)c * ngroups * kRcStarts + k], rc_start(guess[g * kRcGroup], j));
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x, j = lane % kRcStarts;
    const int* __restrict__ bound = wk.bound + c * (wk.nwin + 1);
    double a = 0.0;  // a float throughout
    // a joined with a run (or group): whether it holds, from any of its starts
    // (the rows of lanes agree)
    auto take = [&](const RcCand& q) {
        double d;
        const unsigned m = (unsigned)__ballot(rc_holds(a, q, d)) & 0xffffu;
        if (!m) return false;
        const double e = (double)(float)(q.end + d);
        const int at = __builtin_ctz(m);
        a = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(e), at),
                             __builtin_amdgcn_readlane(__double2loint(e), at));
        return true;
    };
    RcCand q = group[0][j];
    for (int g = 0; g < ngroups; ++g) {
        const RcCand next = group[min(g + 1, ngroups - 1)][j];  // on its way
        const bool held = take(q);
        q = next;
        if (held) continue;
        const int s0 = g * kRcGroup, s1 = min(s0 + kRcGroup, wk.nwin);
        wave_lds_sync();
        for (int k = lane; k < (s1 - s0) * kRcStarts; k += 64)
            one[0][k] = rc_cand(runs[s0 * kRcStarts + k], rc_start(guess[s0 + k / kRcStarts], j));
        const int edge = bound[min(s0 + lane, wk.nwin)];  // lanes 0..kRcGroup
        wave_lds_sync();
        for (int s = s0; s < s1; ++s) {
            if (take(one[s - s0][j])) continue;
            a = rc_chain(pos, vel, c, __shfl(edge, s - s0), __shfl(edge, s + 1 - s0), nfe, mass_fe, mass_si, a, terms);
        }
    }
    if (lane == 0) wk.total[c] = (float)a;
}

__global__ void k_recenter_ref_apply(float4* __restrict__ pos, float4* __restrict__ vel, int n,
                                     const float* __restrict__ total, float tcx, float tcy, float tcz, float tvx,
                                     float tvy, float tvz) {
    __shared__ float shift[6];
    const int lane = threadIdx.x;
    if (lane < 6) {
        // centerOfMass.x /= totalMass in float: the double quotient rounded
        // once to float is the correctly rounded float quotient (53 >= 2*24+2).
        const float mean = (float)((double)total[lane] / (double)total[6]);
        const float target = lane == 0 ? tcx : lane == 1 ? tcy : lane == 2 ? tcz : lane == 3 ? tvx : lane == 4 ? tvy : tvz;
        shift[lane] = target - mean;
    }
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 p = pos[i];
    float4 v = vel[i];
    p.x += shift[0];
    p.y += shift[1];
    p.z += shift[2];
    v.x += shift[3];
    v.y += shift[4];
    v.z += shift[5];
    pos[i] = p;
    vel[i] = v;
}

// Explicit instantiations used by the host code.
#define GI_GRAVITY_INST(R, POT, V) \
    template __global__ void k_gravity<R, 128, POT, V>(const float4*, const GravTask*, int, const SimDesc*, float4*);
GI_GRAVITY_INST(1, false, 0)
GI_GRAVITY_INST(1, false, 1)
GI_GRAVITY_INST(1, true, 0)
GI_GRAVITY_INST(2, false, 0)
GI_GRAVITY_INST(4, false, 0)
GI_GRAVITY_INST(8, false, 0)
GI_GRAVITY_INST(2, false, 1)
GI_GRAVITY_INST(4, false, 1)
GI_GRAVITY_INST(8, false, 1)
GI_GRAVITY_INST(2, true, 0)
GI_GRAVITY_INST(4, true, 0)
GI_GRAVITY_INST(8, true, 0)
#undef GI_GRAVITY_INST
#define GI_MUTUAL_INST(R, POT) \
    template __global__ void k_mutual<R, POT>(const float4*, const MutualTask*, int, const SimDesc*, float*, float*);
#define GI_DIRECT_INST(MOVE)                                                                                     \
    template __global__ void k_direct<MOVE>(const float4*, const float4*, const DirectBlock*, int, const SimDesc*, \
                                            float4*, FusedMove);
GI_DIRECT_INST(0)
GI_DIRECT_INST(1)
GI_DIRECT_INST(2)
#undef GI_DIRECT_INST
#define GI_DIRECT_POT_INST(S) \
    template __global__ void k_direct_potential<S>(const float4*, const DirectBlock*, const SimDesc*, double*);
GI_DIRECT_POT_INST(1)
GI_DIRECT_POT_INST(2)
GI_DIRECT_POT_INST(4)
GI_DIRECT_POT_INST(8)
#undef GI_DIRECT_POT_INST
GI_MUTUAL_INST(1, false)
GI_MUTUAL_INST(2, false)
GI_MUTUAL_INST(4, false)
GI_MUTUAL_INST(8, false)
GI_MUTUAL_INST(1, true)
GI_MUTUAL_INST(2, true)
GI_MUTUAL_INST(4, true)
GI_MUTUAL_INST(8, true)
#undef GI_MUTUAL_INST
#define GI_MUTUAL_GRP_INST(R, POT)                                                                              \
    template __global__ void k_mutual_grp<R, POT>(const float4*, const GroupTask*, int, const MutualTask*,     \
                                                  const SimDesc*, const RowDesc*, float*, float*, float*);
GI_MUTUAL_GRP_INST(4, false)
GI_MUTUAL_GRP_INST(8, false)
GI_MUTUAL_GRP_INST(4, true)
GI_MUTUAL_GRP_INST(8, true)
#undef GI_MUTUAL_GRP_INST

}  // namespace gi
