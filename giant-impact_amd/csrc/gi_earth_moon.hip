// gi_earth_moon.hip -- the Earth / Moon finder and the final statistics on the
// device (findEarthAndMoon and the get*Collision sums of
// Code/ImpactCode/impactBasicFunctions.h:109-217,219-652).
//
// The reference floods groups of elements closer than touch = 1.5 diameters
// on the host, O(N^2) per group, numbering each group by the index of its
// first (smallest) element; the Earth is the largest group and the Moon the
// next largest, ties going to the smaller number.  Here:
//   1. a hashed cell grid with cells a little larger than touch (cell
//      coordinates in FP64, so a touching pair always lies in adjacent cells);
//   2. union-find over the touching pairs found in a cell and its 13 forward
//      neighbours, always hooking the larger root under the smaller (lock-free
//      CAS), so every root is the smallest index of its component -- the
//      reference's group number;
//   3. component sizes by integer atomics (one per workgroup for the group
//      that fills it), the two largest by (size, ~root);
//   4. FP64 moments (mass, mass-weighted position, momentum, position x
//      momentum) of the whole system, the Earth and the Moon, with element
//      counts by body and material, per block in a fixed order, and the
//      blocks' sums and the result's record on the device, so that a call
//      copies one record to the host and waits once.
// Everything is deterministic: the components are unique, the counts are
// integers and the FP64 sums run in a fixed order.
#pragma once

#include "../../include/giant_impact.h"
#include "gi_device.h"

namespace gi {

// Cell coordinate of x for cells of size c, in FP64 (the float product x / c
// could misplace far-out elements by a cell), clamped like cell_coord.
__device__ __forceinline__ int cc_cell(float x, double inv_c) {
    double f = floor((double)x * inv_c);
    f = fmin(fmax(f, -1.0e9), 1.0e9);  // NaN -> -1e9
    return (int)f;
}

// The reference's touch test: mag = sqrt(dx*dx + dy*dy + dz*dz) < touch, all
// in float, products and sums rounded one by one
// (impactBasicFunctions.h:136-140).
__device__ __forceinline__ bool cc_touch(float4 a, float4 b, float touch) {
    const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
    const float r2 = dx * dx + dy * dy + dz * dz;
    return sqrtf(r2) < touch;
}

__global__ void k_cc_count(const float4* __restrict__ pos, int n, double inv_c, unsigned hmask,
                           int* __restrict__ counts, int* __restrict__ cellhash, int* __restrict__ size) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos[i];
    const unsigned h = cell_bucket(0, hmask, cc_cell(p.x, inv_c), cc_cell(p.y, inv_c), cc_cell(p.z, inv_c));
    cellhash[i] = (int)h;
    atomicAdd(&counts[h], 1);
    size[i] = 0;
}

// Particles into their buckets: position and, in w, index.  The order inside
// a bucket does not matter (the groups are unique).
__global__ void k_cc_scatter(const float4* __restrict__ pos, int n, const int* __restrict__ cellhash,
                             const int* __restrict__ starts, int* __restrict__ counts, float4* __restrict__ spos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int h = cellhash[i];
    float4 p = pos[i];
    p.w = __int_as_float(i);
    spos[starts[h] + atomicSub(&counts[h], 1) - 1] = p;
}

__device__ __forceinline__ int cc_load(const int* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Root of x.  Parents only ever point to smaller indices, so the walk ends.
__device__ __forceinline__ int cc_find(int* parent, int x) {
    int p = cc_load(parent + x);
    while (p != x) {
        const int gp = cc_load(parent + p);
        if (gp != p) {
            // path halving; a racing update can only have made parent[x]
            // smaller, and a lost write is harmless
            __hip_atomic_store(parent + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        x = p;
        p = gp;
    }
    return x;
}

// Unites a and b; returns an ancestor of both.  Most pairs are united
// already with the same parent: one round trip finds that out.
__device__ __forceinline__ int cc_union(int* parent, int a, int b) {
    const int pa = cc_load(parent + a), pb = cc_load(parent + b);
    if (pa == pb) return pa;
    a = pa;
    b = pb;
    while (true) {
        int ra = cc_find(parent, a);
        int rb = cc_find(parent, b);
        if (ra == rb) return ra;
        if (ra < rb) {
            const int t = ra;
            ra = rb;
            rb = t;
        }
        // hook the larger root under the smaller one
        int expected = ra;
        if (__hip_atomic_compare_exchange_strong(parent + ra, &expected, rb, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return rb;
        a = ra;
        b = rb;
    }
}

// Every touching pair is united: of particle t (in bucket order) with the
// later ones of its own bucket and with those of its 13 forward neighbour
// cells, cut into the five rows of cells (dy, dz) = (0, 0), (1, 0), (-1, 1),
// (0, 1), (1, 1).  A bucket may hold other cells' particles: a touching pair
// is a touching pair wherever it is found, so no candidate's cell is compared.
//
// Bound by the latency of the finds (loads and compare-and-swaps that other
// CUs' updates keep out of the L1).  Consecutive buckets are close in space,
// so most touching pairs lie in one workgroup's run of kCCLocal particles:
// k_cc_local unites those in LDS and leaves each particle pointing at the
// smallest index of its local group; k_cc_union then unites the pairs that
// cross runs, a lane per (particle, row of cells).  N = 65,536: 22 + 64 us, and
// 197 us a call; runs of 512 with a lane per particle 45 + 53 us and 222 a
// call, of 512 with two 27 + 56, of 256 with two 25 + 65 and 203 a call; every
// pair united globally, five lanes a particle 136-166 us, one lane over all 27
// cells with an index load per candidate 350 us.  (In k_cc_union, one union
// per pair of groups in a wavefront, or four candidates' loads in flight with
// their groups looked up beside them: 62 and 77 us.)
constexpr int kCCRows = 5;
// (320 and 3 were chosen at that size, where the runs give 205 workgroups; a
// call takes 135, 144, 181, 251 and 462 us at N = 12,287, 20,000, 55,555,
// 98,000 and 131,000, and 590, 680, 1,150, 1,600 and 2,240 with every pair
// united globally.)
constexpr int kCCLocal = 320;     // particles of a run
constexpr int kCCLocalLanes = 3;  // lanes per particle of k_cc_local, which share its rows

// Buckets of row `row` (0..4) of the cell (cx, cy, cz): candidates
// [k0[o], k1[o]).  t: the particle's own place.
__device__ __forceinline__ void cc_row(int cx, int cy, int cz, int row, int t, unsigned hmask,
                                       const int* __restrict__ starts, int (&k0)[3], int (&k1)[3]) {
    const int qy = cy + (row == 0 ? 0 : row == 1 ? 1 : row - 3), qz = cz + (row >= 2 ? 1 : 0);
#pragma unroll
    for (int o = 0; o < 3; ++o) {
        const unsigned h = cell_bucket(0, hmask, cx + o - 1, qy, qz);
        k0[o] = starts[h];
        k1[o] = starts[h + 1];
    }
    if (row == 0) {
        k1[0] = k0[0];  // the cell behind has this one ahead
        k0[1] = t + 1;
    }
}

__device__ __forceinline__ int cc_lds_find(int* parent, int x) {
    int p = __hip_atomic_load(parent + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (p != x) {
        const int gp = __hip_atomic_load(parent + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (gp != p) __hip_atomic_store(parent + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        x = p;
        p = gp;
    }
    return x;
}

__global__ __launch_bounds__(kCCLocal * kCCLocalLanes) void k_cc_local(const float4* __restrict__ spos, int n, double inv_c,
                                                       unsigned hmask, float touch, const int* __restrict__ starts,
                                                       int* __restrict__ parent) {
    __shared__ float4 sp[kCCLocal];
    __shared__ int up[kCCLocal], least[kCCLocal];
    const int b0 = blockIdx.x * kCCLocal, b1 = min(b0 + kCCLocal, n);
    const int l = threadIdx.x % kCCLocal, part = threadIdx.x / kCCLocal, t = b0 + l;
    const bool live = t < n;
    const float4 pi = live ? spos[t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const int i = __float_as_int(pi.w);
    if (part == 0) {
        sp[l] = pi;
        up[l] = l;
        least[l] = 0x7fffffff;
    }
    __syncthreads();
    if (live) {
        const int cx = cc_cell(pi.x, inv_c), cy = cc_cell(pi.y, inv_c), cz = cc_cell(pi.z, inv_c);
        constexpr int rows = (kCCRows + kCCLocalLanes - 1) / kCCLocalLanes;  // of this lane's rows part, part + lanes, ...
        int k0[rows][3] = {}, k1[rows][3] = {};  // all the bounds' loads in flight at once
#pragma unroll
        for (int row = 0; row < rows; ++row) {
            const int r = part + row * kCCLocalLanes;
            if (r < kCCRows) cc_row(cx, cy, cz, r, t, hmask, starts, k0[row], k1[row]);
        }
#pragma unroll
        for (int row = 0; row < rows; ++row) {
#pragma unroll
            for (int o = 0; o < 3; ++o)
                for (int k = max(k0[row][o], b0); k < min(k1[row][o], b1); ++k) {
                    if (!cc_touch(pi, sp[k - b0], touch)) continue;
                    int a = l, b = k - b0;
                    while (true) {
                        a = cc_lds_find(up, a);
                        b = cc_lds_find(up, b);
                        if (a == b) break;
                        if (a < b) {
                            const int x = a;
                            a = b;
                            b = x;
                        }
                        int expected = a;
                        if (__hip_atomic_compare_exchange_strong(up + a, &expected, b, __ATOMIC_RELAXED,
                                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
                            break;
                    }
                }
        }
    }
    __syncthreads();
    if (live && part == 0) atomicMin(&least[cc_lds_find(up, l)], i);
    __syncthreads();
    if (live && part == 0) parent[i] = least[cc_lds_find(up, l)];
}

constexpr int kCCUnionWaves = 4;
constexpr int kCCUnionPer = kCCUnionWaves * (64 / kCCRows);  // particles per workgroup

__global__ __launch_bounds__(64 * kCCUnionWaves) void k_cc_union(const float4* __restrict__ spos, int n, double inv_c,
                                                                unsigned hmask, float touch,
                                                                const int* __restrict__ starts,
                                                                int* __restrict__ parent) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int slot = lane / kCCRows, row = lane % kCCRows;
    const int t = blockIdx.x * kCCUnionPer + w * (64 / kCCRows) + slot;
    if (slot >= 64 / kCCRows || t >= n) return;
    const float4 pi = spos[t];
    int k0[3], k1[3];
    cc_row(cc_cell(pi.x, inv_c), cc_cell(pi.y, inv_c), cc_cell(pi.z, inv_c), row, t, hmask, starts, k0, k1);
    const int b0 = t / kCCLocal * kCCLocal, b1 = b0 + kCCLocal;  // this particle's own run: united already
    int a = __float_as_int(pi.w);                                // an ancestor of the particle
#pragma unroll
    for (int o = 0; o < 3; ++o) {
        const int e = k1[o];
        for (int k = k0[o]; k < e; ++k) {
            if (k >= b0 && k < b1) {
                k = b1 - 1;
                continue;
            }
            const float4 pj = spos[k];
            if (cc_touch(pi, pj, touch)) a = cc_union(parent, a, __float_as_int(pj.w));
        }
    }
}

// Root of x without path compression: after the unions the forest is fixed,
// and the only stores to parent are each thread's own final root.
__device__ __forceinline__ int cc_root(const int* parent, int x) {
    int p = cc_load(parent + x);
    while (p != x) {
        x = p;
        p = cc_load(parent + x);
    }
    return x;
}

// root[i] = the smallest index of i's component; size[root]++.  The walk
// must not compress paths: a path-splitting store from another thread's walk
// (a grandparent, not necessarily the root) could land after i's own root
// store and leave parent[i] pointing at an inner node.  Reading a parent
// that another thread has just replaced by its root is harmless: both are
// ancestors.
// The sizes are counted a workgroup at a time for the group of its first
// element (an atomic per element on the size of the largest group took 535 us
// at N = 65,536), and then a wavefront at a time for one other group.
constexpr int kCCCompressThreads = 1024;
__global__ __launch_bounds__(kCCCompressThreads) void k_cc_compress(int* __restrict__ parent, int* __restrict__ size,
                                                                    int n, int* __restrict__ group) {
    __shared__ int common, held;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < n;
    int r = -1;
    if (live) {
        r = cc_root(parent, i);
        __hip_atomic_store(parent + i, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (group) group[i] = r;
    }
    if (threadIdx.x == 0) {
        common = r;
        held = 0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const unsigned long long same = __ballot(live && r == common);
    if (lane == 0 && same) atomicAdd(&held, __popcll(same));
    const unsigned long long others = __ballot(live && r != common);
    if (others) {
        const int lead = __shfl(r, __ffsll((long long)others) - 1);
        const unsigned long long with = __ballot(live && r == lead);
        if (live && r != common) {
            if (r != lead)
                atomicAdd(&size[r], 1);
            else if (lane == __ffsll((long long)with) - 1)
                atomicAdd(&size[r], __popcll(with));
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(&size[common], held);
}

// The two largest components as keys (size << 32 | ~root): ties to the
// smaller root, 0 for none.
struct CCTop {
    unsigned long long first, second;
    int groups, pad;
};

__device__ __forceinline__ void cc_merge(CCTop& a, const CCTop& b) {
    const unsigned long long lo = min(a.first, b.first), hi = max(a.second, b.second);
    a.first = max(a.first, b.first);
    a.second = max(lo, hi);
    a.groups += b.groups;
}

// Over the workgroup's lanes; the result is on thread 0.
__device__ __forceinline__ CCTop cc_block_top(CCTop t) {
    __shared__ CCTop part[kCCCompressThreads / 64];
#pragma unroll
    for (int m = 32; m; m >>= 1) {
        CCTop o;
        o.first = __shfl_xor(t.first, m);
        o.second = __shfl_xor(t.second, m);
        o.groups = __shfl_xor(t.groups, m);
        cc_merge(t, o);
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0)
        for (unsigned w = 1; w < blockDim.x / 64; ++w) cc_merge(t, part[w]);
    return t;
}

constexpr int kCCTopBlocks = 256;
__global__ __launch_bounds__(256) void k_cc_top(const int* __restrict__ size, int n, CCTop* __restrict__ out) {
    CCTop t{0ull, 0ull, 0, 0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int s = size[i];
        if (s == 0) continue;
        cc_merge(t, CCTop{((unsigned long long)(unsigned)s << 32) | (unsigned long long)(~(unsigned)i), 0ull, 1, 0});
    }
    t = cc_block_top(t);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

__device__ __forceinline__ int cc_key_root(unsigned long long key) {
    return key ? (int)~(unsigned)(key & 0xffffffffull) : -1;
}

// Moments of one class: mass, sum m x (3), sum m v (3), sum m x cross v (3).
constexpr int kCCMoments = 10;
constexpr int kCCClasses = 3;  // 0 whole system, 1 Earth, 2 Moon
constexpr int kCCCounts = 8;   // Earth then Moon: Fe body 1, Fe body 2, Si body 1, Si body 2
constexpr int kCCBlock = 256;

// Sum over the wavefront, in every lane.
__device__ __forceinline__ double cc_wave_sum(double v) {
#pragma unroll
    for (int m = 32; m; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

// Per block: the moments of the system, the Earth and the Moon (FP64, a fixed
// grid-stride order and a fixed tree: lanes, then the four wavefronts) and
// the element counts of the Earth and the Moon by body and material.  The
// impact layout is [Fe1, Fe2, Si1, Si2] (impactBasicFunctions.h:910-924).
__global__ __launch_bounds__(kCCBlock) void k_cc_moments(const float4* __restrict__ pos,
                                                         const float4* __restrict__ vel, int n,
                                                         const int* __restrict__ root,
                                                         const CCTop* __restrict__ tops, int ntops,
                                                         CCTop* __restrict__ best, int nfe1, int nfe2, int nsi1,
                                                         double mass_fe, double mass_si, double* __restrict__ out,
                                                         int* __restrict__ counts) {
    constexpr int kWaves = kCCBlock / 64, kAll = kCCClasses * kCCMoments;
    __shared__ double red[kWaves][kAll];
    __shared__ int cnt[kWaves][kCCCounts];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // the two largest groups from the blocks' (every workgroup for itself)
    static_assert(kCCTopBlocks == kCCBlock, "a block's pair per lane");
    __shared__ CCTop top;
    CCTop mine{0ull, 0ull, 0, 0};
    if ((int)threadIdx.x < ntops) mine = tops[threadIdx.x];
    mine = cc_block_top(mine);
    if (threadIdx.x == 0) {
        top = mine;
        if (blockIdx.x == 0) *best = mine;
    }
    __syncthreads();
    const int earth = cc_key_root(top.first), moon = cc_key_root(top.second);
    double m[kCCClasses][kCCMoments];
#pragma unroll
    for (int c = 0; c < kCCClasses; ++c)
#pragma unroll
        for (int k = 0; k < kCCMoments; ++k) m[c][k] = 0.0;
    int have[kCCCounts] = {};
    const int nfe = nfe1 + nfe2;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double mi = i < nfe ? mass_fe : mass_si;
        const float4 p = pos[i], v = vel[i];
        const double x = p.x, y = p.y, z = p.z, vx = v.x, vy = v.y, vz = v.z;
        const double t[kCCMoments] = {mi,          mi * x,      mi * y,      mi * z,      mi * vx,
                                      mi * vy,     mi * vz,     mi * (y * vz - z * vy),
                                      mi * (z * vx - x * vz),   mi * (x * vy - y * vx)};
        const int r = root[i];
        const int cls = r == earth ? 1 : (r == moon ? 2 : 0);
#pragma unroll
        for (int k = 0; k < kCCMoments; ++k) {
            m[0][k] += t[k];
            if (cls == 1) m[1][k] += t[k];
            if (cls == 2) m[2][k] += t[k];
        }
        const int kind = i < nfe1 ? 0 : (i < nfe ? 1 : (i < nfe + nsi1 ? 2 : 3));
#pragma unroll
        for (int k = 0; k < kCCCounts; ++k) have[k] += cls == 1 + k / 4 && kind == k % 4;
    }
#pragma unroll
    for (int c = 0; c < kCCClasses; ++c)
#pragma unroll
        for (int k = 0; k < kCCMoments; ++k) {
            const double s = cc_wave_sum(m[c][k]);
            if (lane == 0) red[w][c * kCCMoments + k] = s;
        }
#pragma unroll
    for (int k = 0; k < kCCCounts; ++k) {
        int s = have[k];
#pragma unroll
        for (int x = 32; x; x >>= 1) s += __shfl_xor(s, x);
        if (lane == 0) cnt[w][k] = s;
    }
    __syncthreads();
    if (threadIdx.x < kAll) {
        double s = red[0][threadIdx.x];
#pragma unroll
        for (int x = 1; x < kWaves; ++x) s += red[x][threadIdx.x];
        out[(size_t)blockIdx.x * kAll + threadIdx.x] = s;
    }
    if (threadIdx.x < kCCCounts) {
        int s = 0;
#pragma unroll
        for (int x = 0; x < kWaves; ++x) s += cnt[x][threadIdx.x];
        counts[blockIdx.x * kCCCounts + threadIdx.x] = s;
    }
}

// The blocks' sums, in a fixed order, and the result's record.  Scope 1
// (Earth-Moon) = Earth + Moon; 0 / 0 = NaN for an empty scope, as the
// reference divides; L about the scope's centre of mass relative to its mean
// velocity: sum m x cross v - (sum m x) cross (sum m v) / M.
constexpr int kCCFinalSegs = 16;
__global__ __launch_bounds__(32 * kCCFinalSegs) void k_cc_final(const double* __restrict__ mom,
                                                               const int* __restrict__ cnt, int nb,
                                                               const CCTop* __restrict__ best,
                                                               gi_earth_moon* __restrict__ out) {
    constexpr int kAll = kCCClasses * kCCMoments;
    static_assert(kAll <= 32 && kCCCounts <= 32, "a column per lane");
    __shared__ double M[4][kCCMoments];
    __shared__ double part[kCCFinalSegs][32];
    __shared__ int cpart[kCCFinalSegs][32];
    const int l = threadIdx.x;
    // kCCFinalSegs runs of blocks side by side, then the runs in order
    const int col = l & 31, seg = l >> 5;
    const int s0 = nb * seg / kCCFinalSegs, s1 = nb * (seg + 1) / kCCFinalSegs;
    double s = 0.0;
    int c = 0;
    if (col < kAll)
#pragma unroll 8
        for (int b = s0; b < s1; ++b) s += mom[(size_t)b * kAll + col];
    if (col < kCCCounts)
#pragma unroll 8
        for (int b = s0; b < s1; ++b) c += cnt[b * kCCCounts + col];
    part[seg][col] = s;
    cpart[seg][col] = c;
    __syncthreads();
    if (seg == 0 && col < kAll) {
        for (int k = 1; k < kCCFinalSegs; ++k) s += part[k][col];
        const int scope = col / kCCMoments;
        M[scope == 0 ? 0 : scope + 1][col % kCCMoments] = s;
    }
    if (seg == 1 && col < kCCCounts) {
        c = 0;
        for (int k = 0; k < kCCFinalSegs; ++k) c += cpart[k][col];
        (&out->earth_fe1)[col] = c;
    }
    __syncthreads();
    if (l < kCCMoments) M[1][l] = M[2][l] + M[3][l];
    __syncthreads();
    if (l == 0) {
        out->n_groups = best->groups;
        out->earth_id = cc_key_root(best->first);
        out->moon_id = cc_key_root(best->second);
        out->earth_count = (int)(best->first >> 32);
        out->moon_count = (int)(best->second >> 32);
    }
    if (l < 4) {
        const double* a = M[l];
        const double mass = a[0];
        out->mass[l] = mass;
        for (int d = 0; d < 3; ++d) {
            out->com[l][d] = a[1 + d] / mass;
            out->vel[l][d] = a[4 + d] / mass;
        }
        const double* X = a + 1;
        const double* Pm = a + 4;
        out->angmom[l][0] = a[7] - (X[1] * Pm[2] - X[2] * Pm[1]) / mass;
        out->angmom[l][1] = a[8] - (X[2] * Pm[0] - X[0] * Pm[2]) / mass;
        out->angmom[l][2] = a[9] - (X[0] * Pm[1] - X[1] * Pm[0]) / mass;
    }
}

}  // namespace gi
