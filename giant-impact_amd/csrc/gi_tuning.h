// gi_tuning.h -- tiling of the all-pairs pass and its tuning table.
//
// R            i-particles held in registers per lane (a wavefront covers 64*R)
// variant      0 = one-sided pass, r^-3 as rsq cubed; 1 = one-sided, rsq *
//              rcp (1 multiply, 2 transcendental ops); 2 = mutual pass (each
//              pair once for both particles, rows of 64*R, rsq cubed);
//              3 = direct pass (small simulations: the whole force in one
//              launch, the same whatever R is; R = 1, 2, 4 or 8 lanes per
//              particle of its energy pass; the sizes unused);
//              4 = mutual pass with row groups (a workgroup's four
//              wavefronts hold four rows and add their j-side sums in LDS
//              before writing them: a quarter of the j-side slab; R = 4 or 8)
// chunk_len    j-particles per task (0 = derive from target_tasks)
// target_tasks wavefront tasks to aim for (several per SIMD of the 256 CUs x
//              4 SIMDs so the tail of the launch stays short)
// min_chunk    lower bound on chunk_len (each chunk costs one partial slot
//              per particle)
//
// The table is written by the autotuner (gi_amd.autotune) to
// tuning/<arch>.txt next to the library's lib/ directory, one row per size
// class: "n_max R variant chunk_len target_tasks min_chunk" (particles of
// one simulation, or sqrt(sum n^2) of several; rows in increasing n_max).  Without a table the defaults
// below apply.
#pragma once

#include <dlfcn.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

namespace gi {

struct Tiling {
    int R;
    int variant;
    long long chunk_len;
    long long target_tasks;
    long long min_chunk;
};

struct TilingOverride {
    int active = 0;
    Tiling t{4, 0, 0, 8192, 512};
};

inline TilingOverride& tiling_override() {
    static TilingOverride o;
    return o;
}

struct TuningRow {
    long long n_max;
    Tiling t;
};

inline void tuning_anchor() {}

// Rows of tuning/gfx950.txt, located relative to this shared library.
inline const std::vector<TuningRow>& tuning_table() {
    static std::vector<TuningRow> rows;
    static std::once_flag once;
    std::call_once(once, [] {
        Dl_info info;
        if (!dladdr((void*)&tuning_anchor, &info) || !info.dli_fname) return;
        std::string path(info.dli_fname);
        size_t cut = path.rfind('/');
        if (cut == std::string::npos) return;
        path = path.substr(0, cut);  // .../lib
        cut = path.rfind('/');
        path = (cut == std::string::npos ? std::string(".") : path.substr(0, cut)) + "/tuning/gfx950.txt";
        FILE* f = std::fopen(path.c_str(), "r");
        if (!f) return;
        char line[256];
        while (std::fgets(line, sizeof line, f)) {
            if (line[0] == '#') continue;
            TuningRow r;
            if (std::sscanf(line, "%lld %d %d %lld %lld %lld", &r.n_max, &r.t.R, &r.t.variant, &r.t.chunk_len,
                            &r.t.target_tasks, &r.t.min_chunk) == 6 &&
                (r.t.R == 1 || r.t.R == 2 || r.t.R == 4 || r.t.R == 8) && r.t.variant >= 0 && r.t.variant <= 4 &&
                (r.t.variant != 4 || r.t.R >= 4) &&
                r.t.chunk_len >= 0 && r.t.target_tasks >= 0 &&
                (r.t.target_tasks > 0 || r.t.chunk_len > 0 || r.t.variant == 3))
                rows.push_back(r);
        }
        std::fclose(f);
    });
    return rows;
}

// Tiling of the batched engine (ensembles and the request loop): one j-chunk
// length for every simulation, whatever its size or company, so that a
// simulation's sums are the same in any batch.  Row "B chunk_len R [variant]"
// of the tuning file; gi_set_batched_tiling overrides it.
struct BatchedTiling {
    long long chunk_len;
    int R;
    int variant;
};

inline BatchedTiling& batched_override() {
    static BatchedTiling b{0, 0, 0};
    return b;
}

inline BatchedTiling batched_tiling() {
    if (batched_override().chunk_len > 0) return batched_override();
    static BatchedTiling from_file{0, 0, 0};
    static std::once_flag once;
    std::call_once(once, [] {
        Dl_info info;
        if (!dladdr((void*)&tuning_anchor, &info) || !info.dli_fname) return;
        std::string path(info.dli_fname);
        size_t cut = path.rfind('/');
        if (cut == std::string::npos) return;
        path = path.substr(0, cut);
        cut = path.rfind('/');
        path = (cut == std::string::npos ? std::string(".") : path.substr(0, cut)) + "/tuning/gfx950.txt";
        FILE* f = std::fopen(path.c_str(), "r");
        if (!f) return;
        char line[256];
        while (std::fgets(line, sizeof line, f)) {
            long long L;
            int R, V = 0;
            const int got = std::sscanf(line, "B %lld %d %d", &L, &R, &V);
            if (got >= 2 && L >= 64 && (R == 1 || R == 2 || R == 4 || R == 8) &&
                (V == 0 || V == 1 || V == 2 || (V == 4 && R >= 4)))
                from_file = BatchedTiling{L, R, V};
        }
        std::fclose(f);
    });
    if (from_file.chunk_len > 0) return from_file;
    return BatchedTiling{4096, 1, 0};
}

// j per piece of a simulation of n particles in the batched engine, whose
// full length is L0.  A piece costs a slot per particle of its rows, written
// and added, and a task's start; a company of a few small simulations lasts as
// long as its longest tasks, a full GPU the longer the more pieces there are.
// What is in company must not change a simulation's sums, so one length has to
// do for both.  Steps of equal simulations, against pieces of n / 32 in lists
// longest first and the walk by particles alone (alone: of a small company,
// then of a GPU full of them):
//   64 to 3,072: 2 of 2,600 94 -> 59 us, 150 of them 356 ->
//     322; up to 4,096 they cost 256 simulations 9%;
//   n / 40 to 16,384: 2 of 4,501 112 -> 73, 150 759 -> 691; 2 of 9,001 162 ->
//     95, 150 2,321 -> 2,330; n / 80 takes 85 and 2,469, and 256 simulations
//     of 4,096 9% longer, 150 of 3,700 to 9,800 3 to 6%;
//   256 at most there: 2 of 12,701 164 -> 115, 64 1,845 -> 1,876; n / 80 takes
//     110 and 1,906, n / 48 (320) 3 of 12,700 to 13,600 10% longer than n / 32;
//     64 simulations of 10,600 to 15,700 1% longer on average, 32 3% shorter;
//   n / 48 to 24,576: 2 of 23,399 304 -> 257, 16 1,673 -> 1,519, 64 the same
//     within 0.6%; 3 of 17,600 and 22,500 11 and 4% longer, where the tasks
//     divide badly among the CUs;
//   n / 32 above: one of 30,000 is 2% faster so than at n / 48.
inline long long batched_piece_len(long long n, long long L0) {
    long long L = n <= 3072 ? 64 : n <= 16384 ? n / 40 : n <= 24576 ? n / 48 : n / 32;
    if (n <= 16384 && L > 256) L = 256;
    return std::min(L0, std::max(64LL, (L + 63) / 64 * 64));
}

// The row for a launch of ntot particles.  Several simulations in one launch
// (the separate bodies) have the work of one with as many pairs, sum n^2,
// and are placed by that size: two of 6,200 (8,768) and two of 8,000 (11,314)
// step in 43 and 58 us by the direct pass's rows, in 55 and 66 by the rows of
// 12,400 and 16,000.
inline Tiling choose_tiling(long long ntot, long long pairs, int nsims) {
    if (tiling_override().active) return tiling_override().t;
    if (nsims > 1) ntot = (long long)std::ceil(std::sqrt((double)pairs));
    for (const TuningRow& r : tuning_table())
        if (ntot <= r.n_max) return r.t;
    Tiling t{4, 0, 0, 8192, 512};
    if (ntot < 4096) t.min_chunk = 128;
    return t;
}

// Whether the contact walk of a plan of so many particles and pairs (sum
// n^2) takes nine lanes per particle.  One lane's walk is a chain of 27 cells
// that the all-pairs pass hides only if it is long enough; nine lanes take a
// ninth of the time and more of the chip, which a pass that fills it pays
// for.  Measured as whole steps of 8 to 384 equal simulations of 1,100 to
// 12,000 particles, nine lanes against one: 1.75 times as fast for 8 of 2,048
// (16,384 particles), 1.23 for 32 of 4,096, 1.07 for 96 of 3,000, 1.03 for 64
// of 4,096, 1.05 for 16 of 8,000, 1.13 for 8 of 12,000; the same for 192 of
// 2,048, 128 of 3,000, 96 of 4,096, 32 of 8,000 and 16 of 12,000; 0.90 for
// 384 of 2,048, 0.96 for 256 of 4,096, 0.97 for 48 of 8,000, 0.98 for 64 of
// 12,000.  The line through those; one simulation, whose pass is the shorter
// for its particles, to 49,152.
inline bool contact_walk_by_rows(double particles, double pairs) {
    return pairs <= 49152.0 * 49152.0 && particles / 450000.0 + pairs / 3.0e9 <= 1.0;
}

}  // namespace gi
