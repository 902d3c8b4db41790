// hm_rules.hpp -- choices of the engine that depend on sizes alone: no device
// code, so that the CPU can check them.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace hm {

// Pairs per tile of a bunch.
inline int64_t pairs_per_tile_for(int64_t npairs, int threads, int32_t tile_pairs) {
    // tiling depends on the bunch size (and the option) alone, so a bunch is
    // reduced in the same order alone and in any batch: by default about 1024
    // tiles of a large bunch (four per CU), at least one pair per thread.  A
    // workgroup streams its run of consecutive tiles of a bunch as one loop,
    // so small tiles cost no extra pipeline start.
    if (tile_pairs > 0) return (int64_t)tile_pairs * threads;
    const int64_t target_tiles = 1024;
    int64_t ppt = (npairs + target_tiles - 1) / target_tiles;
    ppt = ((ppt + threads - 1) / threads) * threads;
    return std::max<int64_t>(ppt, (int64_t)threads);
}

// Histograms of more bins than the LDS holds 32-bit counts for (F_GHIST).  An
// addition to global memory per particle was bound by the crowded lines: 1e7
// particles, 131072 bins: a pass of 0.40 ms; 45056 bins 0.54 ms.  So the pass
// counts a window of kHistWin bins around the centroid in LDS, in 16 bits (a run
// has at most kHistRunPairs pairs, so they cannot overflow), stores each run's
// window to a slab of its own without atomics, and k_hist_slabs adds the slabs
// up; only particles outside the window add to global memory: 0.108 ms and
// 0.083 ms.  49152 bins are +-2.8 sigma of a bunch on 131072 bins over +-7.5
// sigma (one particle in 200 outside) and leave 8000 entries for the window of
// P, which the kick reads; 32768, 40960 and 57344 bins: 0.084, 0.085 and 0.098
// ms against 0.089 at 65536 bins, 0.105, 0.105 and 0.111 at 131072, but 0.173,
// 0.153 and 0.138 against 0.145 at 262144.  Tiles of more than kHistRunPairs pairs
// cannot use 16 bits; kHistMaxPairs bounds the slabs of one bunch to a few
// hundred MB.
constexpr int kHistWin = 49152;
constexpr int kHistRunPairs = 32767;
constexpr int64_t kHistMaxPairs = 1 << 26;
constexpr int kHistMinWin = 3072;

// 32-bit counts of nb bins in LDS, beside two entries of P at least (the
// all-flags pass relies on that): up to 40700 bins.
inline bool hist_fits(int64_t nb, int lds_max) { return 4 * nb + 16 <= (int64_t)lds_max - 1024; }

// The bins of a bunch's window, 0 where it cannot have one, or -1 where it needs
// none: 32-bit counts leave kHistMinWin entries of P (up to 34560 bins).
inline int hist_window(int64_t nb, int64_t npairs, int64_t ppt, int lds_max) {
    if (hist_fits(nb + 2 * kHistMinWin - 4, lds_max)) return -1;
    return ppt <= kHistRunPairs && npairs <= kHistMaxPairs ? (int)std::min<int64_t>(nb, kHistWin) & ~1 : 0;
}

// Whether the bunches of a launch that can have either, 34561 to 40700 bins, take
// the window, from the pairs and tiles of all its windowed bunches.  Its pass
// gathers less of P from global memory, for a launch and slabs that grow to 25 MB
// (one per workgroup) between 1e4 and 5e5 particles and no further.  The counts,
// and with them the results, are the same.  A turn by 32 bits and by the window, the
// energy update on (reference lattice, off), in us:
//   particles     34600 bins                 38000 bins                 40600 bins
//   2e4       46.8, 45.6  (37.4, 38.0)   47.8, 45.8  (38.1, 38.5)   48.4, 46.4  (38.6, 38.6)
//   5e4       46.8, 46.7  (37.2, 39.0)   47.8, 47.4  (38.0, 39.3)   48.7, 47.9  (38.5, 39.6)
//   1e5       47.0, 49.5  (37.4, 41.6)   48.0, 50.2  (38.2, 42.3)   48.9, 51.4  (38.6, 43.1)
//   1e6       57.4, 64.1  (46.3, 55.0)   60.1, 64.7  (47.1, 55.0)   60.6, 65.0  (48.0, 54.9)
//   2e6       64.7, 68.7  (53.9, 58.0)   68.7, 69.8  (55.5, 58.6)   69.9, 69.5  (55.7, 59.6)
//   2.5e6     76.5, 80.3  (63.2, 68.4)   82.3, 81.2  (66.3, 68.8)   86.3, 81.0  (70.3, 69.1)
//   3e6       78.8, 81.3  (65.5, 69.8)   85.7, 82.4  (70.2, 70.1)   90.3, 82.7  (74.3, 70.2)
//   1e7        138,  123  ( 113,  104)    155,  125  ( 130,  107)    164,  125  ( 136,  106)
// Several bunches at 36000 bins: two of 1e5 58, 67 (46, 57), sixteen of 1e5 120, 123
// (100, 107), two of 1e6 77, 80 (62, 67), two of 2e6 94, 86 (72, 70), five of 1e6 114,
// 100 (92, 82), twenty of 5e5 215, 200 (174, 170), 1.2e7 and 1e6 202, 157 (171, 133).
constexpr int64_t kHistMinPairs = 1250000;   // the window from here on,
constexpr int64_t kHistFewTiles = 24;        // and up to here
inline bool hist_window_pays(int64_t pairs, int64_t tiles) {
    return pairs >= kHistMinPairs || tiles <= kHistFewTiles;
}
// The most slabs the windowed histogram of a bunch of ntiles tiles of ppt pairs
// can fill, alone or in any batch, on a device of cus CUs.  The pass has at most
// a workgroup per CU, each with one stretch of the bunch's tiles, and a run of it
// per kHistRunPairs pairs: a stretch of t tiles makes at most (t + per - 1) / per
// runs.  A slab per run, two where tiles are split over two workgroups, which
// takes at most cus / 2 tiles.  1e6 particles 263, 1e7 376 (alone both fill 256).
inline int64_t max_slabs(int64_t ntiles, int64_t ppt, int cus) {
    const int64_t per = std::max<int64_t>(1, kHistRunPairs / ppt);
    const int64_t runs = std::min(ntiles, (ntiles + std::min<int64_t>(ntiles, cus) * (per - 1)) / per);
    return 2 * ntiles <= cus ? 2 * ntiles : runs;
}

// Whether the counters of a bunch leave every other 128 bytes out: additions of
// many workgroups to few consecutive counters queue at few memory channels.  98
// workgroups adding to 1024 counters of 8 bytes: 3.8 us back to back, 2.8 us so (an
// empty kernel 1.6); 246 workgroups and 512 counters of 4 bytes: 6.0 and 4.2 us; no
// difference from 16384 counters on, nor for 49 workgroups, where the bin phase,
// which reads twice the range, loses 0.2 us.  So from kSpreadTiles tiles on; but
// where every particle adds to global memory (global: neither form above fits), the
// gain turns with the bins.  Pass of 3e7 particles, back to back and so, us:
//   45000 bins 1384, 1142     65536  1194, 1139     98304  1191, 1153    104000  1322, 1146
//   112000     1163, 1167    125000  1164, 1222    131072  1171, 1236    138000  1151, 1204
//   150000     1160, 1169    155000  1228, 1160    160000  1216, 1162    262144  1224, 1171
// and of 1e8, 131072 bins 3831, 4081: back to back from 110000 to 150000 bins.
constexpr int kSpreadTiles = 32;
constexpr int64_t kPackedMin = 110000, kPackedMax = 150000;
inline bool spreads_counters(int64_t tiles, int64_t nb, bool global) {
    return tiles >= kSpreadTiles && !(global && nb >= kPackedMin && nb <= kPackedMax);
}

// The particles of bunches with a windowed histogram are read and written
// through the caches, by the pass and by the interpolation sums, where all of them
// and 10 MB of tables a bunch fit the 256 MB of the last one: many particles
// gather from the pair table, and those gathers wait behind the streams (131072
// bins, pass of 1e7 particles: 104 -> 75 us, 4e6: 51 -> 39, 1.3e7: 139 -> 113, 2e7:
// 205 -> 212; one of the two streaming past the caches undoes it).  A turn through
// them and past them, us: 65536 bins, 1.3e7 particles (218 MB) 156, 173; two bunches
// of 6e6 (212 MB) 152, 166, of 7e6 (244 MB) 190, 180, of 1e7 265, 242; three of 4e6
// (222 MB) 156, 172; six of 2e6 (252 MB) 203, 194; ten of 1e6 (260 MB) 217, 205; with
// 36000 and 262144 bins the line lies at the same particles.
constexpr int64_t kCachedBytes = 224ll << 20;
inline int64_t cached_bytes(int64_t n) { return 16 * n + 10000000; }

// Whether z of the active bunches (zbytes in all) goes through the caches, dE past
// them: where z fits the 256 MB of the last one and is not small, the pass and the
// interpolation sums (interp: some bunch has them) find it there again.  28
// bunches, 176 MB of z: 188 -> 170 us a turn; one bunch of 2.8e7 particles (224 MB)
// and 8192 bins 257 -> 239; of 4e7 346 -> 358; of 4e6 (32 MB) 62 -> 66, where z
// drives the bin phase's tables from the caches nearer to the CUs.  Where that
// turns, one bunch, past the caches and through them (three runs of each, 0.5 us):
//   particles     8.5e6         9e6           9.5e6         1e7           1.04e7        1.2e7
//   1024 bins     76.6, 78.3    78.0, 78.7    80.4, 81.1    82.7, 81.8    83.7, 83.6    92.5, 88.0
//   4096 bins     84.4, 87.2    85.5, 88.2    87.8, 89.9    90.8, 91.0    92.5, 93.2    101,  97.4
//   8192 bins     102,  105     105,  106     107,  105     111,  109     112,  110     122,  117
//   16384 bins    103,  107     106,  107     110,  108     112,  111     113,  112     126,  119
//   8192, E0 off  82.4, 86.7    83.8, 87.2    86.4, 87.6    88.2, 88.9    88.6, 89.5    99.7, 99.8
// so from 75 MB with the sums (8192 and 16384 bins), from 84 MB without.
constexpr int64_t kKeepMinInterp = 75000000, kKeepMin = 84000000, kKeepMax = 224ll << 20;
inline bool keeps_z(int64_t zbytes, bool interp) {
    return zbytes > (interp ? kKeepMinInterp : kKeepMin) && zbytes <= kKeepMax;
}

// Pairs per thread of k_free_turns: one until that fills the SIMDs several times
// over, then four in turn (3e6 particles: 6 rounds of waves either way), sixteen
// where a launch still has 32 workgroups per CU of them, and at most about 65536
// items.  A thread's next pair is on its way during the turns of the one before:
// a call of one turn of 1e8 particles takes 1180 to 1200 us (1257 to 1316 by a launch
// of the pass; with four pairs per thread, each loaded when its turn came, 1200 or,
// by the addresses of the two arrays, up to 1445); 3e7 particles, 40 turns, 4.17 ms with
// four, 4.45 with sixteen.
inline int64_t free_pairs_per_thread(int64_t pairs, int threads, int cus) {
    const int64_t wave = (int64_t)threads * cus;
    const int64_t per = pairs > 512 * wave ? 16 : pairs > 32 * wave ? 4 : 1;
    return std::max(per, pairs / ((int64_t)threads << 16) + 1);
}

// Turns of one launch of k_free_turns over `pairs` pairs, for about 40 ms: 4e9
// pair-turns fill the device (27 ms for 1e7 particles), and below 8e4 pairs a
// turn takes the 0.8 us of a thread's own chain however few there are.  Bounded
// by the pair-turns alone, a launch of a few thousand particles ran for 2^20
// turns, 0.8 s.
inline int64_t free_turns_per_launch(int64_t pairs) {
    return std::min<int64_t>(50000, std::max<int64_t>(1, (int64_t)4e9 / std::max<int64_t>(1, pairs)));
}

}  // namespace hm
