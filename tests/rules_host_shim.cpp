// Host build of haissinskijulia_amd/csrc/hm_rules.hpp for tests/test_rules.py.
#include "../haissinskijulia_amd/csrc/hm_rules.hpp"

extern "C" {
int64_t t_max_slabs(int64_t ntiles, int64_t ppt, int cus) { return hm::max_slabs(ntiles, ppt, cus); }
// the form of a lone bunch: -1 32-bit counts, 0 global memory, else the window
int t_hist_form(int64_t nb, int64_t ntiles, int64_t npairs, int64_t ppt, int lds) {
    const int w = hm::hist_window(nb, npairs, ppt, lds);
    if (w < 0) return -1;
    if (w > 0 && (!hm::hist_fits(nb, lds) || hm::hist_window_pays(npairs, ntiles))) return w;
    return hm::hist_fits(nb, lds) ? -1 : 0;
}
int64_t t_pairs_per_tile(int64_t npairs, int tile_pairs) { return hm::pairs_per_tile_for(npairs, 1024, tile_pairs); }
int t_spreads(int64_t tiles, int64_t nb, int global) { return hm::spreads_counters(tiles, nb, global != 0); }
int t_cached(const int64_t *n, int count) {
    int64_t bytes = 0;
    for (int i = 0; i < count; ++i) bytes += hm::cached_bytes(n[i]);
    return bytes <= hm::kCachedBytes;
}
int t_keeps_z(int64_t zbytes, int interp) { return hm::keeps_z(zbytes, interp != 0); }
int64_t t_free_turns(int64_t pairs) { return hm::free_turns_per_launch(pairs); }
int64_t t_free_pairs(int64_t pairs) { return hm::free_pairs_per_thread(pairs, 256, 256); }
}
