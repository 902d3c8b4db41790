"""The engine's choices by size (haissinskijulia_amd/csrc/hm_rules.hpp), compiled
for the CPU from the same source (CPU)."""
import ctypes as C
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    out = tmp_path_factory.mktemp("rules") / "libhmrules.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "rules_host_shim.cpp"),
                    "-o", str(out)], check=True)
    L = C.CDLL(str(out))
    L.t_max_slabs.restype = C.c_int64
    L.t_max_slabs.argtypes = [C.c_int64, C.c_int64, C.c_int]
    L.t_free_pairs.restype = C.c_int64
    L.t_free_pairs.argtypes = [C.c_int64]
    L.t_free_turns.restype = C.c_int64
    L.t_free_turns.argtypes = [C.c_int64]
    L.t_keeps_z.argtypes = [C.c_int64, C.c_int]
    L.t_hist_form.argtypes = [C.c_int64] * 4 + [C.c_int]
    L.t_pairs_per_tile.restype = C.c_int64
    L.t_pairs_per_tile.argtypes = [C.c_int64, C.c_int]
    return L


def test_max_slabs_bounds_every_split(rules):
    """Any split of a bunch's tiles over the pass's workgroups, beside any number
    of other tiles: a run takes up to 32767 pairs, and each tile is split in two
    where the workgroups, one per tile, number at most half the CUs."""
    rng = random.Random(1)
    for _ in range(20_000):
        ppt = 1024 * rng.randint(1, 31)
        ntiles = int(round(2 ** rng.uniform(0, 12)))
        grid = min(ntiles + rng.choice((0, 0, 1, 7, 100, 1000)), CUS)
        slices = 2 if 2 * grid <= CUS else 1
        groups = rng.randint(1, min(ntiles, grid))
        cuts = [0] + sorted(rng.sample(range(1, ntiles), groups - 1)) + [ntiles]
        per = 32767 // ppt
        runs = sum(-(-(b - a) // per) for a, b in zip(cuts, cuts[1:]))
        assert slices * runs <= rules.t_max_slabs(ntiles, ppt, CUS)


def test_max_slabs_of_a_lone_bunch_is_near_what_it_fills(rules):
    assert rules.t_max_slabs(1, 1024, CUS) == 2
    assert rules.t_max_slabs(128, 1024, CUS) == 256
    assert rules.t_max_slabs(489, 1024, CUS) == 263      # 1e6 particles
    assert rules.t_max_slabs(977, 5120, CUS) == 376      # 1e7


@pytest.mark.parametrize("n,tile_pairs,windowed", [
    (1, 0, True), (49_152, 0, True), (49_153, 0, False), (1_000_000, 0, False), (2_499_998, 0, False),
    (2_499_999, 0, True), (10_000_000, 0, True), (50_001, 31, True), (50_001, 32, False), (10_000_000, 32, False)])
def test_histogram_form(rules, n, tile_pairs, windowed):
    """Up to 34560 bins 32-bit counts of all bins; from 40701 on, which they do not
    fit, the window; in between the window where it is the faster one."""
    npairs = (n + 1) // 2
    ppt = rules.t_pairs_per_tile(npairs, tile_pairs)

    def form(nb):
        return rules.t_hist_form(nb, -(-npairs // ppt), npairs, ppt, 163840)
    assert form(34560) == -1
    assert [form(nb) for nb in (34561, 40700)] == ([34560, 40700] if windowed else [-1, -1])
    can = ppt <= 32767
    assert [form(nb) for nb in (40701, 49152, 131073)] == ([40700, 49152, 49152] if can else [0, 0, 0])


@pytest.mark.parametrize("tiles,nb,everywhere,in_lds", [
    (31, 1024, 0, 0), (32, 1024, 1, 1), (100, 109_999, 1, 1), (100, 110_000, 0, 1), (100, 131_072, 0, 1),
    (100, 150_000, 0, 1), (100, 150_001, 1, 1), (31, 150_001, 0, 0)])
def test_where_counters_leave_gaps(rules, tiles, nb, everywhere, in_lds):
    L = rules.t_spreads
    L.argtypes = [C.c_int64, C.c_int64, C.c_int]
    assert (L(tiles, nb, 1), L(tiles, nb, 0)) == (everywhere, in_lds)


def test_cached_particles_fit_the_last_cache_together(rules):
    def cached(*n):
        return bool(rules.t_cached((C.c_int64 * len(n))(*n), len(n)))
    assert cached(10_000_000) and cached(13_000_000) and not cached(15_000_000)
    assert cached(6_000_000, 6_000_000) and not cached(7_000_000, 7_000_000)
    assert not cached(10_000_000, 10_000_000)
    assert cached(*[1_000_000] * 5) and not cached(*[1_000_000] * 10)


@pytest.mark.parametrize("n,with_sums,without", [(9_000_000, 0, 0), (9_500_000, 1, 0), (10_400_000, 1, 0),
                                                 (11_000_000, 1, 1), (29_000_000, 1, 1), (30_000_000, 0, 0)])
def test_where_z_goes_through_the_caches(rules, n, with_sums, without):
    assert (rules.t_keeps_z(8 * n, 1), rules.t_keeps_z(8 * n, 0)) == (with_sums, without)


@pytest.mark.parametrize("pairs", [0, 1, 500, 50_000, 500_000, 5_000_000, 50_000_000, 2 ** 31])
def test_free_turns_of_a_launch_stay_near_40_ms(rules, pairs):
    """0.8 us a turn for a thread's chain, or 6.8e-12 s per pair-turn of a full device."""
    turns = rules.t_free_turns(pairs)
    assert turns >= 1
    assert turns == 1 or turns * max(0.8e-6, 6.8e-12 * pairs) <= 0.045


@pytest.mark.parametrize("pairs", [1, 2_097_152, 2_097_153, 15_000_000, 33_554_432, 33_554_433, 50_000_000, 2 ** 31])
def test_free_items(rules, pairs):
    per = rules.t_free_pairs(pairs)
    items = -(-pairs // (256 * per))
    assert per == (1 if pairs <= 2_097_152 else 4 if pairs <= 33_554_432 else max(16, pairs // (256 << 16) + 1))
    assert items <= 65536
    assert per < 16 or items >= 32 * 256
