"""The patches' radix sort at the edges of its one-workgroup form (rounds of
1,024 items, at most 16): the sorted keys are the sort of all patches' keys,
each patch once, equal codes in patch order; and the tree's candidates are the
oracle's."""

import threading

import numpy as np
import pytest

import oracle
import pdipc
import scenes

pytestmark = pytest.mark.gpu


# cloths of n^2 points and their sphere: below and above one, two and 16 rounds
@pytest.mark.parametrize("n", [3, 8, 31, 32, 45, 127, 128, 140])
def test_sorted_keys(n):
    sc = scenes.cloth_over_sphere(n, 1, ground=False, seed=5, patch_dim=n, sphere_patch_dim=8, height=0.166)
    print(f"case: cloth {n}", flush=True)
    sim, ref = pdipc.Simulator.from_scene(sc), oracle.Oracle(sc)
    x = sim.x()
    # flat in y, so that many codes are equal
    x[: sim.sim, 1] = x[: sim.sim, 1].mean()
    move = np.zeros_like(x)
    move[: sim.sim] = np.random.default_rng(n).normal(0, 2e-3, (sim.sim, 3))
    for dx in (np.zeros_like(x), move):
        got, want = sim.debug_broad_phase(x, dx), ref.debug_broad_phase(x, dx)
        assert np.array_equal(np.unique(got, axis=0), np.unique(want, axis=0)) and len(got) == len(want)
        keys = np.asarray(sim.debug_lbvh()[0])
        print(f"  {len(keys)} patches, {len(got)} records", flush=True)
        assert np.array_equal(keys, np.sort(keys))
        assert np.array_equal(np.sort(keys & np.uint64(0xFFFFFFFF)), np.arange(len(keys), dtype=np.uint64))


def test_sorts_of_two_handles_in_two_threads():
    """About 11,000 and 16,300 patches: both need more LDS than the default limit, which
    is the process's and must never be lowered between another thread's raising
    it and its launch."""
    print("case: two handles sorting in two threads", flush=True)
    sims = [pdipc.Simulator.from_scene(scenes.cloth_over_sphere(n, 1, ground=False, seed=5, patch_dim=n,
                                                                sphere_patch_dim=8, height=0.166)) for n in (105, 127)]
    xs = [s.x() for s in sims]
    want = [s.debug_broad_phase(x, np.zeros_like(x)) for s, x in zip(sims, xs)]
    bad = []

    def go(i):
        try:
            for _ in range(30):
                if not np.array_equal(sims[i].debug_broad_phase(xs[i], np.zeros_like(xs[i])), want[i]):
                    bad.append(i)
        except Exception as e:  # a refused launch
            bad.append(e)

    ts = [threading.Thread(target=go, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
