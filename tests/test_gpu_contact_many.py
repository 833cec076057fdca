"""The record kernels from 2^21 candidate records on, where most records are
settled by an FP32 certificate: the time of impact and the barrier terms against
the oracle, which takes every record through the full FP64 path -- for moves
that keep apart, approach and collide, near the origin and far from it (where
the certificate's rounding allowance settles fewer records)."""

import numpy as np
import pytest
import torch

import oracle
import pdipc
import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pair():
    sc = scenes.cloth_over_sphere(184, 4, ground=False, seed=3, patch_dim=184, sphere_patch_dim=32, height=0.1505)
    return sc, oracle.Oracle(sc), pdipc.Simulator.from_scene(sc)


# FP64 ACCD and barrier sums differ from the oracle's by the compilers' fused
# multiply-adds: a few hundred roundings of relative size 1e-16, amplified by
# distance / coordinate (1e-3 near the origin, 1e-5 at 50 m)
@pytest.mark.parametrize("offset,tol", [(0.0, 1e-10), (50.0, 1e-8)])
@pytest.mark.parametrize("noise", [0.0, 1e-5, 4e-4, 2e-3])
def test_many_records_match_the_oracle(pair, noise, offset, tol):
    sc, ref, sim = pair
    rng = np.random.default_rng(int(noise * 1e6))
    x0 = ref.x() + offset * np.array([1.0, -0.5, 0.25])
    x0[: ref.sim] += rng.normal(0, 0.3 * noise, (ref.sim, 3))
    x1 = x0.copy()
    x1[: ref.sim, 1] -= 0.5 * noise
    x1[: ref.sim] += rng.normal(0, noise, (ref.sim, 3))
    print(f"case: moves of {noise:g}, offset {offset:g}", flush=True)
    recs = sim.debug_broad_phase(x0, x1 - x0)
    assert len(recs) == len(ref.debug_broad_phase(x0, x1 - x0)) and len(recs) >= 1 << 21
    got, want = sim.debug_toi(x0, x1), ref.debug_toi(x0, x1)
    print(f"  {len(recs)} records, time of impact {got!r}", flush=True)
    assert (got < 1.0) == (want < 1.0) and abs(got - want) <= tol * want
    dg, rg, ng = sim.debug_collision(x0)
    do, ro, no = ref.debug_collision(x0)
    assert ng == no
    assert np.abs(dg - do).max() <= tol * np.abs(do).max()
    assert np.abs(rg - ro).max() <= tol * np.abs(ro).max()


def test_no_accd_steps(pair):
    """Without a step of ACCD every record that passes the filter returns 0, and
    none may be settled by its first step."""
    sc, ref, _ = pair
    none = dict(sc, params=dict(sc["params"], ccd_iters=0))
    sim, x0 = pdipc.Simulator.from_scene(none), ref.x()
    x1 = x0.copy()
    x1[: ref.sim] += np.random.default_rng(0).normal(0, 1e-5, (ref.sim, 3))
    print("case: no ACCD steps", flush=True)
    assert len(sim.debug_broad_phase(x0, x1 - x0)) >= 1 << 21
    assert sim.debug_toi(x0, x1) == 0.0


def test_crossing_edges_of_vanishing_normal():
    """Two edges whose centres lie 1e-21 apart, in coordinates so small that the
    square of that line's length is no FP32 number: no bound of their distance
    follows, so the record takes the full path although all around it are
    settled (2^18 records and more on caller's positions) -- the same time of
    impact as one record per thread finds."""
    cl = scenes.cloth_over_sphere(96, 4, ground=False, seed=3, patch_dim=96, sphere_patch_dim=32, height=0.1505)
    sc = dict(cl, cloths=list(cl["cloths"]))
    s = 0.01
    v = s * np.array([[-1.0, 0, 0], [1, 0, 0], [0, -1, 0.25]])
    w = s * np.array([[0.0, 1e-21 / s, -1], [0, 1e-21 / s, 1], [0.25, 1, 0]])
    for q in (v, w):
        sc["cloths"].append(dict(cl["cloths"][0], v=q, f=np.array([[0, 1, 2]], np.int32), patch_dim=2))
    sc["cloths"][0] = dict(cl["cloths"][0], v=np.asarray(cl["cloths"][0]["v"]) + [0.0, 2.0, 0.0])
    sc["statics"] = [dict(t, v=np.asarray(t["v"]) + [0.0, 2.0, 0.0]) for t in cl["statics"]]
    sim = pdipc.Simulator.from_scene(sc)
    x0 = sim.x()
    x1 = x0.copy()
    x1[sim.sim - 3: sim.sim, 1] -= 1e-6  # the second triangle's edge passes through the first's
    recs = sim.debug_broad_phase(x0, x1 - x0)
    print(f"case: vanishing normal, {len(recs)} records", flush=True)
    assert 1 << 18 <= len(recs) < 1 << 21
    want = sim.debug_toi(x0, x1)
    assert want < 1.0
    a, b = (torch.tensor(x.reshape(-1), dtype=torch.float64, device="cuda") for x in (x0, x1))
    out = torch.full((1,), -1.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    sim.toi_noalloc(a.data_ptr(), b.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    assert out.item() == want
