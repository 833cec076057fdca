"""The tile solves (a whole Chebyshev solve in one launch) against the streamed
sweeps: the same bits, over the tilings' edges, both precisions, few and many
sweeps; when a tile gives up waiting; and with several handles stepping at
once from different threads."""

import threading
import time

import numpy as np
import pytest

import pdipc
import scenes

pytestmark = pytest.mark.gpu


def _cloth(n, **kw):
    return scenes.cloth_over_sphere(n, 2, ground=True, seed=2, patch_dim=n, sphere_patch_dim=12, height=0.166, **kw)


# (scene, rows per tile): one tile (4 and 121 rows), tiles of 32 rows with a
# remainder, and every thread mapping above (88, 157, 352 and, FP32 only, 565
# rows per tile); rows of 12 entries per lane, three models
SCENES = [("2", 4), ("11", 121), ("12", 32), ("91", 33), ("150", 88), ("200", 157), ("300", 352), ("380", 565),
          ("tets6", 32), ("tets20", 38), ("layers", 32)]


@pytest.mark.parametrize("which,rows", SCENES)
def test_tile_solves_match_streamed_sweeps(which, rows):
    if which.startswith("tets"):
        sc = scenes.config2(cells=int(which[4:]), cloth_n=20)
    elif which == "layers":
        sc = scenes.config4(n=40, side=80.0 / 1024)
    else:
        sc = _cloth(int(which))
    for iters in (15, 1, 2, 3, 6):
        sc["params"]["cheb_iters"] = iters
        for prec in (pdipc.FP64, pdipc.FP32_SPLIT):
            print(f"case: {which}, {iters} sweeps, precision {prec}", flush=True)
            a = pdipc.Simulator.from_scene(sc, precision=prec)
            b = pdipc.Simulator.from_scene(sc, precision=prec, sell_stage=2)
            info = a.tile_solves()
            assert info["rows_per_tile"] == rows and info["fp32"] == 1 and info["fp64"] == (rows <= 512)
            assert b.tile_solves()["built"] == 0
            rng = np.random.default_rng(iters)
            x = a.x()
            x[: a.sim] += rng.normal(0, 1e-3, (a.sim, 3))
            diag, rhs = rng.uniform(2e5, 4e5, a.sim), rng.normal(0, 1e3, (a.sim, 3))
            for rep in range(3):  # a second launch finds the first one's publications
                assert np.array_equal(a.debug_solve(diag, rhs + rep, x), b.debug_solve(diag, rhs + rep, x)), rep
        if iters == 15:
            for prec in (pdipc.FP64, pdipc.FP32_SPLIT):
                for graphs in (0, 1):
                    sims = [pdipc.Simulator.from_scene(sc, precision=prec, use_graphs=graphs, sell_stage=st)
                            for st in (1, 2)]
                    for s in sims:
                        s.step(3)
                    assert np.array_equal(sims[0].x(), sims[1].x()) and np.array_equal(sims[0].v(), sims[1].v())
                    assert sims[0].tile_solves()["aborts"] == 0


@pytest.mark.parametrize("prec", [pdipc.FP64, pdipc.FP32_SPLIT])
def test_given_up_solve_repeats_with_streamed_sweeps(prec):
    sc = _cloth(40)
    print(f"case: tile abort, precision {prec}", flush=True)
    a = pdipc.Simulator.from_scene(sc, precision=prec, use_graphs=1)
    b = pdipc.Simulator.from_scene(sc, precision=prec, use_graphs=1)
    for k in range(6):
        if k in (1, 4):
            a.tile_solves(request_abort=True)
        a.step(1)
        b.step(1)
        assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v()), k
        assert a.counters() == b.counters()
    assert a.tile_solves()["aborts"] == 2 and b.tile_solves()["aborts"] == 0
    # twice is enough: the handle keeps to the streamed sweeps
    assert a.tile_solves()["fp64"] == 0 and b.tile_solves()["fp64"] == 1
    if prec == pdipc.FP64:
        c = pdipc.Simulator.from_scene(sc, precision=prec)
        d = pdipc.Simulator.from_scene(sc, precision=prec)
        g = np.random.default_rng(0).normal(size=(c.sim, 3))
        c.tile_solves(request_abort=True)
        c.rollout(3, 0)
        d.rollout(3, 0)
        assert np.array_equal(c.x(), d.x())
        for u, w in zip(c.backward(dx=g), d.backward(dx=g)):
            assert np.allclose(u, w, rtol=1e-9, atol=1e-12 * max(np.abs(w).max(initial=0.0), 1e-300))
        assert c.tile_solves()["aborts"] == 1
        # a reverse pass that gives up: the backward is repeated with the streamed sweeps
        e = pdipc.Simulator.from_scene(sc, precision=prec)
        e.rollout(3, 2)
        e.tile_solves(request_abort=2)
        for u, w in zip(e.backward(dx=g), d.backward(dx=g)):
            assert np.allclose(u, w, rtol=1e-9, atol=1e-12 * max(np.abs(w).max(initial=0.0), 1e-300))
        assert e.tile_solves()["aborts"] == 1


@pytest.mark.parametrize("n", [2, 11, 40, 150])
@pytest.mark.parametrize("every", [0, 2])
def test_taped_passes_match_streamed_sweeps(n, every):
    """The recorded rhs and iterates: the same forward bits, and gradients as
    near as the accumulation order of their atomics allows."""
    print(f"case: rollout of cloth {n}, checkpoints every {every}", flush=True)
    sims = [pdipc.Simulator.from_scene(_cloth(n), sell_stage=st) for st in (1, 2)]
    g = np.random.default_rng(1).normal(size=(sims[0].sim, 3))
    for s in sims:
        s.rollout(3, every)
    assert np.array_equal(sims[0].x(), sims[1].x()) and np.array_equal(sims[0].v(), sims[1].v())
    for u, w in zip(sims[0].backward(dx=g, dv=g), sims[1].backward(dx=g, dv=g)):
        assert np.allclose(u, w, rtol=1e-9, atol=1e-12 * max(np.abs(w).max(initial=0.0), 1e-300))


def test_handles_stepping_from_several_threads():
    """One handle at a time has the device's turn for tile solves; the others
    stream meanwhile, and every one gets the bits it gets alone."""
    scs = [_cloth(48), _cloth(33, kappa=2e3), scenes.config2(cells=5, cloth_n=12)]
    print("case: three handles in three threads", flush=True)

    def go(sc, out, i):
        s = pdipc.Simulator.from_scene(sc, use_graphs=i % 2)
        for _ in range(4):
            s.step(2)
        out[i] = (s.x(), s.v(), s.tile_solves()["aborts"])

    alone, together = [None] * 3, [None] * 3
    for i, sc in enumerate(scs):
        go(sc, alone, i)
    ts = [threading.Thread(target=go, args=(sc, together, i)) for i, sc in enumerate(scs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for p, q in zip(alone, together):
        assert np.array_equal(p[0], q[0]) and np.array_equal(p[1], q[1])
        assert p[2] == 0 and q[2] == 0


# Few sweeps leave few publications between two of the same slot: whole steps,
# whose passes follow each other in one launch (cloths) or in alternating sets.
# 32 and 88 rows per tile, the latter with four threads per row; several models.
@pytest.mark.parametrize("iters", [1, 2, 3])
@pytest.mark.parametrize("which", ["20", "150", "layers"])
def test_fp32_steps_of_few_sweeps_match_streamed_sweeps(which, iters):
    sc = scenes.config4(n=40, side=80.0 / 1024) if which == "layers" else _cloth(int(which))
    sc["params"]["cheb_iters"] = iters
    print(f"case: {which}, FP32 steps of {iters} sweeps", flush=True)
    a, b = (pdipc.Simulator.from_scene(sc, precision=pdipc.FP32_SPLIT, sell_stage=st) for st in (1, 2))
    assert a.tile_solves()["fp32"] == 1 and a.tile_solves()["tiles"] > 1 and b.tile_solves()["built"] == 0
    for k in range(4):
        a.step(1)
        b.step(1)
        assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v()), k
    assert a.tile_solves()["aborts"] == 0


# the same in FP64: cloths in one launch per outer iteration and, over 128 rows
# per tile, in separate solves that read their neighbours' rows of X and write
# their own; tet scenes have only those
@pytest.mark.parametrize("iters", [1, 2, 3])
@pytest.mark.parametrize("which", ["20", "200", "tets6", "tets20"])
def test_fp64_steps_of_few_sweeps_match_streamed_sweeps(which, iters):
    sc = scenes.config2(cells=int(which[4:]), cloth_n=20) if which.startswith("tets") else _cloth(int(which))
    sc["params"]["cheb_iters"] = iters
    print(f"case: {which}, FP64 steps of {iters} sweeps", flush=True)
    a, b = (pdipc.Simulator.from_scene(sc, sell_stage=st) for st in (1, 2))
    assert a.tile_solves()["fp64"] == 1 and a.tile_solves()["tiles"] > 1 and b.tile_solves()["built"] == 0
    for k in range(4):
        a.step(1)
        b.step(1)
        assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v()), k
    for s in (a, b):
        s.rollout(2, 0)
    assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v())
    assert a.tile_solves()["aborts"] == 0
    if which.startswith("tets"):
        return
    g = np.random.default_rng(iters).normal(size=(a.sim, 3))  # the bound of the 15-sweep rollouts above
    for u, w in zip(a.backward(dx=g, dv=g), b.backward(dx=g, dv=g)):
        assert np.allclose(u, w, rtol=1e-9, atol=1e-12 * max(np.abs(w).max(initial=0.0), 1e-300))


@pytest.mark.parametrize("which", ["tets6", "tets20", "layers"])
def test_fp32_tet_steps_of_few_sweeps_match_streamed_sweeps(which):
    sc = scenes.config4(n=40, side=80.0 / 1024) if which == "layers" else scenes.config2(cells=int(which[4:]), cloth_n=20)
    for iters in (1, 2, 3):
        for timed in (False, True):  # with kernel timing the passes run as separate launches
            sc["params"]["cheb_iters"] = iters
            print(f"case: {which}, FP32 steps of {iters} sweeps, timed {timed}", flush=True)
            a, b = (pdipc.Simulator.from_scene(sc, precision=pdipc.FP32_SPLIT, sell_stage=st) for st in (1, 2))
            a.kernel_timing(timed)
            a.step(3)
            b.step(3)
            assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v())


def test_handle_that_gave_up_twice_tries_again():
    """It rests from tile solves for two seconds, with the same bits meanwhile."""
    print("case: two tile aborts, then a rest", flush=True)
    a, b = (pdipc.Simulator.from_scene(_cloth(40), use_graphs=1) for _ in range(2))
    for k in range(2):
        a.tile_solves(request_abort=True)
        a.step(2)
        b.step(2)
    assert a.tile_solves()["aborts"] == 2 and a.tile_solves()["fp64"] == 0
    a.step(1)
    b.step(1)
    time.sleep(2.1)
    assert a.tile_solves()["fp64"] == 1
    a.step(2)
    b.step(2)
    assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v())
    assert a.tile_solves()["aborts"] == 2
    a.tile_solves(request_abort=True)  # the tiles ran: the next request is seen, and the rest is longer
    a.step(1)
    b.step(1)
    time.sleep(2.1)
    assert a.tile_solves()["aborts"] == 3 and a.tile_solves()["fp64"] == 0
    assert np.array_equal(a.x(), b.x()) and np.array_equal(a.v(), b.v())


# (scene, precision): the loop in one launch in both precisions; separate solves
# of one and two rows per thread and of tets.  One tile gives up when the others
# are under way: some have written X, others have not.
@pytest.mark.parametrize("which,prec", [("40", pdipc.FP64), ("40", pdipc.FP32_SPLIT), ("150", pdipc.FP32_SPLIT),
                                        ("200", pdipc.FP64), ("300", pdipc.FP32_SPLIT), ("380", pdipc.FP32_SPLIT),
                                        ("tets6", pdipc.FP64), ("tets6", pdipc.FP32_SPLIT)])
def test_solve_given_up_under_way_repeats_with_streamed_sweeps(which, prec):
    sc = scenes.config2(cells=6, cloth_n=20) if which == "tets6" else _cloth(int(which))
    ref = pdipc.Simulator.from_scene(sc, precision=prec, sell_stage=2)
    xs = []
    for _ in range(3):
        ref.step(1)
        xs.append((ref.x(), ref.v(), ref.counters()))
    for j in (0, 1, 5, 12):
        print(f"case: {which}, precision {prec}, first tile gives up at publication {j}", flush=True)
        a = pdipc.Simulator.from_scene(sc, precision=prec, use_graphs=j % 2)
        assert a.tile_solves()["tiles"] > 1
        for k in range(3):
            if k == 1:
                a.tile_solves(request_abort=65536 + j)
            a.step(1)
            assert np.array_equal(a.x(), xs[k][0]) and np.array_equal(a.v(), xs[k][1]), k
            assert a.counters()["outer_iters"] == xs[k][2]["outer_iters"]
        assert a.tile_solves()["aborts"] == 1


def test_passes_given_up_under_way_repeat_with_streamed_sweeps():
    """Recorded passes (their iterates are recorded again) and reverse sweeps."""
    sc = _cloth(40)
    d = pdipc.Simulator.from_scene(sc)
    g = np.random.default_rng(0).normal(size=(d.sim, 3))
    d.rollout(3, 2)
    want = d.backward(dx=g)
    for every in (0, 2):
        for j in (0, 7, 13):
            for back in (0, 1):
                print(f"case: checkpoints every {every}, {'backward' if back else 'rollout'} publication {j}", flush=True)
                c = pdipc.Simulator.from_scene(sc)
                if not back:
                    c.tile_solves(request_abort=65536 + j)
                c.rollout(3, every)
                assert np.array_equal(c.x(), d.x()) and c.tile_solves()["aborts"] == 1 - back
                if back:
                    c.tile_solves(request_abort=131072 + j)
                for u, w in zip(c.backward(dx=g), want):
                    assert np.allclose(u, w, rtol=1e-9, atol=1e-12 * max(np.abs(w).max(initial=0.0), 1e-300))
                assert c.tile_solves()["aborts"] == 1
