"""The tile solves' tables on the host (no device): every row in one tile,
tiles compact enough for their LDS, halos that are exactly the columns other
tiles own and a symmetric neighbour relation, and every thread's entries
pointing at the LDS row of their M^2 column (checked against the SELL layout
the streamed sweeps use)."""

import numpy as np
import pytest

import pdipc
import scenes


def _scene(which):
    if which == "tets":
        return scenes.config2(cells=6, cloth_n=9)
    if which == "layers":
        sc = scenes.config4(n=20, side=40.0 / 1024)
        sc["statics"] = sc["statics"][1:]
        return sc
    n = int(which)
    return scenes.cloth_over_sphere(n, 2, ground=True, seed=1, patch_dim=n, sphere_patch_dim=16)


# rows 4 to 9,216 over 1 to 256 tiles: one tile, tiles of 32 rows, and 2, 4
# and 8 lanes per thread, two rows per thread; cloths of varying and of the common width 8, tets
# (12 entries per lane), several models
@pytest.mark.parametrize("which,max_tiles", [("2", 256), ("11", 256), ("12", 256), ("96", 256), ("96", 100),
                                             ("96", 40), ("96", 20), ("96", 10), ("tets", 256), ("tets", 3), ("layers", 256)])
def test_tiles_cover_the_rows_and_entries(which, max_tiles):
    sim = pdipc.Simulator.from_scene(_scene(which), init=False)
    sim.host_setup()
    n = sim.sim
    T = sim.tile_layout(max_tiles)
    assert T is not None
    rows, off, halo = T["rows"], T["halo_off"], T["halo"]
    nt, R = rows.shape
    assert nt <= max_tiles and (R >= 32 or nt == 1)
    assert nt == -(-n // R) and (nt == 1) == (n <= 128)
    flat = rows.reshape(-1)
    assert np.array_equal(np.sort(flat[flat >= 0]), np.arange(n))
    owner, place = np.zeros(n, int), np.zeros(n, int)
    for t in range(nt):
        r = rows[t][rows[t] >= 0]
        owner[r], place[r] = t, np.arange(len(r))
        assert np.array_equal(rows[t][: len(r)], r) and (np.diff(r) > 0).all()
    S = sim.sell_layout(8)
    col, so, sw, perm = S["col"], S["slice_off"], S["slice_w"], S["perm"]
    slot_of = np.arange(len(sw) * 8)
    if perm is not None:
        slot_of[perm] = np.arange(len(perm))
    W, tpr, BT = T["width"], T["tpr"], T["threads"]
    assert sw.max() <= W and R <= BT // tpr
    rw, subs = 64 // tpr, 8 // tpr
    E = subs * W
    loc = T["loc"].reshape(nt, E // 8, BT, 8)
    neighbours = []
    for t in range(nt):
        h = halo[off[t]: off[t + 1]]
        assert (np.diff(h) > 0).all() and (owner[h] != t).all() and R + len(h) <= T["cap"]
        neighbours.append(set(owner[h].tolist()))
        at = np.full(n, -1)
        at[h] = R + np.arange(len(h))
        r = rows[t][rows[t] >= 0]
        at[r] = np.arange(len(r))
        read = set()
        for rl, row in enumerate(r):
            slot = slot_of[row]
            s = slot // 8
            for part in range(tpr):
                th = (rl // rw) * 64 + part * rw + rl % rw
                for g in range(subs):
                    lane = (slot % 8) * 8 + part + g * tpr
                    for c in range(W):
                        e = g * W + c
                        got = loc[t, e // 8, th, e % 8]
                        if c >= sw[s]:
                            assert got == rl
                            continue
                        k = so[s] + (lane * 8 + c if S["uniform_w"] == 8 else c * 64 + lane)
                        assert got == at[col[k]]
                        read.add(int(col[k]))
        # the halo is what the entries read (an added row only where the pattern is not symmetric)
        assert set(r.tolist()) | set(h.tolist()) >= read
        assert len(set(h.tolist()) - read) <= 1
    for t in range(nt):
        for o in neighbours[t]:
            assert t in neighbours[o]


def test_scenes_that_do_not_tile():
    sim = pdipc.Simulator.from_scene(_scene("96"), init=False)
    sim.host_setup()
    assert sim.tile_layout(8) is None  # 1,152 rows per tile: over a workgroup's registers
