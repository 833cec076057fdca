"""pdipc_toi_noalloc of several handles at once: every live handle has its own
place for the minima, also after many others came and went and when there are
more handles than slots of the library's array."""

import numpy as np
import pytest
import torch

import pdipc
import scenes

pytestmark = pytest.mark.gpu


class _Caller:
    """A handle with candidate records, device positions and a stream of its own."""

    def __init__(self, scale, seed):
        sc = scenes.cloth_over_sphere(16, 2, ground=True, seed=5, patch_dim=16, sphere_patch_dim=12, height=0.16)
        self.sim = pdipc.Simulator.from_scene(sc)
        x0 = self.sim.x()
        n = self.sim.sim
        dx = np.zeros_like(x0)
        dx[:n] = np.random.default_rng(seed).normal(0.0, 0.5 * scale, (n, 3)) + [0.0, -2.0 * scale, 0.0]
        self.records = len(self.sim.debug_broad_phase(x0, dx))
        self.want = self.sim.debug_toi(x0, x0 + dx)
        self.x0 = torch.tensor(x0.reshape(-1), dtype=torch.float64, device="cuda")
        self.x1 = torch.tensor((x0 + dx).reshape(-1), dtype=torch.float64, device="cuda")
        self.out = torch.full((64,), -1.0, dtype=torch.float64, device="cuda")
        self.stream = torch.cuda.Stream()
        torch.cuda.synchronize()

    def call(self, i):
        self.sim.toi_noalloc(self.x0.data_ptr(), self.x1.data_ptr(), self.out[i:].data_ptr(), self.stream.cuda_stream)


def _overlap(callers):
    for i in range(64):
        for c in callers:
            c.call(i)
    torch.cuda.synchronize()
    for c in callers:
        assert (c.out.cpu().numpy() == c.want).all()


def test_two_handles_left_of_many():
    print("case: 33rd handle beside the first", flush=True)
    first = _Caller(2e-2, 1)
    tiny = scenes.cloth_over_sphere(4, 1, ground=False, seed=5, patch_dim=4, sphere_patch_dim=4, height=0.4)
    for _ in range(31):
        pdipc.Simulator.from_scene(tiny).close()
    last = _Caller(4e-2, 2)
    assert first.records > 0 and last.records > 0 and first.want != last.want and min(first.want, last.want) < 1.0
    _overlap([first, last])


def test_more_handles_than_slots():
    print("case: 36 handles at once", flush=True)
    callers = [_Caller(1e-2 * (1 + k % 6), k) for k in range(36)]
    assert len({c.want for c in callers}) > 3
    _overlap(callers)
