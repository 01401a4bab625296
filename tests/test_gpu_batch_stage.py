"""The batch's stage launches against the grid path, at the edges of their
tiles: strips of 63 or 64 columns, one row to several tiles of rows, the
smallest problems, every variant, corners included.

Both paths evaluate the same faces, updates and ends, with the same
operations per node, so a few steps may differ by rounding at most: 1e-13 of
each variable's largest value, 3 steps times 3 stages times a handful of
units in the last place."""
import numpy as np
import pytest
import torch

from sonicsolver_amd import workloads as wl
from sonicsolver_amd._native import Grid, make_desc
from sonicsolver_amd.batch import Batch, item_nodes, make_item

pytestmark = pytest.mark.gpu

SIZES = [(4, 1), (5, 1), (65, 1), (66, 1), (128, 1), (129, 1), (1000, 1),
         (4, 4), (5, 7), (64, 9), (65, 34), (66, 35), (67, 36), (130, 67), (131, 5), (9, 130)]


def _grid_run(kw, q, steps):
    nx, ny = (list(kw["n"]) + [1])[:2]
    desc = dict(n=(nx, ny, 1), active=(1, int(ny > 1), 0), bc=("transmissive",) * 3,
                d=(kw["d"][0], kw["d"][1] if ny > 1 else 1.0, 1.0), scheme=kw["scheme"],
                flux=kw["flux"], time="ssprk3")
    with Grid(make_desc(**desc)) as g:
        g.upload(q)
        g.run(steps, kw["cfl"])
        return g.download().reshape(5, -1), g.clock()


@pytest.mark.parametrize("shape", [None, (127, 4, 0), (255, 32, 2)])
@pytest.mark.parametrize("fused", [True, False])
def test_batch_equals_grid(shape, fused):
    probs = []
    for k, n in enumerate(SIZES):
        kw = dict(n=n, d=(0.01, 0.013), scheme=("weno5", "teno5")[k % 2],
                  flux=("rusanov", "hllc")[k // 2 % 2], cfl=0.4)
        probs.append((kw, wl.smooth_field(n, seed=k + 1)))
    cap = sum(item_nodes(make_item(**kw)) for kw, _ in probs)
    with Batch(cap, len(probs)) as b:
        b.set_schedule(fused)
        if shape:
            b.set_tiles(*shape[:2])
            b.set_occupancy(shape[2])
        slots = [b.add(make_item(**kw), q) for kw, q in probs]
        b.step(1)
        b.step(2, graph=False)
        outs = [(b.download(s).reshape(5, -1), b.clock(s)) for s in slots]
    for (kw, q), (out, clock) in zip(probs, outs):
        print(kw, flush=True)
        ref, rclock = _grid_run(kw, q, 3)
        tol = 1e-13 * np.abs(ref).max(axis=1, keepdims=True)
        assert (np.abs(out - ref) <= tol).all(), kw
        assert clock[1] == 3 and abs(clock[0] - rclock[0]) <= 1e-13 * rclock[0], kw


def test_first_state_of_a_fresh_arena_or_grid():
    """A state that arrives right after its memory was allocated, while the
    clearing of some gigabytes is still under way, is not cleared with it."""
    kw = dict(n=(64, 64), d=(0.01, 0.01), scheme="weno5", flux="hllc", cfl=0.4)
    q = wl.smooth_field((64, 64), seed=2)
    ref, _ = _grid_run(kw, q, 2)
    for _ in range(2):
        with Batch(60_000_000, 4) as b:
            slot = b.add(make_item(**kw), q)
            b.step(2, graph=False)
            assert np.abs(b.download(slot).reshape(5, -1) - ref).max() <= 1e-13 * np.abs(ref).max()
    n = (512, 512, 96)
    desc = make_desc(n=n, bc=("periodic",) * 3, d=(0.01,) * 3)
    field = torch.rand(5, n[0] * n[1] * n[2], dtype=torch.float64, device="cuda") + 1.0
    back = torch.empty_like(field)
    torch.cuda.synchronize()
    for _ in range(2):
        with Grid(desc) as g:
            g.upload_device(field.data_ptr())
            g.download_device(back.data_ptr())
            g.synchronize()
        assert torch.equal(back, field)
