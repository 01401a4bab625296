"""The automatic launch shape of a batch (tile lengths by cost, a workgroup per
tile) can be asked for again, the autotuner weighs it and reports it in the
setters' own values, and what a batch holds no problems for stays automatic."""
import numpy as np
import pytest

from sonicsolver_amd import SonicError, workloads as wl
from sonicsolver_amd.batch import Batch, item_nodes, make_item
from sonicsolver_amd.serve import Server

pytestmark = pytest.mark.gpu

KINDS = {"1d": [(300,), (1000,), (64,)], "2d": [(40, 30), (66, 35)],
         "mixed": [(300,), (40, 30), (66, 35), (90,)]}


def _problems(kind):
    return [(dict(n=n, d=(0.01, 0.013)[:len(n)], scheme=("weno5", "teno5")[k % 2],
                  flux=("rusanov", "hllc")[k // 2 % 2], cfl=0.4), wl.smooth_field(n, seed=k + 1))
            for k, n in enumerate(KINDS[kind])]


def _batch(probs):
    b = Batch(sum(item_nodes(make_item(**kw)) for kw, _ in probs), len(probs))
    return b, [b.add(make_item(**kw), q) for kw, q in probs]


def _apply(to, t):
    to.set_tiles(t["xlen"], t["ylen"])
    to.set_occupancy(t["blocks_per_cu"])
    to.set_schedule(bool(t["fused"]))


def test_setters_take_the_automatic_values():
    probs = _problems("mixed")
    outs = []
    for change in (False, True):
        b, slots = _batch(probs)
        with b:
            if change:
                _apply(b, dict(xlen=127, ylen=8, blocks_per_cu=2, fused=0))
                b.step(1)
                _apply(b, dict(xlen=0, ylen=0, blocks_per_cu=-1, fused=1))
            else:
                b.step(1)
            b.step(3)
            outs.append([b.download(s) for s in slots])
            for call in (lambda: b.set_tiles(1, 0), lambda: b.set_tiles(0, 3),
                         lambda: b.set_tiles(0, -1), lambda: b.set_tiles(63, 4097),
                         lambda: b.set_occupancy(-2), lambda: b.set_occupancy(65)):
                with pytest.raises(SonicError):
                    call()
    for a, c in zip(*outs):
        assert np.array_equal(a, c)


@pytest.mark.parametrize("kind,candidates", [("1d", 30), ("2d", 30), ("mixed", 90)])
@pytest.mark.parametrize("steps", [1, 9])
def test_autotune_keeps_what_it_cannot_weigh(kind, candidates, steps):
    probs = _problems(kind)
    b, slots = _batch(probs)
    with b:
        b.step(2)
        before = [b.download(s) for s in slots]
        t = b.autotune(steps)
        print(f"autotune {kind}: {t}", flush=True)
        assert t["candidates"] == candidates and t["ms_per_step"] > 0
        if kind == "1d":
            assert t["ylen"] == 0
        if kind == "2d":
            assert t["xlen"] == 0
        for s, q in zip(slots, before):
            assert np.array_equal(b.download(s), q)
        b.step(2)
        out = [b.download(s) for s in slots]
    other, slots = _batch(probs)
    with other:
        _apply(other, t)   # the values it reports are the setters' own
        other.step(4)
        for s, q in zip(slots, out):
            assert np.array_equal(other.download(s), q)


def test_server_takes_the_automatic_shape():
    kw, q = _problems("2d")[0]
    outs = []
    for shape in (None, (0, 0, -1, 1), (255, 16, 4, 0)):
        with Server(1 << 26, max_items=4) as s:
            if shape:
                s.set_shape(*shape)
            t = s.submit(make_item(**kw), q, 6)
            assert s.wait(t) == 1
            outs.append(s.result(t)[0])
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
