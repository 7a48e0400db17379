"""What a run by the launch schemes brings to the device and back: strategies written 64 layers at a time by the kernel that walks back,
tables below and above the size that a kernel brings over, against the C oracle."""
import numpy as np
import pytest

from galvatron_dp import _lib
from oracle import dp_oracle as O


def _instance(L, S, V, seed):
    rng = np.random.Generator(np.random.PCG64([L, S, V, seed]))
    per = V // L
    mem = rng.integers(max(1, per // 4), 2 * per + 1, size=(L, S)).astype(np.int32)
    # keys: a budget that binds, one that hardly does, none left for any path, below the table
    return mem, rng.lognormal(2.5, 0.5, size=(L, S)), rng.uniform(0, 5, size=(L, S, S)), [V // 10, 0, V - 1, V + 3], [0.5, 0.25, 0.0, 1.0]


def _same(prob, x, V, tag):
    keys = range(len(x[3]))
    total, res, left = O.solve(x[0], x[1], x[2], V, dict(zip(keys, x[3])), dict(zip(keys, x[4])))[:3]
    for k in keys:
        assert np.float64(prob.total[k]).tobytes() == np.float64(total[k]).tobytes(), f"{tag} key {k}"
        assert int(prob.remaining[k]) == left[k], f"{tag} key {k}"
        if left[k] >= 0:
            assert [int(v) for v in prob.res[k]] == [int(v) for v in res[k]], f"{tag} key {k}"


# Layers around a multiple of 64 and a single one; strategies of one wave's lanes and more; tables of 0.36, 0.41 and 1.2 MB
@pytest.mark.gpu
@pytest.mark.parametrize("L,S,V", [(1, 5, 300), (2, 6, 640), (63, 6, 2500), (64, 6, 2500), (65, 6, 2500), (128, 7, 3000), (129, 7, 3000),
                                   (66, 70, 2000), (28, 40, 1500), (32, 40, 1500), (40, 60, 1500)])
@pytest.mark.parametrize("way", ["call", "layers", "plan", "batch"])
def test_against_the_oracle(L, S, V, way, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    xs = [_instance(L, S, V, k) for k in range(3 if way == "batch" else 1)]
    probs = [_lib.Problem(x[0], x[1], x[2], V, x[3], x[4], **({"launch": "per_layer"} if way == "layers" else {})) for x in xs]
    if way == "plan":
        with _lib.Plan(probs) as plan:
            for again in range(3):
                plan.run()
                plan.fetch()
                _same(probs[0], xs[0], V, f"{L} {S} {V} run {again}")
        return
    _lib.solve_batch(probs)
    for x, prob in zip(xs, probs):
        _same(prob, x, V, f"{L} {S} {V} {way}")
