"""The DP over labels with a workgroup for every key of an instance: at the numbers of labels, strategies, layers and keys around which
its kernel branches, against the C oracle, which sees the whole instance."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from galvatron_dp import _lib
from oracle import dp_oracle as O


def _instance(L, S, V, kind, n_keys):
    """Two thirds of the strategies are dominated by another ('each', 'alike': random costs; 'trade': what is left trades memory for
    time and is the same in all layers, so that labels are many; 'ties': small whole numbers; 'runs': one strategy is the best by
    far in most layers)."""
    rng = np.random.Generator(np.random.PCG64([L, S, V, n_keys]))
    per, n = max(2, V // L), 1 if kind in ("trade", "alike") else L
    mem = rng.integers(max(1, per // 4), 3 * per, size=(n, S)).astype(np.int32)
    intra, inter = rng.lognormal(2.5, 0.5, size=(n, S)), rng.uniform(0, 5, size=(n, S, S))
    if kind == "trade":
        intra, inter = 40.0 * per / mem * rng.uniform(0.98, 1.02, size=mem.shape), inter * 0.05
        worse = rng.permutation(S)[:2 * S // 3]
        intra[:, worse] = intra.max() + 1.0 + worse
    if kind == "ties":
        mem, intra, inter = (mem // max(1, per // 4) + 1).astype(np.int32), rng.integers(1, 5, size=(n, S)).astype(float), rng.integers(0, 3, size=(n, S, S)).astype(float)
    if kind == "runs":
        for l in range(L):
            if l % 7 != 3:
                intra[l, rng.integers(S)] = 1e-3
                mem[l, np.argmin(intra[l])] = 1
    if n == 1:
        mem, intra, inter = np.repeat(mem, L, 0), np.repeat(intra, L, 0), np.repeat(inter, L, 0)
    om = [int(V * f) for f in (0.1, 0.3, 0.0, 0.45, 0.2, 0.999, 0.25, 2.0)[:n_keys]]
    return mem, intra, inter, om, [k / 3 for k in range(n_keys)]


def _same(prob, x, V, tag):
    keys = range(len(x[3]))
    total, res, left = O.solve(x[0], x[1], x[2], V, dict(zip(keys, x[3])), dict(zip(keys, x[4])))[:3]
    for k in keys:
        assert np.float64(prob.total[k]).tobytes() == np.float64(total[k]).tobytes(), f"{tag} key {k}: {prob.total[k]} {total[k]}"
        assert int(prob.remaining[k]) == left[k], f"{tag} key {k}"
        if left[k] >= 0:
            assert [int(v) for v in prob.res[k]] == [int(v) for v in res[k]], f"{tag} key {k}"


def _executed(probs, solve=_lib.solve_batch):
    """The share of the relaxations that are looked at: next to none where labels solve them."""
    _lib.batch_stats_begin()
    solve(probs)
    s = _lib.batch_stats_end()
    return s.executed / s.relaxations


# Layers: 2, around 64 (a word of marks), 128, and one more, which has a workgroup per instance; strategies: 2, around 64 (the
# words of a layer's marks), 128; labels: one (runs of layers with one strategy), up to 16, 32 and 64 beside each other, more, in buckets
# (trade: 485 with L = 16, 1200 with L = 24 are given up); layers whose strategies and transitions do not fit into LDS at a time (ties, L = 50:
# 472 and 4406).  How many there are, and that the kernel solves them, is checked on the CPU as well (test_key_labels_on_cpu.py).
@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V", [("each", 2, 2, 60), ("each", 9, 12, 3000), ("each", 20, 63, 4000), ("each", 20, 64, 4000), ("each", 20, 65, 4000),
                                        ("each", 6, 128, 2000), ("each", 63, 7, 6000), ("each", 64, 7, 6000), ("each", 65, 7, 6000), ("runs", 127, 6, 4000),
                                        ("runs", 128, 6, 4000), ("runs", 129, 6, 4000), ("runs", 40, 20, 5000), ("alike", 30, 24, 5000),
                                        ("trade", 8, 9, 2000), ("trade", 12, 24, 5000), ("trade", 16, 33, 9000), ("trade", 24, 48, 12000), ("ties", 12, 24, 300),
                                        ("ties", 30, 40, 900), ("ties", 70, 9, 1000), ("ties", 50, 40, 1500)])
@pytest.mark.parametrize("n_keys", [1, 3, 4, 8])
def test_calls_against_the_oracle(kind, L, S, V, n_keys, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    x = _instance(L, S, V, kind, n_keys)
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4])
    _lib.batch_stats_begin()
    _lib.solve_batch([prob])
    s = _lib.batch_stats_end()
    _same(prob, x, V, f"{kind} {L} {S} {V}")
    if V > 60:                                              # (of a small instance labels are no small part)
        given_up = (kind, L) == ("trade", 24) and n_keys != 3
        assert (s.executed < 0.01 * s.relaxations) == (not given_up)


@pytest.mark.gpu
@pytest.mark.parametrize("many", [2, 60, 130])
def test_batches_of_different_shapes(many, monkeypatch):
    """More keys than compute units, more layers than the shortest of them has, strategies on both sides of 64."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    V, xs = 1500, [_instance(3 + i % 9, 5 + 11 * (i % 7), 1500 + i, ("each", "ties")[i % 2], 1 + i % 6) for i in range(many)]
    probs = [_lib.Problem(x[0], x[1], x[2], V, x[3], x[4]) for x in xs]
    assert _executed(probs) < 0.01
    for i, (x, prob) in enumerate(zip(xs, probs)):
        _same(prob, x, V, f"instance {i}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V,n_keys", [("each", 30, 24, 5000, 4), ("trade", 20, 30, 6000, 2), ("runs", 60, 9, 6000, 3), ("ties", 20, 30, 600, 4)])
def test_static_calls_and_plans(kind, L, S, V, n_keys, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    x = _instance(L, S, V, kind, n_keys)
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4])
    assert _executed(prob, _lib.solve_static) < 0.01
    _same(prob, x, V, f"static {kind}")
    prob.total[:], prob.remaining[:], prob.res[:] = 0, 0, 0
    with _lib.Plan([prob]) as plan:
        for _ in range(2):
            assert plan.run().relax_launches == 0
            plan.fetch()
            _same(prob, x, V, f"plan {kind}")


def test_the_kernel_needs_nothing_obtained_for_a_launch(tmp_path):
    """It is one of gdp_solve_static's: no scratch memory, and a launcher that calls no allocator."""
    from galvatron_dp import _build
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    flags = [f for f in _build.HIPCC_FLAGS if f != "-shared"]
    source, obj = os.path.join(_build.CSRC, "gdp_key_labels.hip"), str(tmp_path / "o.o")
    log = subprocess.run([hipcc] + flags + ["-c", "-Rpass-analysis=kernel-resource-usage", source, "-o", obj], check=True, capture_output=True,
                         text=True).stderr
    found = re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", log, re.S)
    assert [int(size) for name, size in found if "key_labels" in name] == [0]
    undefined = subprocess.run(["nm", "-u", "-C", obj], stdout=subprocess.PIPE, text=True, check=True).stdout
    for name in (ln.split(None, 1)[1].strip() for ln in undefined.splitlines() if ln.strip().startswith("U ")):
        assert not name.startswith(("hipMalloc", "hipHost", "hipMem", "hipStream", "hipEvent", "hipFree", "operator", "malloc", "calloc", "std::__throw")), name


# On either side of each term of the rule for a call: 3e7 relaxations, undominated strategies over layers and keys, their share, the
# layers a workgroup has words for; initial costs that take longer to look through than the launch schemes, and that do not
@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V,n_keys,zeros,labels", [("alike", 24, 22, 16384, 4, False, True), ("alike", 24, 22, 16384, 8, False, False),
                                                            ("alike", 24, 22, 2500, 4, False, False), ("trade", 20, 24, 16000, 4, False, False),
                                                            ("runs", 128, 8, 9000, 1, False, True), ("runs", 129, 8, 9000, 1, False, False),
                                                            ("alike", 24, 22, 16384, 4, True, True), ("each", 8, 24, 60000, 2, True, False),
                                                            ("each", 8, 24, 60000, 2, False, True)])
def test_calls_around_the_rule(kind, L, S, V, n_keys, zeros, labels, monkeypatch):
    monkeypatch.delenv("GALVATRON_DP_REDUCE", raising=False)
    monkeypatch.delenv("GALVATRON_DP_SKIP", raising=False)
    x = _instance(L, S, V, kind, n_keys)
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4], f0=np.zeros((V, S)) if zeros else None)
    _lib.batch_stats_begin()
    _lib.solve_batch([prob])
    s = _lib.batch_stats_end()
    assert (s.executed < 0.01 * s.relaxations) == labels
    _same(prob, x, V, f"{kind} {L} {S} {V} {n_keys} {zeros}")


# One key with many labels among keys with few, which by themselves are solved by labels: what it is given up for takes them along, and
# the next run starts from bounds of its own.  In a batch the other instances go on by labels.
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 6])
def test_a_key_that_is_given_up_takes_the_others_along(n, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    L, S, V = 24, 64, 12000
    xs = []
    for k in (3, 0, 1, 2, 4, 5)[:n]:
        rng = np.random.Generator(np.random.PCG64([L, S, k]))
        per = V // L
        mem = np.repeat(rng.integers(per // 4, 3 * per, size=(1, S)), L, 0).astype(np.int32)
        intra = 40.0 * per / mem
        intra[:, ::3] += 1e3                       # a third is dominated
        xs.append((mem, intra, np.repeat(rng.uniform(0, 0.05, size=(1, S, S)), L, 0), [0, V // 2, 6 * V // 10], [0.0, 0.5, 1.0]))
    probs = [_lib.Problem(x[0], x[1], x[2], V, x[3], x[4]) for x in xs]
    given_up = [_executed([prob]) for prob in probs]
    assert given_up[0] > 0.01 and max(given_up[1:], default=0) < 1e-3
    x = xs[0]
    assert all(_executed([_lib.Problem(x[0], x[1], x[2], V, x[3][k:k + 1], x[4][k:k + 1])]) < 1e-3 for k in (1, 2))
    for _ in range(3):
        _lib.solve_batch(probs)
    for x, prob in zip(xs, probs):
        _same(prob, x, V, f"{n}")


# The bounds of 128 multipliers beside 4 keys need 70.6 of 67.1 MB
@pytest.mark.gpu
def test_static_calls_whose_bounds_need_most_of_the_workspace(monkeypatch):
    monkeypatch.delenv("GALVATRON_DP_REDUCE", raising=False)
    monkeypatch.delenv("GALVATRON_DP_SKIP", raising=False)
    L, S, V, T = 128, 128, 2000, 40
    mem, intra, inter, om, ot = _instance(L, S, V, "each", 4)
    index = (np.arange(L) * T // L).astype(np.int32)
    prob = _lib.Problem(mem, intra, inter[:T], V, om, ot, inter_index=index)
    _lib.batch_stats_begin()
    _lib.solve_static(prob)
    s = _lib.batch_stats_end()
    _same(prob, (mem, intra, np.ascontiguousarray(inter[:T][index]), om, ot), V, "static")
    assert s.executed < 0.01 * s.relaxations


# Less memory than a workgroup for every key works in, of the device or allowed for, and not less than one for all of them (8 keys), or
# than 64 multipliers (1 key, 24 MB with 128)
@pytest.mark.gpu
@pytest.mark.parametrize("L,S,n_keys,limit_mb", [(40, 20, 8, 3), (80, 64, 1, 20)])
@pytest.mark.parametrize("limit", ["GALVATRON_DP_ARENA_MB", "GALVATRON_DP_DEVICE_LIMIT_MB"])
def test_calls_and_batches_whose_bounds_have_little_room(L, S, n_keys, limit_mb, limit, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    monkeypatch.setenv(limit, str(limit_mb))
    _lib.cache_trim()
    V = 4000
    for many in (1, 2):
        xs = [_instance(L, S, V + i, "each", n_keys) for i in range(many)]
        probs = [_lib.Problem(x[0], x[1], x[2], V, x[3], x[4]) for x in xs]
        if many > 1 and limit == "GALVATRON_DP_DEVICE_LIMIT_MB":
            monkeypatch.setenv(limit, str(many * limit_mb))   # (a batch whose bounds are not to be had in one piece is solved whole)
        _lib.batch_stats_begin()
        _lib.solve_batch(probs)
        s = _lib.batch_stats_end()
        assert s.executed < 0.01 * s.relaxations
        for x, prob in zip(xs, probs):
            _same(prob, x, V, f"{many} {limit}")


@pytest.mark.gpu
@pytest.mark.parametrize("L,S,n_keys,limit_mb", [(40, 20, 8, 3), (80, 64, 1, 20)])
def test_plans_whose_bounds_have_little_room(L, S, n_keys, limit_mb, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    monkeypatch.setenv("GALVATRON_DP_ARENA_MB", str(limit_mb))
    V, x = 2000, _instance(L, S, 2000, "each", n_keys)
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4])
    with _lib.Plan([prob]) as plan:
        assert plan.run().relax_launches == 0
        plan.fetch()
    _same(prob, x, V, "plan")
