"""Instances whose strategies are thinned out by bounds before the DP: results against the C oracle, which sees the
whole instance.  The bounds take part in every instance of the form here (``GALVATRON_DP_REDUCE=1``; by default
only from a certain amount of work on)."""
import numpy as np
import pytest

import helpers as H
from galvatron_dp import _lib, workloads as W
from oracle import dp_oracle as O

pytestmark = pytest.mark.gpu

# L, S, V: two layers and the most; strategies around the parts of a pass (32, 33, 64, 65), elements per thread 1 to
# 16 (89 and 128 need 16) and the largest; budgets from a few bins on
SHAPES = [(2, 2, 40), (2, 128, 300), (3, 5, 64), (5, 31, 400), (4, 32, 333), (6, 33, 500), (4, 44, 1000), (3, 64, 700),
          (7, 65, 512), (5, 88, 900), (4, 89, 600), (12, 9, 3000), (40, 6, 4001), (24, 22, 2500), (512, 3, 2600)]


def _instance(rng, L, S, V, kind):
    per = max(2, V // L)
    same = kind in ("same", "ties_same")
    n = 1 if same else L
    mem = rng.integers(max(1, per // 4), 3 * per + 1, size=(n, S)).astype(np.int32)
    if kind.startswith("ties"):
        intra, inter = rng.integers(1, 5, size=(n, S)).astype(float), rng.integers(0, 3, size=(n, S, S)).astype(float)
        mem = (mem // 4 + 1).astype(np.int32)
    else:
        intra, inter = rng.lognormal(2.5, 0.5, size=(n, S)), rng.uniform(0, 5, size=(n, S, S))
    if kind == "trade":                    # what saves memory costs time: few strategies are dominated by another
        intra = 40.0 * per / mem * rng.uniform(0.98, 1.02, size=mem.shape)
    if kind == "negative":
        intra, inter = intra - 20.0, inter - 2.5
    if kind == "holes":
        intra[rng.uniform(size=intra.shape) < 0.2] = np.inf
        inter[rng.uniform(size=inter.shape) < 0.2] = np.inf
        mem[rng.uniform(size=mem.shape) < 0.2] = V + 3
        intra[:, 0], mem[:, 0] = 10.0, max(1, per // 2)
        inter[:, 0, 0] = 0.0
    if kind == "loose":
        mem = np.minimum(mem, max(1, per // 2)).astype(np.int32)
    if n == 1:
        mem, intra, inter = np.repeat(mem, L, 0), np.repeat(intra, L, 0), np.repeat(inter, L, 0)
    # a key with the whole budget, tighter ones, one without a solution, one below the table
    om = {1: 0, 2: V // 10, 4: V // 4, 8: V - 2, 16: V + 5}
    ot = {k: float(k) / 3 for k in om}
    return mem, intra, inter, om, ot


def _problem(x, V):
    mem, intra, inter, om, ot = x
    keys = sorted(om)
    return _lib.Problem(mem, intra, inter, V, [om[k] for k in keys], [ot[k] for k in keys])


def _check(x, V, prob, tag):
    mem, intra, inter, om, ot = x
    keys = sorted(om)
    got = ({k: prob.total[i] for i, k in enumerate(keys)}, {k: [int(v) for v in prob.res[i]] for i, k in enumerate(keys)},
           {k: int(prob.remaining[i]) for i, k in enumerate(keys)})
    wt, wr, wm = O.solve(mem, intra, inter, V, om, ot)[:3]
    H.assert_same_results(got, (wt, wr, wm), tag)


@pytest.mark.parametrize("shape", SHAPES)
def test_reduced_instances_against_oracle(shape, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    L, S, V = shape
    for n, kind in enumerate(["each", "same", "ties", "ties_same", "negative", "holes", "loose"]):
        x = _instance(np.random.Generator(np.random.PCG64([5, L, S, n])), L, S, V, kind)
        prob = _problem(x, V)
        _lib.solve_batch([prob])
        _check(x, V, prob, f"{shape} {kind}")


def test_batch_of_different_shapes_and_shared_tables(monkeypatch):
    """One set of launches over instances of different sizes, some of them without the form (a memory cost of 0), some
    of them with the same matrices."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    rng = np.random.Generator(np.random.PCG64(99))
    xs, probs = [], []
    for n, (L, S, V) in enumerate(SHAPES[:12]):
        x = _instance(rng, L, S, V, ["each", "ties", "same"][n % 3])
        if n == 5:
            x[0][1, 1] = 0
        xs.append((x, V))
        probs.append(_problem(x, V))
    tables = rng.uniform(0, 4, size=(2, 20, 20))
    for L in (4, 7, 9):
        mem, intra, _, om, ot = _instance(rng, L, 20, 800, "each")
        index = (np.arange(L) % 2).astype(np.int32)
        x = (mem, intra, tables[index], om, ot)
        keys = sorted(om)
        xs.append((x, 800))
        probs.append(_lib.Problem(mem, intra, tables, 800, [om[k] for k in keys], [ot[k] for k in keys], inter_index=index))
    _lib.solve_batch(probs)
    for n, ((x, V), prob) in enumerate(zip(xs, probs)):
        _check(x, V, prob, f"instance {n}")


def _work(probs):
    """Relaxations carried out of all a batch stands for."""
    _lib.batch_stats_begin()
    _lib.solve_batch(probs)
    s = _lib.batch_stats_end()
    assert s.instances == len(probs) and s.relaxations == sum(prob.relaxations for prob in probs)
    return s.executed / s.relaxations


# The limits of the form -- layers, strategies, both together, keys -- and one beyond each; costs that trade memory
# for time.  Compared with the whole instance, which other tests compare with the oracle.
@pytest.mark.parametrize("L,S,V,keys,kind,taken", [
    (512, 24, 6000, 3, "each", True), (513, 24, 6000, 3, "each", False), (512, 80, 3000, 2, "each", True), (320, 128, 3000, 2, "each", True),
    (321, 128, 3000, 2, "each", False), (12, 128, 4000, 2, "each", True), (12, 129, 4000, 2, "each", False), (16, 40, 4000, 8, "each", True),
    (16, 40, 4000, 9, "each", False), (16, 40, 8000, 1, "trade", True), (24, 64, 12000, 4, "trade", True), (6, 89, 9000, 3, "trade", True)])
def test_bounds_take_part_up_to_their_limits(L, S, V, keys, kind, taken, monkeypatch):
    rng = np.random.Generator(np.random.PCG64([L, S, keys]))
    mem, intra, inter, _, _ = _instance(rng, L, S, V, kind)
    om, ot = [V // 3 * k // keys for k in range(keys)], [float(k) for k in range(keys)]
    probs = [_lib.Problem(mem, intra, inter, V, om, ot) for _ in range(2)]
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    whole = _work(probs[:1])
    assert np.isfinite(probs[0].total).all()
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    done = _work(probs[1:])
    assert done < 0.6 * whole if taken else done == whole
    assert probs[0].total.tobytes() == probs[1].total.tobytes()
    assert np.array_equal(probs[0].remaining, probs[1].remaining) and np.array_equal(probs[0].res, probs[1].res)


# instances, L, S, V: on the far side of each term of the rule -- too little work, too many layers, more than 88
# strategies, too many transition costs that stay in a batch -- and on the near one
@pytest.mark.parametrize("shape,kind,bounds", [
    ((1, 24, 40, 30000), "each", False), ((1, 16, 64, 40000), "each", True), ((1, 256, 16, 33000), "each", False),
    ((1, 40, 64, 30000), "each", True), ((1, 24, 96, 12000), "each", False), ((1, 4, 96, 80000), "each", True),
    ((64, 14, 40, 4000), "trade", False), ((64, 14, 40, 4000), "each", True), ((8, 14, 24, 45000), "each", True)])
def test_bounds_are_taken_where_they_pay(shape, kind, bounds, monkeypatch):
    n, L, S, V = shape
    rng = np.random.Generator(np.random.PCG64(list(shape)))
    xs = [_instance(rng, L, S, V, kind) for _ in range(n)]
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    whole = [_problem(x, V) for x in xs]
    all_of_it = _work(whole)
    monkeypatch.delenv("GALVATRON_DP_REDUCE")
    probs = [_problem(x, V) for x in xs]
    done = _work(probs)
    assert done < 0.5 * all_of_it if bounds else done == all_of_it
    for a, b in zip(probs, whole):
        assert a.total.tobytes() == b.total.tobytes()
        assert np.array_equal(a.remaining, b.remaining) and np.array_equal(a.res, b.res)


@pytest.mark.parametrize("limit_mb", [32, 1])
def test_bounds_stay_within_the_largest_allocation(limit_mb, monkeypatch):
    """40 instances whose bounds take 1.1 MB of device memory each: within GALVATRON_DP_ARENA_MB = 32 they are taken in
    two slices; with 1 MB, less than an instance needs, all instances are solved whole.  (The first limit is one the
    device sets as well.)"""
    rng = np.random.Generator(np.random.PCG64(32))
    L, S, V = 24, 40, 2500
    xs = [_instance(rng, L, S, V, "each") for _ in range(40)]
    probs = [_problem(x, V) for x in xs]
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    whole = _work(probs)
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    monkeypatch.setenv("GALVATRON_DP_ARENA_MB", str(limit_mb))
    if limit_mb == 32:
        monkeypatch.setenv("GALVATRON_DP_DEVICE_LIMIT_MB", str(limit_mb))
    done = _work(probs)
    assert done < 0.3 * whole if limit_mb == 32 else done > 0.7 * whole   # (the tiles of a part are those of its size)
    for n, (x, prob) in enumerate(zip(xs[::13], probs[::13])):
        _check(x, V, prob, f"instance {13 * n}")


def test_no_page_locked_memory_for_the_bounds(monkeypatch):
    """260 instances whose marks of what stays are 1.7 MB, and whose results are less than the 1 MB that can be had:
    solved whole, in two parts.  (The inputs of a part, 18 MB and more, are laid out in ordinary memory anyway.)"""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    monkeypatch.setenv("GALVATRON_DP_PINNED_LIMIT_MB", "1")
    rng = np.random.Generator(np.random.PCG64(260))
    L, S, V, n = 60, 100, 200, 260
    tables = rng.uniform(0, 5, size=(1, S, S))
    index = np.zeros(L, np.int32)
    mem, intra, _, om, ot = _instance(rng, L, S, V, "same")
    keys = sorted(om)
    probs = []
    for i in range(n):
        probs.append(_lib.Problem(mem, np.roll(intra, i, axis=1), tables, V, [om[k] for k in keys], [ot[k] for k in keys], inter_index=index))
    _lib.solve_batch(probs)
    for i in (0, 17, n - 1):
        _check((mem, probs[i].intra, np.repeat(tables, L, 0), om, ot), V, probs[i], f"instance {i}")


def test_initial_costs_that_are_not_zeros(monkeypatch):
    """The bounds take the initial costs to be zeros; a caller's array with others is solved whole."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    rng = np.random.Generator(np.random.PCG64(3))
    inst = W.with_initial_costs(W.random_instance(rng, 6, 12, 700, mem_hi=200), rng)
    got = H.hip_solve(inst)
    want = O.solve(inst.mem, inst.intra, inst.inter, inst.V, inst.other_mem, inst.other_time, f0=inst.f0)[:3]
    H.assert_same_results(got, want)


@pytest.mark.parametrize("strategies", [(22,), (23, 32), (33, 44, 9), (45, 8)])
def test_batches_with_narrow_passes(strategies, monkeypatch):
    """18 instances of up to 9, 22, 32, 44 and 45 strategies in one set of launches: passes as wide as the widest of them needs."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    rng = np.random.Generator(np.random.PCG64([7, *strategies]))
    V, xs = 400, []
    for n in range(18):
        L, S = (2, 5, 9)[n % 3], strategies[n % len(strategies)]
        xs.append(_instance(rng, L, S, V, ["each", "same", "ties", "negative", "holes", "loose"][n % 6]))
    probs = [_problem(x, V) for x in xs]
    _lib.solve_batch(probs)
    for n, (x, prob) in enumerate(zip(xs, probs)):
        _check(x, V, prob, f"{strategies} instance {n}")


@pytest.mark.parametrize("many", [63, 64, 80])
def test_instances_of_very_different_budgets(many, monkeypatch):
    """Many instances of one S whose budgets differ by a factor of 80: one group, and with it one launch."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    rng = np.random.Generator(np.random.PCG64(many))
    xs, probs = [], []
    for n in range(many):
        V = (40, 41, 160, 161, 640, 2560, 33, 50)[n % 8] if n else 2560
        x = _instance(rng, 3 + n % 4, 9, V, ["each", "ties"][n % 2])
        xs.append((x, V))
        probs.append(_problem(x, V))
    _lib.solve_batch(probs)
    for n, ((x, V), prob) in enumerate(zip(xs, probs)):
        _check(x, V, prob, f"instance {n}")
    with _lib.Plan(probs) as plan:
        t = plan.run(1)
        assert t.relax_launches == (1 if t.fused or t.flow else max(prob.L for prob in probs))


@pytest.mark.parametrize("shape", [(36, 96, 87000), (36, 96, 88000), (8, 96, 88000)])
@pytest.mark.parametrize("at", [None, 0, -1])
def test_large_initial_costs(shape, at):
    """Initial costs around 64 MB, from where on several threads look through them where the device takes longer (not
    with 8 layers): a call with zeros gives what one without gives, and one with a single other value at either end
    what a plan gives, which uploads them as they are."""
    L, S, V = shape
    x = _instance(np.random.Generator(np.random.PCG64([L, V])), L, S, V, "each")
    mem, intra, inter, om, ot = x
    f0 = np.zeros((V, S))
    if at is not None:
        f0.reshape(-1)[at] = -3.0
    keys = sorted(om)
    def problem(f):
        return _lib.Problem(mem, intra, inter, V, [om[k] for k in keys], [ot[k] for k in keys], f0=f)
    got, want = problem(f0), problem(None if at is None else f0)
    _lib.solve_batch([got])
    plan = _lib.Plan([want])
    plan.run()
    plan.fetch()
    assert got.total.tobytes() == want.total.tobytes()
    assert np.array_equal(got.remaining, want.remaining) and np.array_equal(got.res, want.res)


@pytest.mark.parametrize("threads", ["0", "1", "64"])
def test_as_many_helper_threads_as_told(threads, monkeypatch):
    """GALVATRON_DP_SCAN_THREADS: none, one and more than the machine may have look through the array as the caller's
    thread does, a single value included."""
    L, S, V = 36, 96, 88000
    mem, intra, inter, om, ot = _instance(np.random.Generator(np.random.PCG64([L, V])), L, S, V, "each")
    keys = sorted(om)
    f0 = np.zeros((V, S))

    def solved():
        prob = _lib.Problem(mem, intra, inter, V, [om[k] for k in keys], [ot[k] for k in keys], f0=f0)
        _lib.solve_batch([prob])
        return prob.total.tobytes(), prob.remaining.tobytes(), prob.res.tobytes()
    zeros = solved()
    monkeypatch.setenv("GALVATRON_DP_SCAN_THREADS", threads)
    assert solved() == zeros
    f0[50000, 7] = -300.0
    assert solved()[0] != zeros[0]
