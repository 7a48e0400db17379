"""The DP over what the bounds leave, as labels: numbers of keys, labels and strategies around which the kernels branch,
in batches, plans and static calls; against the C oracle, which sees the whole instance."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from galvatron_dp import _lib
from oracle import dp_oracle as O


def _instance(rng, L, S, V, kind, n_keys):
    """kind: 'each' random costs per layer; 'trade' equal layers that trade memory for time, whose labels are many;
    'narrow' layers in which one strategy is the best by far, between random ones."""
    per = V // L
    n = 1 if kind == "trade" else L
    mem = rng.integers(max(1, per // 4), max(2, 3 * per), size=(n, S)).astype(np.int32)
    intra, inter = rng.lognormal(2.5, 0.5, size=(n, S)), rng.uniform(0, 5, size=(n, S, S))
    if kind == "trade":
        intra, inter = 40.0 * per / mem * rng.uniform(0.98, 1.02, size=mem.shape), inter * 0.05
        mem, intra, inter = np.repeat(mem, L, 0), np.repeat(intra, L, 0), np.repeat(inter, L, 0)
    if kind == "narrow":
        intra[::3] += 1e4
        intra[::3, S // 2], mem[::3, S // 2] = 1.0, 1
    om = [int(V * f) for f in (0.3, 0.1, 0.0, 0.45, 0.2, 0.999, 0.25, 2.0)[:n_keys]]
    return mem, intra, inter, om, [k / 3 for k in range(n_keys)]


def _problem(x, V):
    return _lib.Problem(x[0], x[1], x[2], V, x[3], x[4])


def _want(x, V):
    keys = range(len(x[3]))
    return O.solve(x[0], x[1], x[2], V, dict(zip(keys, x[3])), dict(zip(keys, x[4])))[:3]


def _check(prob, want, tag):
    total, res, left = want
    for k in total:
        assert np.float64(prob.total[k]).tobytes() == np.float64(total[k]).tobytes(), f"{tag} key {k}: {prob.total[k]} {total[k]}"
        assert int(prob.remaining[k]) == left[k], f"{tag} key {k}"
        if left[k] >= 0:
            assert [int(v) for v in prob.res[k]] == [int(v) for v in res[k]], f"{tag} key {k}"


def _solved_by_labels(probs):
    _lib.batch_stats_begin()
    _lib.solve_batch(probs)
    s = _lib.batch_stats_end()
    return s.executed < 0.01 * s.relaxations


# Labels of the layers that have the most: 1 to 64 (a turn), to 128 and 192 (lanes share the keys), more (buckets), more
# than fit (the smaller instance, or the whole one); a set: with so many keys they fit
@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V,labels", [("each", 9, 12, 6000, True), ("narrow", 20, 16, 9000, True), ("trade", 6, 7, 3000, True),
                                               ("trade", 10, 8, 6000, True), ("trade", 16, 9, 9000, True), ("trade", 24, 24, 12000, {1, 5}),
                                               ("each", 40, 64, 9000, True), ("each", 64, 17, 9000, True), ("narrow", 512, 4, 20000, False)])
@pytest.mark.parametrize("n_keys", [1, 2, 3, 5, 8])
def test_batches_by_labels(kind, L, S, V, labels, n_keys, monkeypatch):
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    x = _instance(np.random.Generator(np.random.PCG64([L, S, n_keys])), L, S, V, kind, n_keys)
    prob = _problem(x, V)
    by_labels = _solved_by_labels([prob])
    _check(prob, _want(x, V), f"{kind} {L} {S} {V}")
    assert by_labels == (n_keys in labels if isinstance(labels, set) else labels)


@pytest.mark.gpu
@pytest.mark.parametrize("S", [2, 16, 17, 24, 25, 32, 33, 40, 41, 48, 49, 64, 65, 88, 89, 128])
def test_passes_over_one_matrix_some_and_many(S, monkeypatch):
    """Matrices: the same for all layers, another from the middle on (both held), another for every second layer."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    rng, L, V, probs, xs = np.random.Generator(np.random.PCG64(S)), 9, 2000, [], []
    for index in ([0] * L, [0] * 5 + [1] * 4, [l // 2 for l in range(L)]):
        x = _instance(rng, L, S, V, "each", 3)
        x = (x[0], x[1], np.ascontiguousarray(x[2][index]), x[3], x[4])
        xs.append(x)
        probs.append(_problem(x, V))
    for x, prob in zip(xs, probs):
        assert _solved_by_labels([prob])     # (bounds of no use leave too many of them)
        _check(prob, _want(x, V), f"S {S}")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["each", "trade"])
def test_plans_by_labels(kind, monkeypatch):
    """Runs in turn, what is fetched after the bounds were given back, and the launch schemes after it."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    V, rng = 5000, np.random.Generator(np.random.PCG64(8))
    xs = [_instance(rng, L, 12, V, kind, 3) for L in (12, 5)] + [_instance(rng, 30, 30, V, kind, 2)]
    want, probs = [_want(x, V) for x in xs], [_problem(x, V) for x in xs]

    def fetched(plan):
        for p in probs:
            p.total[:], p.remaining[:], p.res[:] = 0, 0, 0
        plan.fetch()
        for i, (p, w) in enumerate(zip(probs, want)):
            _check(p, w, f"{kind} instance {i}")
    with _lib.Plan(probs) as plan:
        by_labels = plan.run().relax_launches == 0
        assert by_labels or kind == "trade"
        fetched(plan)
        t = plan.run(1)
        assert t.total_ms > 0 and (t.relax_launches == 0) == by_labels
        fetched(plan)
        assert plan.run(2).relax_launches > 0
        fetched(plan)
        plan.run()
        plan.set_option(1, 0)              # GDP_OPT_FUSED: about the launch schemes, which run from here on
        fetched(plan)
        assert plan.run(1).relax_launches > 0
        fetched(plan)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V,n_keys,labels", [("each", 2, 3, 200, 2, False), ("each", 5, 8, 3000, 3, False), ("each", 5, 11, 3000, 3, True),
                                                      ("each", 30, 30, 5000, 8, True), ("trade", 10, 8, 6000, 2, True), ("trade", 30, 30, 9000, 1, True),
                                                      ("narrow", 21, 16, 6000, 5, False)])
def test_static_calls_by_labels(kind, L, S, V, n_keys, labels):
    """labels: False below the 36 us of layer launches from which bounds are taken, and where the labels are too many."""
    if "GALVATRON_DP_REDUCE" in os.environ or "GALVATRON_DP_SKIP" in os.environ:
        pytest.skip("the environment presets the rule")
    x = _instance(np.random.Generator(np.random.PCG64([L, S])), L, S, V, kind, n_keys)
    prob = _problem(x, V)
    for _ in range(2):
        prob.total[:], prob.remaining[:], prob.res[:] = 0, 0, 0
        _lib.batch_stats_begin()
        _lib.solve_static(prob)
        s = _lib.batch_stats_end()
        _check(prob, _want(x, V), f"{kind} {L} {S}")
        assert (s.executed < 0.01 * s.relaxations) == labels


@pytest.mark.parametrize("source", ["gdp_bounds.hip", "gdp_frontier.hip"])
def test_the_kernels_launchers_allocate_nothing(source, tmp_path):
    """gdp_solve_static calls them: no allocator, no stream or event, and no function of the library beside them."""
    from galvatron_dp import _build
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    obj = str(tmp_path / "o.o")
    flags = [f for f in _build.HIPCC_FLAGS if f != "-shared"]
    subprocess.run([hipcc] + flags + ["-c", os.path.join(_build.CSRC, source), "-o", obj], check=True, capture_output=True)
    undefined = subprocess.run(["nm", "-u", "-C", obj], stdout=subprocess.PIPE, text=True, check=True).stdout
    names = [ln.split(None, 1)[1].strip() for ln in undefined.splitlines() if ln.strip().startswith("U ")]
    assert any(n.startswith("hipLaunchKernel") for n in names), names
    for n in names:
        assert not n.startswith(("hipMalloc", "hipHost", "hipExtMalloc", "hipMem", "hipStream", "hipEvent", "hipFree", "operator", "gdp_",
                                 "malloc", "calloc", "realloc", "posix_memalign", "aligned_alloc", "std::__throw")), n


@pytest.mark.parametrize("source,kernels", [("gdp_bounds.hip", ("pass", "upper", "keep", "transpose")), ("gdp_frontier.hip", ("frontier",)),
                                            ("gdp_kernels.hip", ("gdp_relax_kernel", "init", "zero_pass", "epilogue"))])
def test_kernels_of_static_calls_have_no_scratch_memory(source, kernels):
    """Scratch memory is device memory that the runtime may have to obtain for a launch: the kernels of gdp_solve_static spill nothing."""
    from galvatron_dp import _build
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    flags = [f for f in _build.HIPCC_FLAGS if f != "-shared"]
    log = subprocess.run([hipcc] + flags + ["-c", "--offload-device-only", "-Rpass-analysis=kernel-resource-usage",
                                            os.path.join(_build.CSRC, source), "-o", os.devnull], check=True, capture_output=True, text=True).stderr
    found = re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", log, re.S)
    for part in kernels:
        own = [(name, int(size)) for name, size in found if part in name]
        assert own and all(size == 0 for _, size in own), (part, own)


@pytest.mark.gpu
def test_what_is_given_up_goes_on_after_the_initial_costs_were_begun(monkeypatch):
    """The calling thread looks through initial costs while the bounds run, and asks between pieces whether they are done;
    the launches of the smaller instance come after that."""
    L, S, V = 40, 24, 200000
    x = _instance(np.random.Generator(np.random.PCG64(3)), L, S, V, "trade", 2)
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    whole = _problem(x, V)
    _lib.solve_batch([whole])
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4], f0=np.zeros((V, S)))
    assert not _solved_by_labels([prob])
    assert prob.total.tobytes() == whole.total.tobytes() and np.array_equal(prob.remaining, whole.remaining)
    assert np.array_equal(prob.res, whole.res)


# The line of a single call: 3e7 relaxations where layers are their own and few strategies undominated, 5e7 a layer (3e8 at
# least) otherwise; initial costs that take longer than the chain of layers
@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V,zeros,labels", [("each", 10, 20, 7400, False, False), ("each", 10, 20, 7600, False, True),
                                                     ("each", 10, 20, 7600, True, True), ("each", 10, 20, 60000, True, False),
                                                     ("each", 3, 89, 7600, False, False), ("trade", 6, 20, 20000, False, False),
                                                     ("trade", 3, 20, 250100, False, True), ("each", 256, 8, 9000, False, False)])
def test_single_calls_around_the_rule(kind, L, S, V, zeros, labels):
    if "GALVATRON_DP_REDUCE" in os.environ or "GALVATRON_DP_SKIP" in os.environ:
        pytest.skip("the environment presets the rule")
    x = _instance(np.random.Generator(np.random.PCG64([L, S])), L, S, V, kind, 3)
    prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4], f0=np.zeros((V, S)) if zeros else None)
    by_labels = _solved_by_labels([prob])
    _check(prob, _want(x, V), f"{kind} {L} {S} {V}")
    assert by_labels == labels


@pytest.mark.gpu
@pytest.mark.parametrize("kind,L,S,V", [("each", 30, 30, 5000), ("each", 24, 16, 6000), ("trade", 10, 8, 6000)])
def test_static_calls_do_without_bounds_where_told(kind, L, S, V, monkeypatch):
    """By labels unless the environment or the caller asks for every cell; told by the statistics."""
    monkeypatch.delenv("GALVATRON_DP_REDUCE", raising=False)
    monkeypatch.delenv("GALVATRON_DP_SKIP", raising=False)
    x = _instance(np.random.Generator(np.random.PCG64([L, S])), L, S, V, kind, 3)
    want = _want(x, V)

    def share(**flags):
        prob = _lib.Problem(x[0], x[1], x[2], V, x[3], x[4], **flags)
        _lib.batch_stats_begin()
        _lib.solve_static(prob)
        s = _lib.batch_stats_end()
        _check(prob, want, f"{kind} {flags}")
        assert s.instances == 1 and s.relaxations == prob.relaxations
        return s.executed / s.relaxations
    assert share() < 0.01 and share(launch="fused") < 0.01
    assert share(compute_all=True) == 1
    monkeypatch.setenv("GALVATRON_DP_SKIP", "0")
    assert share() == 1
    monkeypatch.setenv("GALVATRON_DP_SKIP", "1")
    assert share() < 0.01
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
    assert share() == 1


@pytest.mark.gpu
@pytest.mark.parametrize("L,S,V,n_keys,shared", [(30, 37, 9000, 2, False), (24, 30, 8000, 8, False), (40, 16, 9000, 3, True), (24, 40, 5000, 6, True)])
def test_static_calls_left_with_many_labels(L, S, V, n_keys, shared):
    """Every layer trades memory for time and has other strategies, a third of them, that cannot pay: what stays is solved by
    the dense recurrence, and said in the terms of the whole instance; `shared`: matrices behind an index."""
    if "GALVATRON_DP_REDUCE" in os.environ or "GALVATRON_DP_SKIP" in os.environ:
        pytest.skip("the environment presets the rule")
    rng = np.random.Generator(np.random.PCG64([L, S, n_keys]))
    mem, intra, inter, om, ot = _instance(rng, L, S, V, "trade", n_keys)
    for l in range(L):
        order = rng.permutation(S)
        mem[l], intra[l] = mem[l][order], intra[l][order]
        intra[l][rng.permutation(S)[:S // 3 + l % 3]] += 1e4
    if shared:
        tables, index = inter[:3], (np.arange(L) % 3).astype(np.int32)
        prob = _lib.Problem(mem, intra, tables, V, om, ot, inter_index=index)
        inter = np.ascontiguousarray(tables[index])
    else:
        prob = _lib.Problem(mem, intra, inter, V, om, ot)
    _lib.batch_stats_begin()
    _lib.solve_static(prob)
    s = _lib.batch_stats_end()
    _check(prob, _want((mem, intra, inter, om, ot), V), f"{L} {S} {V}")
    assert 0.1 < s.executed / s.relaxations < 0.75


@pytest.mark.gpu
@pytest.mark.parametrize("L,S,V,n_keys,kinds,seed", [(39, 9, 5072, 5, 2, 167), (31, 11, 4894, 4, 1, 346), (23, 13, 6952, 5, 23, 654), (42, 20, 3016, 2, 2, 887)])
def test_labels_are_not_given_up_near_the_last_layer(L, S, V, n_keys, kinds, seed):
    """Labels that are many, and late: what they have taken counts no more than what is ahead.  `kinds` of layers that trade
    memory for time."""
    if "GALVATRON_DP_REDUCE" in os.environ or "GALVATRON_DP_SKIP" in os.environ:
        pytest.skip("the environment presets the rule")
    rng = np.random.Generator(np.random.PCG64(seed))
    rng.integers(12, 48), rng.integers(8, 24), rng.integers(1, 6), rng.integers(1500, 7000)
    per, which = V // L, np.arange(L) * kinds // L
    mem = rng.integers(max(1, per // 4), max(2, 3 * per), size=(kinds, S)).astype(np.int32)
    intra, inter = 40.0 * per / mem * rng.uniform(0.98, 1.02, size=(kinds, S)), rng.uniform(0, 0.25, size=(kinds, S, S))
    om = [int(V * f) for f in (0.3, 0.1, 0.0, 0.45, 0.2)[:n_keys]]
    x = mem[which], intra[which], inter[which], om, [k / 3 for k in range(n_keys)]
    prob = _problem(x, V)
    _lib.batch_stats_begin()
    _lib.solve_static(prob)
    s = _lib.batch_stats_end()
    _check(prob, _want(x, V), f"{L} {S} {V}")
    assert s.executed < 0.01 * s.relaxations


@pytest.mark.gpu
def test_a_call_by_labels_needs_no_dense_buffers(monkeypatch):
    """A device too full for the dense recurrence, but not for the bounds and the labels: solved by them,
    below the line of batches and above it; refused where they are switched off, or where the labels are too many."""
    for name in ("GALVATRON_DP_REDUCE", "GALVATRON_DP_SKIP"):
        monkeypatch.delenv(name, raising=False)
    _lib.cache_trim()
    monkeypatch.setenv("GALVATRON_DP_DEVICE_LIMIT_MB", "4")
    for L, S, V in ((12, 40, 12000), (8, 40, 200000)):     # 2.3e8 relaxations, 2.6e9; 8 MB and 130 at least
        x = _instance(np.random.Generator(np.random.PCG64([L, S])), L, S, V, "each", 3)
        prob = _problem(x, V)
        assert _solved_by_labels([prob])
        _check(prob, _want(x, V), f"{L} {S} {V}")
        monkeypatch.setenv("GALVATRON_DP_REDUCE", "0")
        with pytest.raises(MemoryError):
            _lib.solve_batch([_problem(x, V)])
        monkeypatch.delenv("GALVATRON_DP_REDUCE")
    x = _instance(np.random.Generator(np.random.PCG64(3)), 40, 24, 200000, "trade", 2)
    with pytest.raises(MemoryError):
        _lib.solve_batch([_problem(x, 200000)])


@pytest.mark.gpu
@pytest.mark.parametrize("limit_mb", [None, 8, 2])
def test_plans_hold_no_more_for_their_bounds_than_a_batch_works_in(limit_mb, monkeypatch):
    """4 instances whose bounds take 1 MB each."""
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    if limit_mb is not None:
        monkeypatch.setenv("GALVATRON_DP_ARENA_MB", str(limit_mb))
    L, S, V, rng = 12, 24, 3000, np.random.Generator(np.random.PCG64(12))
    xs = [_instance(rng, L, S, V, "each", 2) for _ in range(4)]
    probs = [_problem(x, V) for x in xs]
    with _lib.Plan(probs) as plan:
        by_labels = plan.run().relax_launches == 0
        plan.fetch()
    for x, prob in zip(xs, probs):
        _check(prob, _want(x, V), f"limit {limit_mb}")
    assert by_labels == (limit_mb != 2)


@pytest.mark.gpu
@pytest.mark.parametrize("L,S,n_keys,V,seed", [(8, 48, 5, 44101, 203), (10, 52, 3, 35964, 205)])
def test_single_calls_whose_labels_take_longer_than_what_stays(L, S, n_keys, V, seed, monkeypatch):
    """Equal layers that trade memory for time: their labels fit (GALVATRON_DP_REDUCE=1 waits for them), but the smaller instance
    takes less."""
    for name in ("GALVATRON_DP_REDUCE", "GALVATRON_DP_SKIP"):
        monkeypatch.delenv(name, raising=False)
    rng = np.random.Generator(np.random.PCG64(seed))
    rng.integers(5, 16), rng.integers(20, 56), rng.integers(1, 6), rng.integers(20000, 90000)
    per = V // L
    mem = rng.integers(max(1, per // 4), max(2, 3 * per), size=(1, S)).astype(np.int32)
    intra, inter = 40.0 * per / mem * rng.uniform(0.98, 1.02, size=(1, S)), rng.uniform(0, 0.25, size=(1, S, S))
    om = [int(V * f) for f in (0.3, 0.1, 0.0, 0.45, 0.2)[:n_keys]]
    x = np.repeat(mem, L, 0), np.repeat(intra, L, 0), np.repeat(inter, L, 0), om, [k / 3 for k in range(n_keys)]
    prob, want = _problem(x, V), _want(x, V)
    assert not _solved_by_labels([prob])
    _check(prob, want, f"{L} {S}")
    monkeypatch.setenv("GALVATRON_DP_REDUCE", "1")
    assert _solved_by_labels([prob])
    _check(prob, want, f"{L} {S} by labels")
