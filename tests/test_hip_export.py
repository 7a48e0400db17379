"""The exported tables through the plugin signature: pieces and widths of the copy, and the caller's arrays that are
written directly or through a copy."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import galvatron_dp_core as shim
from galvatron_dp import _build, _lib, workloads as W
from oracle import dp_oracle as O

pytestmark = pytest.mark.gpu


# S = 255: a byte per entry of the argmin table, 256: four; 1 MB pieces: less than one, one and a bit, several
@pytest.mark.parametrize("L,S,V", [(2, 1, 40), (3, 255, 60), (3, 256, 60), (3, 22, 16000), (9, 7, 40000)])
@pytest.mark.parametrize("direct", [True, False])
def test_exported_tables(L, S, V, direct):
    inst = W.random_instance(np.random.Generator(np.random.PCG64([L, S, V])), L, S, V, mem_hi=max(2, V // L), inf_frac=0.1, n_keys=2)
    want = O.solve(inst.mem, inst.intra, inst.inter, V, inst.other_mem, inst.other_time, keep=True)
    f, mark = np.zeros((V, S)), np.full((L, V, S), -1, dtype=np.int32)
    if not direct:                                   # other strides and another type: written through a copy
        f, mark = np.zeros((S, V)).T, mark.astype(np.int64)
    res = {k: np.full(L, -1, dtype=np.int32) for k in inst.other_mem}
    shim.set_export(True)
    try:
        total, left = shim.dynamic_programming_core(L, V, S, inst.mem, mark, f, inst.inter, inst.intra, inst.other_mem, inst.other_time, res)
    finally:
        shim.set_export(False)
    assert np.array_equal(mark, want[4]) and np.ascontiguousarray(f).tobytes() == want[3].tobytes()
    for k in want[0]:
        assert np.float64(total[k]).tobytes() == np.float64(want[0][k]).tobytes() and left[k] == want[2][k]


# 12 layers as twice 6, 11 as 6 and 5, 3 (four bytes an entry) as 2 and 1, 5 one at a time
@pytest.mark.parametrize("L,S,V,limit_mb", [(12, 8, 12000, 1), (11, 16, 7000, 1), (3, 256, 1000, 2), (5, 10, 100000, 1)])
def test_exported_tables_in_what_memory_there_is(L, S, V, limit_mb, monkeypatch):
    """The device grants less than all layers take after the run: the table comes in several parts."""
    inst = W.random_instance(np.random.Generator(np.random.PCG64([L, S])), L, S, V, mem_hi=V // L, n_keys=1)
    want = O.solve(inst.mem, inst.intra, inst.inter, V, inst.other_mem, inst.other_time, keep=True)
    keys = sorted(inst.other_mem)
    prob = _lib.Problem(inst.mem, inst.intra, inst.inter, V, [inst.other_mem[k] for k in keys], [inst.other_time[k] for k in keys],
                        export_f=V * S * 8 <= limit_mb << 20, export_mark=True)
    with _lib.Plan([prob]) as plan:
        plan.run()
        monkeypatch.setenv("GALVATRON_DP_DEVICE_LIMIT_MB", str(limit_mb))
        plan.fetch()
    assert np.array_equal(prob.mark_out, want[4])
    assert prob.f_out is None or prob.f_out.tobytes() == want[3].tobytes()


def test_no_host_memory_for_the_pieces(tmp_path):
    """An error code, and nothing written to the costs, where the pieces of the copy cannot be had."""
    here, exe = os.path.dirname(os.path.abspath(__file__)), str(tmp_path / "export_check")
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(here, "sanitize", "export_check.cpp"), _build.LIB_PATH, "-Wl,-rpath," + _build.LIB_DIR,
                    "-Wl,--allow-shlib-undefined", "-o", exe], check=True, capture_output=True)
    run = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert run.returncode == 0 and "fetched" in run.stdout, run.stdout
