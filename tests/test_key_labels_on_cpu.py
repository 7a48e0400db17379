"""The kernel of the DP over labels that has a workgroup for every key, its own source emulated on the CPU (emulation/): LDS holds garbage
at first, waves run in different orders, and another key's workgroup writes to this one's upper bound while it begins.  Bounds are numpy's, the
results are checked against the C oracle, which sees the whole instance."""
import ctypes
import os
import platform
import re
import shutil
import subprocess

import numpy as np
import pytest

from galvatron_dp import _build
from oracle import dp_oracle as O
from test_hip_key_labels import _instance

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
pytestmark = pytest.mark.skipif(shutil.which(CLANG) is None or platform.machine() != "x86_64", reason="needs clang for x86-64")
FAR, GIVEN_UP = 1e200, 2**64 - 2

_POINTERS = ("mem intra inter_f inter_t index lam budget P Q P_mem Q_mem end ub best keep marks other_time hist hist_mem hist_turns hist_intra out "
             "res").split()


class Instance(ctypes.Structure):   # GdpBoundInst
    _fields_ = ([(name, ctypes.c_void_p) for name in _POINTERS] + [("magnitude", ctypes.c_double), ("limit", ctypes.c_double)] +
                [(name, ctypes.c_int32) for name in ("L", "V", "S", "K", "T", "n_hist", "n_hist_turns", "n_lam")])


class Out(ctypes.Structure):        # GdpFrontierOut
    _fields_ = [("total", ctypes.c_double * 8), ("executed", ctypes.c_double * 8), ("remaining", ctypes.c_int32 * 8),
                ("status", ctypes.c_int32 * 8)]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    where = tmp_path_factory.mktemp("emulated")

    for name in ("gdp_key_labels.hip", "gdp_label_ops.h"):
        text = open(os.path.join(_build.CSRC, name)).read().split("hipError_t bounds::launch_key_labels")[0]
        text = text.replace('"gdp_bounds.h"', f'"{_build.CSRC}/gdp_bounds.h"')
        text = text.replace("extern __shared__ __align__(16) char lds[];", "char *const lds = emulated_lds;")
        text = re.sub(r'asm\("v_(min|max)_f64[^;]*;', r"r = std::\1(a, b);", text)
        text = re.sub(r'asm volatile\("ds_add_rtn.*?"memory"\);', "old = *p; *p += n;", text, flags=re.S)
        (where / name).write_text(text)
    so = str(where / "emulated.so")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-ffp-contract=off", "-w", "-shared", "-fPIC", "-I", os.path.join(HERE, "emulation"),
                    f'-DKERNEL="{where}/gdp_key_labels.hip"', os.path.join(HERE, "emulation", "key_labels.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.instance_size.restype = lib.result_size.restype = ctypes.c_size_t
    lib.run_key.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 2 + [ctypes.c_uint, ctypes.c_int]
    assert lib.instance_size() == ctypes.sizeof(Instance) and lib.result_size() == ctypes.sizeof(Out)
    return lib


class Emulated:
    """An instance with its bounds, as the kernels before this one leave them."""
    def __init__(self, lib, x, V, n_lam=64, limit=1e12):
        mem, intra, inter, other_mem, other_time = x
        (L, S), K = mem.shape, len(other_mem)
        least = int(mem.min(1).astype(np.int64).sum())
        budget = np.array([V - 1 - o if V - 1 - o >= least else -1 for o in other_mem], np.int64)
        lam = np.zeros(n_lam)
        base = (intra.max() - intra.min() or 1.0) / max(1.0, float(mem.max() - mem.min()))
        lam[1:] = base * np.exp2(-6.0 + 12.0 * np.arange(n_lam - 1) / (n_lam - 2))
        cost = np.where(mem < V, intra + lam[:, None, None] * mem, FAR)
        P, Q, P_mem, Q_mem = np.zeros((n_lam, L, S)), np.zeros((n_lam, L, S)), np.zeros((n_lam, L, S), np.uint32), np.zeros((n_lam, L, S), np.uint32)
        for l in range(L):
            ways = (P[:, l - 1] if l else np.zeros((n_lam, S)))[:, :, None] + inter[l]
            by = ways.argmin(1)
            P[:, l] = ways.min(1) + cost[:, l]
            P_mem[:, l] = (np.take_along_axis(P_mem[:, l - 1], by, 1) if l else 0) + mem[l].astype(np.uint32)
        for l in range(L - 2, -1, -1):
            ways = inter[l + 1] + (Q[:, l + 1] + cost[:, l + 1])[:, None, :]
            by = ways.argmin(2)
            Q[:, l] = ways.min(2)
            Q_mem[:, l] = np.take_along_axis(Q_mem[:, l + 1] + mem[l + 1].astype(np.uint32), by, 1)
        end = P[:, L - 1].min(1)
        magnitude = float(sum(np.abs(intra[l]).max() + np.abs(inter[l]).max() for l in range(L)))
        margin = 4.0 * (L + 4) * 2.0**-45 * (magnitude + lam * ((L + 1.0) * V))
        ub, best, marks = np.full(K, 2**64 - 1, np.uint64), np.zeros(K, np.int32), np.zeros((K, L, 2), np.uint64)
        for k in range(K):
            if budget[k] < 0:
                continue
            best[k] = np.argmax(end - lam * float(budget[k]))
            first = max(0, min(int(best[k]) - 4, n_lam - 8))
            time_to, time_on = (t[first:first + 8] - lam[first:first + 8, None, None] * m[first:first + 8] for t, m in ((P, P_mem), (Q, Q_mem)))
            fits = P_mem[first:first + 8, None].astype(np.int64) + Q_mem[None, first:first + 8] <= budget[k]
            path = np.where(fits, time_to[:, None] + time_on[None], np.inf).min() + margin[first + 7]
            assert 0 <= path < FAR
            ub[k] = np.float64(path).view(np.uint64) | np.uint64(1 << 63)
            stays = (P + Q - lam[:, None, None] * float(budget[k]) <= path + margin[:, None, None]).all(0)
            for s in range(S):
                marks[k, :, s // 64] |= stays[:, s].astype(np.uint64) << np.uint64(s % 64)
        self.lib, self.L, self.K, self.out, self.res = lib, L, K, Out(), np.full((K, L), -7, np.int32)
        self.arrays = dict(mem=mem, intra=intra, inter_f=inter, index=np.arange(L, dtype=np.int32), lam=lam, budget=budget, P=P, Q=Q, P_mem=P_mem,
                           Q_mem=Q_mem, end=end, best=best, marks=marks, other_time=np.array(other_time, np.float64), res=self.res,
                           hist=np.zeros(16 * K * L * lib.labels_a_layer(), np.uint8))
        self.ub = ub
        self.told = ub.copy()
        self.inst = Instance(**{name: a.ctypes.data for name, a in self.arrays.items()}, ub=self.told.ctypes.data, out=ctypes.addressof(self.out),
                             magnitude=magnitude, limit=limit, L=L, V=V, S=S, K=K, T=L, n_hist=L * lib.labels_a_layer(), n_hist_turns=0, n_lam=n_lam)

    def run(self, key, order=0, seed=1, told_at=-1):
        self.told[:] = self.ub
        self.out.status[key] = -7
        assert self.lib.run_key(ctypes.byref(self.inst), key, order, seed, told_at) == 0
        return self.out.status[key]

    def seen(self):
        found = [ctypes.c_int() for _ in range(3)]
        self.lib.seen(self.L, *map(ctypes.byref, found))
        return [v.value for v in found]

    def check(self, key, want):
        total, res, left = want
        assert np.float64(self.out.total[key]).tobytes() == np.float64(total[key]).tobytes()
        assert self.out.remaining[key] == left[key]
        assert left[key] < 0 or self.res[key].tolist() == [int(v) for v in res[key]]


def _want(x, V):
    keys = range(len(x[3]))
    return O.solve(x[0], x[1], x[2], V, dict(zip(keys, x[3])), dict(zip(keys, x[4])))[:3]


# One wave's labels and all waves' (trade: hundreds, in buckets), runs of layers with one strategy, ties; strategies on both sides of 64, more
# layers than a word of marks; more strategies or transitions than LDS holds at a time (448, 3072).  least: labels of a layer, strategies that
# stay and transitions that some key has.
@pytest.mark.parametrize("kind,L,S,V,n_lam,least", [("each", 2, 2, 60, 64, (1, 2, 2)), ("each", 9, 12, 3000, 64, (2, 9, 9)), ("each", 20, 65, 4000, 64, (2, 20, 20)),
                                                    ("runs", 128, 6, 4000, 64, (1, 128, 128)), ("alike", 30, 24, 5000, 64, (33, 200, 1000)),
                                                    ("trade", 16, 33, 9000, 64, (193, 128, 900)), ("trade", 16, 48, 9000, 128, (65, 64, 300)),
                                                    ("ties", 30, 40, 900, 64, (9, 300, 3073)), ("ties", 50, 40, 1500, 64, (9, 449, 3073))])
@pytest.mark.parametrize("order", [0, 1, 2])
def test_in_any_order_of_waves(lib, kind, L, S, V, n_lam, least, order):
    x = _instance(L, S, V, kind, 4)
    e, want, seen = Emulated(lib, x, V, n_lam), _want(x, V), []
    for key in range(4):
        assert e.run(key, order) == 0
        e.check(key, want)
        seen.append(e.seen())
    assert all(max(most) >= bound for most, bound in zip(zip(*seen), least)), seen


# Another key's workgroup writes into the upper bound of this one between its waves: all of them go by the one or by the other
@pytest.mark.parametrize("order", [0, 1, 2])
def test_told_to_give_up_while_it_begins(lib, order):
    x = _instance(9, 12, 3000, "each", 2)
    e, want = Emulated(lib, x, 3000), _want(x, 3000)
    for told_at in range(9):
        status = e.run(1, order, told_at=told_at)
        assert status in (0, 4) and (told_at > 0 or status == 4)
        if status == 0:
            e.check(1, want)
