"""Workgroup sizes of the sweep kernels: fixed for small clusters and for W with
implicit pending rows, the caller's elsewhere; the autotuner times a launch
shape once."""
import pytest

from kagome_systems import system
from test_gpu_complex import complex_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,cplx,prec,delay,asked,runs", [
    (4, False, 1, 8, 256, 64), (6, False, 0, 1, 128, 64), (8, False, 0, 1, 256, 128), (10, False, 1, 8, 64, 192),
    (12, False, 0, 4, 64, 256), (14, False, 0, 1, 512, 512), (8, True, 0, 1, 256, 128), (8, True, 1, 8, 256, 256),
    (8, True, 1, 8, 128, 128),
])
def test_threads_where_the_kernel_leaves_a_choice(L, cplx, prec, delay, asked, runs):
    from kagome_vmc import _native as nat
    ham = complex_system(L) if cplx else system(L)
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, 4, precision=prec, delay=delay,
                           threads=asked) as ds:
        assert ds.sweep_threads() == runs


@pytest.mark.parametrize("L,cplx,prec,launches", [(8, False, 0, 3), (4, False, 1, 3), (8, True, 1, 6)])
def test_autotune_times_a_launch_once(monkeypatch, L, cplx, prec, launches):
    from kagome_vmc import _native as nat
    from kagome_vmc.autotune import autotune, candidates
    ham = complex_system(L) if cplx else system(L)
    starts = []
    init = nat.DeviceSampler.init_random
    monkeypatch.setattr(nat.DeviceSampler, "init_random", lambda self, seed: starts.append(seed) or init(self, seed))
    r = autotune(ham, 16, prec, 64, steps=1, cache_path=None)
    assert [(t["threads"], t["delay"]) for t in r["trials"]] == candidates(ham.ns, prec)
    assert len(starts) == launches
    rates = {}
    for t in r["trials"]:
        rates.setdefault(t["delay"], set()).add(t["walker_sweeps_per_s"])
    assert sum(map(len, rates.values())) <= launches
