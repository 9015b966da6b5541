"""Local energies while terms of W are pending, against the same walkers with
every term applied to W (get_w applies a walker's): both spins' terms in LDS
or one spin's at a time, workgroups of 256 and of 512 threads, more bonds than
one pass of the workgroup takes (588 sites), unequal fillings.

Bars: FP64 to 1e-9 of the energy (W of condition below 1e6), FP32 to 1e-4 (a
term applied in float rounds each element by 2^-24 of the largest).
"""
import numpy as np
import pytest

from kagome_systems import system, well_conditioned_configs
from test_gpu_complex import complex_system, conditioned
from test_gpu_sweep_fp64 import real_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,n_up,cplx,prec,delay", [
    (4, 24, False, 0, 3), (8, 99, False, 0, 1), (8, 96, False, 0, 16), (12, 216, False, 0, 1), (12, 216, False, 0, 13),
    (14, 294, False, 0, 2), (14, 294, False, 0, 8), (6, 54, True, 0, 4), (8, 96, True, 0, 1), (12, 216, True, 0, 1),
    (8, 96, False, 1, 5), (12, 216, False, 1, 16), (14, 294, False, 1, 12), (12, 216, True, 1, 4), (12, 216, True, 1, 12),
])
def test_energies_with_terms_pending(oracle_mod, L, n_up, cplx, prec, delay):
    from kagome_vmc import _native as nat
    ham = complex_system(L) if cplx else system(L) if 2 * n_up == 3 * L * L else real_system(L, n_up)
    nw = 5
    ku, kd = (conditioned(oracle_mod, ham, nw, 23) if cplx else well_conditioned_configs(oracle_mod, 29, nw, ham))
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw, precision=prec, delay=delay,
                           refresh_policy=nat.REFRESH_EVERY_K, refresh_k=10_000, seed=13) as ds:
        ds.set_configs(ku, kd)
        for n in (7, 40, 41, 42):           # the walkers' terms differ in number
            acc = ds.sweep(n)[0]["accepted"]
            e, nap = ds.measure()
            for w in range(nw):
                ds.get_w(w, 0)
            e0, nap0 = ds.measure()
            assert nap == nap0
            np.testing.assert_allclose(e, e0, rtol=1e-9 if prec == 0 else 1e-4, atol=1e-9)
        assert acc > 0


def test_terms_of_immediate_updates_do_not_slow_energies():
    """A default FP64 handle keeps terms of its own between calls: its
    energies read them once, so that a launch stays within 2.6 times that of
    the same walkers without any (1.6 measured; gathered from memory for every
    bond they took 3.4 to 4 times as long)."""
    from kagome_vmc import _native as nat
    from kagome_vmc.batch import flux_cluster
    ham = flux_cluster(12, 0.3)

    def launch_ms(ds):
        best = np.inf
        for _ in range(5):
            ds.profile(True)
            for _ in range(10):
                ds.measure()
            p = ds.profile()
            best = min(best, p["measure_ms"] / p["measure_launches"])
        ds.profile(False)
        return best

    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, 512, seed=3) as ds:
        ds.init_random(3)
        ds.sweep(216)
        pending = launch_ms(ds)
        ds.refresh()
        assert pending < 2.6 * launch_ms(ds)
