"""Calls that only read a handle, from two threads at once: each gets its own
results (energies and log-determinants come back through separate buffers)."""
import threading

import numpy as np
import pytest

from kagome_systems import system

pytestmark = pytest.mark.gpu


def test_energies_and_log_determinants_from_two_threads():
    from kagome_vmc import _native as nat
    ham, nw = system(4), 8192
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw, seed=3) as ds:
        ds.init_random(3)
        ds.sweep(24)
        e, nap = ds.measure()
        ld = ds.logdet()
        assert not np.array_equal(e, ld)
        wrong = []

        def energies():
            for _ in range(400):
                x, n = ds.measure()
                if n != nap or not np.array_equal(x, e):
                    wrong.append("energies")

        def log_determinants():
            for _ in range(400):
                if not np.array_equal(ds.logdet(), ld):
                    wrong.append("log-determinants")

        ts = [threading.Thread(target=f) for f in (energies, log_determinants, log_determinants)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not wrong, (len(wrong), wrong[:3])
