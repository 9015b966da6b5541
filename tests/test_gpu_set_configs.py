"""Configurations are checked on the device: each kind of wrong one is refused
with the first wrong walker and the reason, and leaves the handle as it was."""
import numpy as np
import pytest

from kagome_systems import system, well_conditioned_configs

pytestmark = pytest.mark.gpu


def doubly(ku, kd, w):
    kd[w, np.flatnonzero(ku[w])[0]] = 1


def empty(ku, kd, w):
    ku[w, np.flatnonzero(ku[w])[0]] = 0


def repeated(ku, kd, w):
    s = np.flatnonzero(ku[w])
    ku[w, s[0]] = ku[w, s[1]]


def too_large(ku, kd, w):
    kd[w, np.flatnonzero(kd[w])[0]] = 25


def negative(ku, kd, w):
    kd[w, np.flatnonzero(kd[w])[3]] = -2


@pytest.mark.parametrize("spoil,text", [(doubly, "doubly occupied"), (empty, "unoccupied"), (repeated, "repeated up label"),
                                        (too_large, "out of bounds"), (negative, "out of bounds")])
@pytest.mark.parametrize("at", [0, 16, 66])
def test_wrong_configurations_are_refused(oracle_mod, spoil, text, at):
    from kagome_vmc import _native as nat
    ham = system(4)
    nw = 67
    ku, kd = well_conditioned_configs(oracle_mod, 5, nw, ham)
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw) as ds:
        ds.set_configs(ku, kd)
        e0, _ = ds.measure()
        bu, bd = ku[::-1].copy(), kd[::-1].copy()
        for w in {at, nw - 1}:
            spoil(bu, bd, w)
        with pytest.raises(nat.KvmcError, match=f"walker {at}: .*{text}"):
            ds.set_configs(bu, bd)
        got = ds.get_configs()
        assert np.array_equal(got[0], ku) and np.array_equal(got[1], kd)
        assert np.array_equal(ds.measure()[0], e0)
        ds.sweep(30)        # and it still runs
