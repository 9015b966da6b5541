"""Sweeps of small clusters (W resident in LDS, one wavefront per walker)
against the oracle's immediate updates, at the edges of the kernel's range:
up to 64 labels and rows per spin and 128 sites, more of either beyond it,
unequal spins, each delay instance, real and complex FP64, and bond lists with
uneven numbers of neighbours.  Orbitals are seeded Gaussian matrices.

Bars: decisions identical (those within 1e-12 of a tie excepted), W and local
energies to 1e-9 of their largest element (FP64, condition below 1e5).
"""
import numpy as np
import pytest

from kagome_systems import first_divergence_is_near_tie, tape
from test_gpu_refresh_tiles import configs, gaussian_system

pytestmark = pytest.mark.gpu


class System:
    def __init__(self, n_up, n_dn, cplx, seed):
        _, self.U_up, self.U_down = gaussian_system(n_up, n_dn, cplx, seed)
        self.ns, self.N_up, self.N_down = n_up + n_dn, n_up, n_dn
        rng = np.random.default_rng(seed + 5)
        pairs = {(int(min(p)), int(max(p))) for p in rng.integers(1, self.ns + 1, (2 * self.ns, 2)) if p[0] != p[1]}
        pairs |= {(1, i) for i in range(2, self.ns + 1)}          # one site with a bond to every other
        self.nn = sorted(pairs, key=lambda p: (p[1], p[0]))


@pytest.mark.parametrize("n_up,n_dn,cplx,delay", [
    (64, 64, False, 1), (64, 64, False, 4), (61, 60, False, 8), (64, 58, False, 16), (65, 60, False, 1), (3, 2, False, 1),
    (1, 1, False, 1), (24, 24, False, 5), (33, 40, False, 12), (45, 44, True, 1), (40, 38, True, 12), (20, 24, True, 4),
])
def test_small_cluster_tape_parity(oracle_mod, n_up, n_dn, cplx, delay):
    from kagome_vmc import _native as nat
    ham = System(n_up, n_dn, cplx, 100 + n_up)
    nw, n = 4, 150
    ku, kd = configs(np.array(ham.nn), (ham.U_up, ham.U_down), nw, 3)
    tu, tb = tape(nw, n, len(ham.nn), 7 + n_up)
    with nat.DeviceSampler(np.array(ham.nn, dtype=np.int32), ham.U_up, ham.U_down, nw, delay=delay) as ds:
        ds.set_configs(ku, kd)
        c1, o1 = ds.sweep(70, tu[:, :70], tb[:, :70], record=True)      # leaves terms pending
        c2, o2 = ds.sweep(n - 70, tu[:, 70:], tb[:, 70:], record=True)
        e, nap = ds.measure()
        kf = ds.get_configs()
        W = [(ds.get_w(w, 0), ds.get_w(w, 1)) for w in range(nw)]
    out = np.concatenate([o1, o2], axis=1)
    assert c1["sweeps"] + c2["sweeps"] == nw * n
    assert c1["accepted"] + c2["accepted"] == int((out == 3).sum())
    assert c1["moves"] + c2["moves"] == int((out >= 2).sum())
    zs = 0
    for w in range(nw):
        ch = oracle_mod.Chain.start(ham.nn, ham.U_up, ham.U_down, ku[w], kd[w])
        oc, _, _ = oracle_mod.run_chain(ch, n, tape_u=tu[w], tape_bond=tb[w])
        if not np.array_equal(out[w], oc):
            t, m, _ = first_divergence_is_near_tie(oracle_mod, ham, ku[w], kd[w], tu[w], tb[w], out[w], oc)
            assert m < 1e-12, f"walker {w}: decision differs at sweep {t} with margin {m:.3e}"
            zs = None
            continue
        np.testing.assert_array_equal(kf[0][w], ch.kup)
        np.testing.assert_array_equal(kf[1][w], ch.kdn)
        for got, ref in ((W[w][0], ch.Wup), (W[w][1], ch.Wdn)):
            assert np.abs(got - ref).max() < 1e-9 * np.abs(ref).max()
        e_or = oracle_mod.getol(ham.nn, ch.kup, ch.kdn, ch.Wup, ch.Wdn)
        assert abs(e[w] - e_or) < 1e-9 * max(np.abs(ch.Wup).max() * np.abs(ch.Wdn).max(), abs(e_or))
        if zs is not None:
            zs += oracle_mod.z_count(ham.nn, ch.kup, ch.kdn)
    assert zs is None or nap == zs
