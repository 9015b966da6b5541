"""FP64 sweeps through pending terms (W streamed from HBM, at most 256 rows)
against the oracle's immediate updates, at the edges of the kernel's ranges:
columns of 56 to 220 rows (one, two and four 16-byte units per lane; one to
four wavefronts per walker), each delay instance and one between two, real and
complex W, and walkers whose last refresh found pivots over more than 1e7
(these update W at once).

Bars: decisions identical (those within 1e-12 of a tie excepted), W and local
energies to 1e-9: 300 updates of a W whose condition is below 1e6 in FP64.
"""
import numpy as np
import pytest

from kagome_systems import BC, first_divergence_is_near_tie, tape, well_conditioned_configs
from test_gpu_complex import conditioned, complex_system

pytestmark = pytest.mark.gpu
_CACHE = {}


def real_system(L, n_up):
    from kagome_vmc import DoubleKagome, Hamiltonian
    key = (L, n_up)
    if key not in _CACHE:
        pbc, apbc = BC[L]
        _CACHE[key] = Hamiltonian.build(n_up, 3 * L * L - n_up, DoubleKagome.build(1.0, L, L, pbc, apbc))
    return _CACHE[key]


def check_chain(oracle_mod, ham, ku, kd, tu, tb, out, kf, W, e):
    moved = 0
    for w in range(len(ku)):
        ch = oracle_mod.Chain.start(ham.nn, ham.U_up, ham.U_down, ku[w], kd[w])
        oc, _, _ = oracle_mod.run_chain(ch, tu.shape[1], tape_u=tu[w], tape_bond=tb[w])
        if not np.array_equal(out[w], oc):
            t, m, _ = first_divergence_is_near_tie(oracle_mod, ham, ku[w], kd[w], tu[w], tb[w], out[w], oc)
            assert m < 1e-12, f"walker {w}: decision differs at sweep {t} with margin {m:.3e}"
            continue
        moved += int((out[w] == 3).sum())
        np.testing.assert_array_equal(kf[0][w], ch.kup)
        np.testing.assert_array_equal(kf[1][w], ch.kdn)
        for got, ref in ((W[w][0], ch.Wup), (W[w][1], ch.Wdn)):
            assert np.abs(got - ref).max() < 1e-9 * np.abs(ref).max()
        e_or = oracle_mod.getol(ham.nn, ch.kup, ch.kdn, ch.Wup, ch.Wdn)
        assert abs(e[w] - e_or) < 1e-9 * max(1.0, abs(e_or))
    assert moved > 0


@pytest.mark.parametrize("L,n_up,cplx,delay", [
    (8, 96, False, 1), (8, 99, False, 4), (8, 96, False, 5), (8, 96, False, 12), (8, 96, False, 16),
    (10, 150, False, 1), (10, 152, False, 10),
    (12, 216, False, 1), (12, 219, False, 1), (12, 216, False, 4), (12, 216, False, 16),
    (6, 54, True, 1), (6, 54, True, 4), (8, 96, True, 1), (8, 96, True, 3), (10, 150, True, 1), (12, 216, True, 4),
])
def test_fp64_pending_terms_tape_parity(oracle_mod, L, n_up, cplx, delay):
    from kagome_vmc import _native as nat
    ham = complex_system(L) if cplx else real_system(L, n_up)
    nw, n = 3, 200
    ku, kd = (conditioned(oracle_mod, ham, nw, 31) if cplx
              else well_conditioned_configs(oracle_mod, 83, nw, ham))
    tu, tb = tape(nw, n, len(ham.nn), 41 + L)
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw, delay=delay) as ds:
        ds.set_configs(ku, kd)
        c1, o1 = ds.sweep(77, tu[:, :77], tb[:, :77], record=True)      # leaves terms pending
        c2, o2 = ds.sweep(n - 77, tu[:, 77:], tb[:, 77:], record=True)
        e, _ = ds.measure()
        kf = ds.get_configs()
        W = [(ds.get_w(w, 0), ds.get_w(w, 1)) for w in range(nw)]
    out = np.concatenate([o1, o2], axis=1)
    acc = int((out == 3).sum())
    assert c1["accepted"] + c2["accepted"] == acc and c1["sweeps"] + c2["sweeps"] == nw * n
    if delay == 1:   # every accepted move counts as an update of W
        assert c1["flushes"] + c2["flushes"] == acc
    check_chain(oracle_mod, ham, ku, kd, tu, tb, out, kf, W, e)


@pytest.mark.parametrize("L,cplx", [(8, False), (12, False), (8, True)])
def test_fp64_walkers_with_spread_pivots_update_at_once(oracle_mod, L, cplx):
    """W does not change when a column of U is scaled, but the pivots of its
    LU do: a last column 1e-9 times the others takes every walker through the
    immediate update."""
    from kagome_vmc import _native as nat
    ham = complex_system(L) if cplx else real_system(L, 3 * L * L // 2)
    nw, n = 3, 200
    ku, kd = (conditioned(oracle_mod, ham, nw, 57) if cplx
              else well_conditioned_configs(oracle_mod, 57, nw, ham))
    tu, tb = tape(nw, n, len(ham.nn), 5)
    scale = np.ones(ham.N_up)
    scale[-1] = 1e-9
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up * scale, ham.U_down * scale, nw) as ds:
        ds.set_configs(ku, kd)
        _, out = ds.sweep(n, tu, tb, record=True)
        e, _ = ds.measure()
        kf = ds.get_configs()
        W = [(ds.get_w(w, 0), ds.get_w(w, 1)) for w in range(nw)]
    check_chain(oracle_mod, ham, ku, kd, tu, tb, out, kf, W, e)


@pytest.mark.parametrize("kernel", [0, 1])
def test_windows_longer_than_the_draws_held(kernel):
    """One call of many sweeps against the same sweeps one to seven at a time
    (calls end inside the 64 draws a wavefront holds): the same chains."""
    from kagome_vmc import _native as nat
    ham = real_system(8, 96)
    res = []
    for parts in ([700], [7] * 100, [1] * 20 + [63, 64, 65, 128, 360]):
        with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, 16, kernel=kernel, seed=9) as ds:
            ds.init_random(4)
            tot = 0
            for p in parts:
                tot += ds.sweep(p)[0]["moves"]
            res.append((tot, ds.get_configs(), ds.measure()[0]))
    for tot, kap, e in res[1:]:
        assert tot == res[0][0]
        np.testing.assert_array_equal(kap[0], res[0][1][0])
        np.testing.assert_array_equal(kap[1], res[0][1][1])
        np.testing.assert_allclose(e, res[0][2], rtol=1e-8)
