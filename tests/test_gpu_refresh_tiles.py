"""W refresh at the edges of its instances: electron counts at, below and
above each number of 16-label tiles and 32-column panels, with unequal spins.
Orbitals are seeded Gaussian matrices (any U is a valid orbital matrix to the
library), so every size is well conditioned; W against numpy in 64 bits.

Bar: errors of an LU solve grow with the condition of tildeU (below 1e5 here)
in units of 1.1e-16, so 1e-9 relative to the largest element.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def gaussian_system(n_up, n_dn, cplx, seed):
    rng = np.random.default_rng(seed)
    ns = n_up + n_dn

    def orb(n):
        u = rng.standard_normal((ns, n))
        return u + 1j * rng.standard_normal((ns, n)) if cplx else u

    bonds = np.array([(i, i + 1) for i in range(1, ns)], dtype=np.int32)
    return bonds, orb(n_up), orb(n_dn)


def configs(bonds, U, nw, seed, max_cond=1e5):
    rng = np.random.default_rng(seed)
    ns, n_up = U[0].shape
    ku = np.zeros((nw, ns), dtype=np.int32)
    kd = np.zeros((nw, ns), dtype=np.int32)
    w = 0
    while w < nw:
        p = rng.permutation(ns)
        if max(np.linalg.cond(U[0][p[:n_up]]), np.linalg.cond(U[1][p[n_up:]])) > max_cond:
            continue
        ku[w, p[:n_up]] = np.arange(1, n_up + 1)
        kd[w, p[n_up:]] = np.arange(1, ns - n_up + 1)
        w += 1
    return ku, kd


def check_refresh(n_up, n_dn, cplx, prec, seed):
    from kagome_vmc import _native as nat
    bonds, *U = gaussian_system(n_up, n_dn, cplx, seed)
    nw = 5
    ku, kd = configs(bonds, U, nw, seed + 1)
    with nat.DeviceSampler(bonds, *U, nw, precision=prec) as ds:
        ds.set_configs(ku, kd)
        logdet = ds.logdet()
        W = [[ds.get_w(w, s) for s in (0, 1)] for w in range(nw)]
        drift = ds.w_drift()
    tol = 1e-9 if prec == 0 else 1e-6
    assert drift < tol
    for w in range(nw):
        ld = 0.0
        for s, k in ((0, ku[w]), (1, kd[w])):
            order = np.argsort(np.where(k > 0, k, 1 << 20), kind="stable")[: U[s].shape[1]]
            t = U[s][order]
            ref = np.linalg.solve(t.T, U[s].T).T
            assert np.abs(W[w][s] - ref).max() < tol * np.abs(ref).max()
            ld += np.linalg.slogdet(t)[1]
        assert abs(logdet[w] - ld) < 1e-9 * max(1.0, abs(ld))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n_up,n_dn", [(1, 1), (16, 15), (17, 32), (33, 31), (64, 65), (96, 97), (100, 129), (128, 5),
                                       (160, 161), (176, 193), (208, 209), (225, 224), (241, 255), (256, 257)])
def test_refresh_at_tile_edges(n_up, n_dn, prec):
    check_refresh(n_up, n_dn, False, prec, 1000 + n_up)
