"""Orbital derivatives summed site by site: one to four parameters (an instance
each) and five (the general kernel), site counts around the 192 sites a
wavefront has under way, walkers short of a full workgroup; against
O_k = sum_s tr(dU tildeU^-1) in numpy at 64 bits.

Orbitals with orthonormal columns, as eigenvectors have, so that the sums over
sites, O_k = sum W Q with Q = dU U^H, are that trace.  Bar: the error of W in
the refresh tests, 1e-9 (1e-6 for single precision) of its largest element,
times the sum of the magnitudes of Q.
"""
import numpy as np
import pytest

from test_gpu_refresh_tiles import configs, gaussian_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n_up,n_dn,nparams", [(3, 4, 1), (32, 31, 2), (33, 32, 3), (96, 95, 4), (97, 96, 1), (70, 123, 4),
                                               (96, 96, 3), (20, 173, 5)])
def test_sums_by_site(n_up, n_dn, nparams, prec, cplx):
    from kagome_vmc import _native as nat
    bonds, *U = gaussian_system(n_up, n_dn, cplx, 5000 + n_up)
    U = [np.linalg.qr(u)[0] for u in U]
    rng = np.random.default_rng(5100 + n_up)
    ns, nw = n_up + n_dn, 5
    dU = [rng.standard_normal((nparams, ns, n)) + (1j * rng.standard_normal((nparams, ns, n)) if cplx else 0.0)
          for n in (n_up, n_dn)]
    ku, kd = configs(bonds, U, nw, 5200 + n_up)
    with nat.DeviceSampler(bonds, *U, nw, precision=prec) as ds:
        ds.set_orbital_derivs(*[[np.asfortranarray(x) for x in d] for d in dU])
        ds.set_configs(ku, kd)
        _, O = ds.measure_grad()
    O = np.asarray(O)
    tol = 1e-9 if prec == 0 else 1e-6
    for w in range(nw):
        ref, scale = np.zeros(nparams, dtype=U[0].dtype), np.zeros(nparams)
        for u, d, k in ((U[0], dU[0], ku[w]), (U[1], dU[1], kd[w])):
            order = np.argsort(np.where(k > 0, k, 1 << 20), kind="stable")[: u.shape[1]]
            inv = np.linalg.inv(u[order])
            ref += (d[:, order, :] * inv.T[None]).sum(axis=(1, 2))
            scale += np.abs(u @ inv).max() * np.abs(d[:, order, :] @ u.conj().T).sum(axis=(1, 2))
        assert (np.abs(O[w] - ref) < tol * scale).all()
