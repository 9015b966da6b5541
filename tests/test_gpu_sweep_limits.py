"""Handles at the limits of a sweep kernel's LDS run on the kernel that still
takes them: 86 sites with thousands of bonds, whose tables and 16 pending terms
leave k_sweep within 160 KiB and the one-wavefront kernel beyond it."""
import numpy as np
import pytest

from test_gpu_refresh_tiles import configs, gaussian_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [7150, 7200])
def test_small_cluster_with_thousands_of_bonds(nb):
    from kagome_vmc import _native as nat
    _, U_up, U_dn = gaussian_system(43, 43, True, 5)
    rng = np.random.default_rng(9)
    bonds = np.sort(rng.choice(86, (3 * nb, 2)) + 1, axis=1).astype(np.int32)
    bonds = bonds[bonds[:, 0] != bonds[:, 1]][:nb]
    assert len(bonds) == nb
    nw = 3
    ku, kd = configs(bonds, (U_up, U_dn), nw, 3)
    res = []
    for delay in (16, 4):
        with nat.DeviceSampler(bonds, U_up, U_dn, nw, delay=delay, seed=21) as ds:
            ds.set_configs(ku, kd)
            cnt, _ = ds.sweep(120)
            res.append((cnt["moves"], cnt["accepted"], ds.get_configs(), ds.get_w(1, 0), ds.measure()[0]))
    (m0, a0, k0, W0, e0), (m1, a1, k1, W1, e1) = res
    assert (m0, a0) == (m1, a1) and a0 > 0
    np.testing.assert_array_equal(k0, k1)
    assert np.abs(W0 - W1).max() < 1e-9 * np.abs(W1).max()
    np.testing.assert_allclose(e0, e1, rtol=1e-9, atol=1e-6)
