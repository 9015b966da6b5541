"""LU of the refresh at the edges of its panels: electron counts around half
panels (16 columns), panels (32), the 64 rows a register of the pivoting
wavefront holds, and the bounds between its instances, with unequal spins, so
that one spin runs far below the instance of the other.  Same systems and bar
as the tile edges of the solve.
"""
import numpy as np
import pytest

from test_gpu_refresh_tiles import check_refresh, gaussian_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n_up,n_dn", [(2, 31), (32, 15), (47, 49), (63, 48), (66, 80), (81, 95), (113, 112), (127, 17),
                                       (130, 145), (159, 162), (191, 3), (194, 207), (223, 226), (242, 239)])
def test_refresh_at_panel_edges(n_up, n_dn, prec):
    check_refresh(n_up, n_dn, False, prec, 3000 + n_up)


@pytest.mark.parametrize("n,col", [(20, 3), (40, 37), (100, 70), (150, 149), (216, 100)])
def test_zero_pivot_is_refused(n, col):
    """A column that is zero on the occupied sites: singular, wherever its panel lies."""
    from kagome_vmc import _native as nat
    bonds, Uu, Ud = gaussian_system(n, n, False, 3500 + n)
    Uu[:n, col] = 0.0
    k = np.zeros((2, 2, 2 * n), dtype=np.int32)
    k[0, :, :n] = k[1, :, n:] = np.arange(1, n + 1)
    with nat.DeviceSampler(bonds, Uu, Ud, 2) as ds:
        with pytest.raises(nat.SingularError):
            ds.set_configs(k[0], k[1])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n_up,n_dn,cplx", [(257, 31, False), (288, 289, False), (320, 321, False),
                                            (385, 352, False), (449, 448, False), (511, 512, False),
                                            (40, 512, False), (513, 500, False), (129, 128, True), (144, 145, True), (160, 161, True),
                                            (225, 3, True), (240, 256, True), (257, 250, True)],
                         ids=lambda x: str(x))
def test_refresh_split_over_two_wavefronts(n_up, n_dn, cplx, prec):
    """257 to 512 labels (twice as many as complex orbitals): edges of its
    32-label blocks and pairs of blocks, a spin far below, and one beyond."""
    check_refresh(n_up, n_dn, cplx, prec, 4000 + n_up)
