"""Reads and writes of W that a sweep call reports (kvmc_get_w_passes), from
which byte rates are formed: the flushes of pending terms, whether the terms
were asked for or an FP64 handle keeps them for immediate updates."""
import os
import sys

import pytest

from kagome_systems import system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,prec,delay,held", [(8, 0, 1, 8), (12, 0, 1, 12), (14, 0, 1, 1), (8, 0, 4, 4), (8, 1, 12, 12)])
def test_passes_are_those_of_the_terms_held(L, prec, delay, held):
    from kagome_vmc import _native as nat
    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    import bench
    ham, nw = system(L), 16
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw, precision=prec, delay=delay, seed=8,
                           refresh_policy=nat.REFRESH_EVERY_K, refresh_k=100_000) as ds:
        ds.init_random(8)
        for _ in range(3):                  # random starts can be nearly singular: those update W at once
            ds.sweep(8)
            ds.refresh()
        cnt, _ = ds.sweep(3 * L * L)
        cnt["w_passes"] = ds.w_passes()
        assert cnt["flushes"] == (cnt["accepted"] if delay == 1 else cnt["w_passes"])
        # a walker's moves since the refresh: whole groups of `held` have been applied
        assert cnt["accepted"] - nw * (held - 1) <= held * cnt["w_passes"] <= cnt["accepted"]
        s, n = (8, 4)[prec], 3 * L * L // 2
        moved = cnt["w_passes"] * 2 * s * 2 * n * n
        rest = bench.sweep_bytes(cnt, s, ham.ns, n, n, nw) - moved
        assert rest == bench.sweep_bytes(dict(cnt, w_passes=0), s, ham.ns, n, n, nw) > 0
        ds.sweep(0)
        assert ds.w_passes() == cnt["w_passes"]   # nothing was swept
