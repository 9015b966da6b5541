"""Sweep kernel instances that the faster kernels leave over, and the float
instances of the one-wavefront kernel.

FP64: pending terms where W has more than 256 rows, where W lies in LDS with
more than 64 labels, and complex W with more than 8 terms, against the oracle
with the bars of the tests that they run through.
FP32: W in LDS, at most 64 labels; the bars of the float parity tests (a flip
only at a near tie of margin 1e-3, W to 2e-4 of its largest element, energies to
1e-4), W rebuilt every 40 accepted moves.
"""
import numpy as np
import pytest

import test_gpu_sweep_fp64
import test_gpu_sweep_small
from kagome_systems import first_divergence_is_near_tie, tape, well_conditioned_configs
from test_gpu_complex import complex_system, conditioned
from test_gpu_sweep_fp64 import real_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,n_up,cplx,delay", [
    (14, 294, False, 3), (14, 290, False, 8), (14, 294, False, 12), (8, 96, True, 9), (8, 96, True, 12), (8, 96, True, 16)])
def test_fp64_terms_in_the_general_kernel(oracle_mod, L, n_up, cplx, delay):
    test_gpu_sweep_fp64.test_fp64_pending_terms_tape_parity(oracle_mod, L, n_up, cplx, delay)


@pytest.mark.parametrize("n_up,n_dn,delay", [(65, 60, 2), (60, 65, 8), (63, 66, 12), (65, 62, 16)])
def test_fp64_terms_with_w_in_lds(oracle_mod, n_up, n_dn, delay):
    test_gpu_sweep_small.test_small_cluster_tape_parity(oracle_mod, n_up, n_dn, False, delay)


@pytest.mark.parametrize("L,n_up,cplx,delay", [
    (6, 54, False, 1), (6, 57, False, 4), (6, 54, False, 8), (6, 50, False, 12), (6, 54, False, 16), (4, 27, False, 5),
    (6, 54, True, 1), (4, 24, True, 4), (6, 54, True, 7), (6, 54, True, 12), (6, 54, True, 16)])
def test_fp32_one_wavefront_per_walker(oracle_mod, L, n_up, cplx, delay):
    from kagome_vmc import _native as nat
    ham = complex_system(L) if cplx else real_system(L, n_up)
    nw, n, k = 3, 250, 40
    ku, kd = (conditioned(oracle_mod, ham, nw, 71, max_cond=1e4) if cplx
              else well_conditioned_configs(oracle_mod, 67, nw, ham, max_cond=1e4))
    tu, tb = tape(nw, n, len(ham.nn), 19)
    with nat.DeviceSampler(ham.bonds_array(), ham.U_up, ham.U_down, nw, precision=nat.PREC_FP32, delay=delay,
                           refresh_policy=nat.REFRESH_EVERY_K, refresh_k=k) as ds:
        assert ds.sweep_threads() == 64
        ds.set_configs(ku, kd)
        c1, o1 = ds.sweep(99, tu[:, :99], tb[:, :99], record=True)
        c2, o2 = ds.sweep(n - 99, tu[:, 99:], tb[:, 99:], record=True)
        e, _ = ds.measure()
        kf = ds.get_configs()
        W = [(ds.get_w(w, 0), ds.get_w(w, 1)) for w in range(nw)]
    out = np.concatenate([o1, o2], axis=1)
    assert c1["accepted"] + c2["accepted"] == int((out == 3).sum()) > 0
    same = 0
    for w in range(nw):
        ch = oracle_mod.Chain.start(ham.nn, ham.U_up, ham.U_down, ku[w], kd[w])
        oc, _, _ = oracle_mod.run_chain(ch, n, tape_u=tu[w], tape_bond=tb[w], policy=1, k=k)
        if not np.array_equal(out[w], oc):
            t, m, ok = first_divergence_is_near_tie(oracle_mod, ham, ku[w], kd[w], tu[w], tb[w], out[w], oc,
                                                    policy=1, k=k)
            assert ok, f"walker {w}: decision differs at sweep {t} with margin {m:.3e}"
            continue
        same += 1
        np.testing.assert_array_equal(kf[0][w], ch.kup)
        np.testing.assert_array_equal(kf[1][w], ch.kdn)
        e_or = oracle_mod.getol(ham.nn, ch.kup, ch.kdn, ch.Wup, ch.Wdn)
        assert abs(e[w] - e_or) < 1e-4 * max(1.0, abs(e_or))
        for got, ref in ((W[w][0], ch.Wup), (W[w][1], ch.Wdn)):
            assert np.abs(got - ref).max() < 2e-4 * np.abs(ref).max()
    assert same >= nw - 1
