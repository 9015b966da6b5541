"""A handle that fits the GPU with immediate updates is created also where
the pending terms that an FP64 handle keeps for them would no longer fit.  The
rest of the memory is held by tensors; nothing is launched meanwhile but
the fills of kvmc_create."""
import pytest

from kagome_systems import system

pytestmark = pytest.mark.gpu


def test_fp64_handle_without_room_for_its_own_terms():
    import torch
    from kagome_vmc import _native as nat
    ham, nw = system(12), 8192
    args = (ham.bonds_array(), ham.U_up, ham.U_down, nw)
    free = lambda: torch.cuda.mem_get_info()[0]
    with nat.DeviceSampler(*args):
        pass
    torch.cuda.empty_cache()
    before = free()
    with nat.DeviceSampler(*args):
        need = before - free()
    terms = nw * 2 * (12 - 4) * (216 + 216) * 8          # of 12 slots a row instead of 4
    assert terms > 400 << 20
    # the bulk, then steps of half of the terms until a handle that asks
    # for 12 terms no longer fits (the free memory that HIP reports is not exact)
    hold, full = [], False
    try:
        hold.append(torch.empty(free() - need - (1 << 30), dtype=torch.uint8, device="cuda"))
        for _ in range(20):
            try:
                nat.DeviceSampler(*args, delay=12).close()
            except nat.KvmcError as e:
                assert e.code == nat.KVMC_ERR_NOMEM
                full = True
                break
            hold.append(torch.empty(terms // 2, dtype=torch.uint8, device="cuda"))
        if full:
            with nat.DeviceSampler(*args) as ds:
                assert ds.nwalkers == nw
    except torch.cuda.OutOfMemoryError:
        full = False
    finally:
        hold.clear()
        torch.cuda.empty_cache()
    if not full:
        pytest.skip("the memory could not be filled")
    with nat.DeviceSampler(*args) as ds:                  # nothing is left behind
        ds.init_random(1)
        assert ds.sweep(4)[0]["sweeps"] == 4 * nw
