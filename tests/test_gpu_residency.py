"""Encode launches whose units are numbered by workgroup: the whole grid is
resident at once, by registers as well as by LDS, for every kernel a plan may
choose."""

import ctypes

import numpy as np
import pytest
import torch

import oracle as O
from fast_compressai import synthetic
from fast_compressai.coders import _native, gaans
from fast_compressai.coders.tables import prepare_tables

pytestmark = pytest.mark.gpu


def small_tables(C, device):
    cdfs, sizes, offsets = synthetic.build_tables([synthetic.laplace_pmf(2.0, 30)] * C)
    offsets[:] = -30
    return (cdfs, sizes, offsets), prepare_tables(
        *(torch.from_numpy(a).to(device) for a in (cdfs, sizes, offsets)))


# units of a few steps (8-step blocks, or 4-step ones) and of 258 (16-step
# blocks), one to four workgroups per CU and more than the device holds
@pytest.mark.parametrize("mode,explicit", [
    (_native.MODE_SYMBOLS, False), (_native.MODE_SYMBOLS, True), (_native.MODE_LATENTS, False),
    (_native.MODE_LATENTS, True), (_native.MODE_GAUSSIAN, True)])
def test_grids_without_tickets_are_resident(gpu_device, mode, explicit):
    C, index = 32, gaans._index(gpu_device)
    _, tables = small_tables(C, gpu_device)
    tickets = set()
    for n in (19 * 64, 128 * 129):
        for B in (1, 8, 9, 16, 17, 24, 25, 32, 40, 200):
            print("case:", mode, explicit, n, B * C, flush=True)
            _, plan, _ = gaans._plan(tables, False, mode, explicit, B, C * n, C, 1, 1, index,
                                     *((64, 0.11) if mode == _native.MODE_GAUSSIAN else ()))
            out = (ctypes.c_int64 * 3)()
            _native.check(_native.lib().gaans_debug_plan(plan, out), "debug plan")
            assert out[0] == B * C and out[1] >= 256
            assert out[2] == 1 or out[0] <= out[1], list(out)
            tickets.add(out[2])
    assert tickets == {0, 1}


# more than 256 units of 258 steps, the last step ragged: 16-step blocks with four
# mappers; explicit indexes at 960 units also reach the register limit
@pytest.mark.parametrize("B,explicit", [(10, False), (10, True), (30, True)])
def test_long_latent_units_match_oracle(gpu_device, B, explicit):
    C, n, index = 32, 128 * 129 - 5, gaans._index(gpu_device)
    print("case: long latent units", B, explicit, flush=True)
    (cdfs, sizes, offsets), tables = small_tables(C, gpu_device)
    rng = np.random.default_rng(B)
    med = rng.normal(0, 1, C).astype(np.float32)
    sym = np.rint(rng.laplace(0, 2.0, (B, C * n))).astype(np.int32)
    sym[:, ::1001] = 4000
    y = torch.from_numpy(sym).to(gpu_device).float() + torch.from_numpy(med).to(
        gpu_device).repeat_interleave(n)
    med_d = torch.from_numpy(med).to(gpu_device)
    want = torch.round(y - med_d.repeat_interleave(n)).int()
    idx = np.tile(np.repeat(np.arange(C, dtype=np.int32), n), (B, 1))
    if explicit:
        idx = np.roll(idx, 77, axis=1)
        enc = gaans.encode(tables, B, C * n, C, 1, gpu_device, y=y, medians=med_d,
                           indexes=torch.from_numpy(idx).to(gpu_device))
    else:
        y_hat = torch.full((B, C * n), float("nan"), device=gpu_device)
        enc = gaans.encode_latents_begin(tables, B, C * n, C, 1, gpu_device, y=y, medians=med_d,
                                         y_hat=y_hat).finish()
        assert torch.equal(y_hat, want.float() + med_d.repeat_interleave(n))
    ref = O.gaans_encode(want.cpu().numpy(), idx, cdfs, sizes, offsets, 1, C, 1)
    assert enc.packed.cpu().numpy().tobytes() == ref
