"""The coder's step groups at their edges: 16- and 8-step blocks, what is left
over after them (groups of 4 and of 1, a last step with idle lanes), units of
256 and more steps, tables that need a second look-up in most steps, tables
that need almost no stream words, escapes in every group, and more workgroups
than the chip has CUs.  Payload bytes against the oracle, symbols against the
input."""

import numpy as np
import pytest
import torch

import oracle as O
from fast_compressai import synthetic
from fast_compressai.coders import gaans
from fast_compressai.coders.tables import prepare_tables
from hyperprior_stub import gaussian_tables

pytestmark = pytest.mark.gpu


def pmf(kind):
    if kind == "skew":
        return synthetic.laplace_pmf(2.0, 30)
    if kind == "dense":  # 254 equal values: nearly every bucket holds a boundary
        return np.full(254, 1.0 / 254), 1e-9
    return synthetic.laplace_pmf(0.05, 3)  # "low": a few hundredths of a bit per symbol


# symbols per channel: one lane; a step less one; 1, 3, 4, 5 steps; blocks of 8
# and 16 with 0, 1, 3, 4 and 7 steps left over, with whole and ragged last
# steps; 257 steps (the encoder's 16-step blocks for long units)
LENGTHS = [1, 63, 64, 192, 256, 300, 512, 1024, 1025, 16 * 64 + 192, 20 * 64, 23 * 64 - 5,
           33 * 64 + 1, 257 * 64 - 31]


@pytest.mark.parametrize("kind", ["skew", "dense", "low"])
@pytest.mark.parametrize("escapes", [0.0, 0.02])
@pytest.mark.parametrize("explicit", [False, True])
def test_step_groups_match_oracle(gpu_device, kind, escapes, explicit):
    rng = np.random.default_rng(11)
    p, tail = pmf(kind)
    C = 2
    cdfs, sizes, offsets = synthetic.build_tables([(p, tail)] * C)
    offsets[:] = -(len(p) // 2)
    tables = prepare_tables(*(torch.from_numpy(a).to(gpu_device)
                              for a in (cdfs, sizes, offsets)))
    for n in LENGTHS:
        print("case:", kind, escapes, explicit, n, flush=True)
        sym = rng.choice(len(p), size=(1, C * n), p=p / p.sum()).astype(np.int32) + offsets[0]
        hit = rng.random(sym.shape) < escapes
        hit[0, -1] = escapes > 0
        sym = np.where(hit, sym + rng.choice([-70000, 900], sym.shape), sym).astype(np.int32)
        idx = np.repeat(np.arange(C, dtype=np.int32), n)[None]
        if explicit:
            idx = rng.integers(0, C, (1, C * n)).astype(np.int32)
        for segments in (1, 2) if n > 64 else (1,):
            d, i = torch.from_numpy(sym).to(gpu_device), torch.from_numpy(idx).to(gpu_device)
            i = i if explicit else None
            enc = gaans.encode(tables, 1, C * n, C, 1, gpu_device, symbols=d, indexes=i,
                               segments=segments)
            ref = O.gaans_encode(sym, idx, cdfs, sizes, offsets, 1, C, segments)
            assert enc.packed.cpu().numpy().tobytes() == ref
            out = gaans.decode(enc.packed, tables, 1, C * n, C, 1, gpu_device, indexes=i,
                               segments=segments)
            assert torch.equal(out, d)


@pytest.mark.parametrize("n", [1, 70, 256, 1024 + 65, 19 * 64, 259 * 64 - 7])
def test_gaussian_step_groups_match_oracle(gpu_device, n):
    rng = np.random.default_rng(n)
    table, cdfs, sizes, offsets = gaussian_tables()
    scales = np.exp(rng.uniform(np.log(0.05), np.log(300.0), (1, 3 * n))).astype(np.float32)
    y = (rng.standard_normal((1, 3 * n)) * scales * 2).astype(np.float32)
    print("case: gaussian", n, flush=True)
    idx, sym = O.build_indexes(scales, table, 0.11), O.quantize_elem(y)
    t = prepare_tables(*(torch.from_numpy(a).to(gpu_device) for a in (cdfs, sizes, offsets)))
    y_d, s_d, tab = (torch.from_numpy(a).to(gpu_device) for a in (y, scales, table))
    enc = gaans.encode_gaussian(t, 1, 3 * n, 3, 1, gpu_device, y=y_d, scales=s_d,
                                scale_table=tab, scale_bound=0.11)
    ref = O.gaans_encode(sym, idx, cdfs, sizes, offsets, 1, 3, 1)
    assert enc.packed.cpu().numpy().tobytes() == ref
    out = gaans.decode_gaussian(enc.packed, t, 1, 3 * n, 3, 1, gpu_device, scales=s_d,
                                scale_table=tab, scale_bound=0.11)
    assert torch.equal(out, torch.from_numpy(O.dequantize_elem(sym)).to(gpu_device))


def test_more_workgroups_than_cus_match_oracle(gpu_device):
    w = synthetic._factorized("many", 40, 24, 9, 19, 0.1, 32, 256, 1, (1, 1), 2)
    print("case: 960 units of 3 steps", flush=True)
    t = prepare_tables(*(torch.from_numpy(a).to(gpu_device)
                         for a in (w.cdfs, w.cdf_sizes, w.offsets)))
    d = torch.from_numpy(w.symbols).to(gpu_device)
    B, N = w.symbols.shape
    enc = gaans.encode(t, B, N, 24, 1, gpu_device, symbols=d)
    ref = O.gaans_encode(w.symbols, w.indexes, w.cdfs, w.cdf_sizes, w.offsets, 1, None, 1)
    assert enc.packed.cpu().numpy().tobytes() == ref
    assert torch.equal(gaans.decode(enc.packed, t, B, N, 24, 1, gpu_device), d)
