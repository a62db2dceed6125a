"""z of the hyperpriors coded without a wait before ``h_s`` and y: z_hat as the
encode kernel writes it, and whose error is raised when z and y both fail."""

import numpy as np
import pytest
import torch

import fast_compressai
import oracle as O
from fast_compressai import synthetic
from fast_compressai.coders import CoderInputError, WarpDivPayload, gaans
from fast_compressai.coders.tables import prepare_tables
from hyperprior_stub import make_hyperprior

pytestmark = pytest.mark.gpu


# one lane; less than a step; whole steps; a ragged last step; 16-step blocks
# (12 units) and a chunk of several units.  Every 7th value lies outside its
# table (an escape), the last one far outside.
@pytest.mark.parametrize("shape,p_ch,segments", [
    ((1, 1, 1, 1), 1, 1), ((2, 3, 5, 7), 2, 1), ((1, 8, 8, 16), 4, 1), ((3, 6, 11, 13), 5, 2),
    ((1, 24, 32, 48), 16, 1)])
@pytest.mark.parametrize("escapes", [False, True])
def test_encode_writes_the_dequantized_latents(gpu_device, shape, p_ch, segments, escapes):
    B, C, H, W = shape
    print("case:", shape, p_ch, segments, escapes, flush=True)
    w = synthetic._factorized("z", B, C, H, W, 0.1, 8, 64, p_ch, (1, 1), 3)
    rng = np.random.default_rng(5)
    med = rng.normal(0, 1, C).astype(np.float32)
    y = (w.symbols.reshape(B, C, -1) + med[None, :, None]
         + rng.uniform(-0.49, 0.49, (B, C, H * W))).astype(np.float32)
    if escapes:
        y.reshape(-1)[::7] += 4000.0
        y.reshape(-1)[-1] = -3000000.0
    tables = prepare_tables(*(torch.from_numpy(a).to(gpu_device)
                              for a in (w.cdfs, w.cdf_sizes, w.offsets)))
    y_dev, med_dev = (torch.from_numpy(a).to(gpu_device) for a in (y, med))
    want = torch.round(y_dev - med_dev[None, :, None]).int().float() + med_dev[None, :, None]
    y_hat = torch.full((B, C * H * W), float("nan"), device=gpu_device)
    enc = gaans.encode_latents_begin(tables, B, C * H * W, C, p_ch, gpu_device, y=y_dev,
                                     medians=med_dev, y_hat=y_hat, segments=segments).finish()
    assert torch.equal(y_hat.reshape(want.shape), want)
    sym = np.rint(y - med[None, :, None]).astype(np.int64).astype(np.int32).reshape(B, -1)
    ref = O.gaans_encode(sym, w.indexes, w.cdfs, w.cdf_sizes, w.offsets, p_ch, None, segments)
    assert enc.packed.cpu().numpy().tobytes() == ref


@pytest.mark.parametrize("h_s_fails", [False, True])
def test_error_of_z_is_raised_first(gpu_device, h_s_fails):
    model = make_hyperprior(mean_scale=True).to(gpu_device)
    x = torch.rand(1, 3, 64, 64, device=gpu_device)
    fast = fast_compressai.accelerate(model, P=4, device=str(gpu_device))
    out = fast.compress(x)
    good = fast.decompress(out["strings"], out["shape"])["x_hat"]
    y_payload, z_payload = out["strings"]
    blob = bytearray(z_payload.to_bytes())
    blob[-1] ^= 0x55  # the last unit's words: its final state no longer fits
    bad = WarpDivPayload._from_encoder(
        packed=torch.frombuffer(blob, dtype=torch.uint8).to(gpu_device),
        header_bytes=z_payload.header_bytes, chunk_len=z_payload.chunk_len,
        p_ch=z_payload.p_ch, batch=z_payload.batch,
        symbols_per_batch=z_payload.symbols_per_batch, cdf_count=z_payload.cdf_count,
        coding_fingerprint=z_payload.coding_fingerprint, channels=z_payload.channels,
        segments=z_payload.segments)
    codec = fast._coder
    latents = codec.analyze(x)
    nan_z = (latents[0], torch.full_like(latents[1], float("nan")))
    params = codec._params
    if h_s_fails:
        def fail(z_hat):
            raise RuntimeError("h_s")
        codec._params = fail
        with pytest.raises(RuntimeError, match="h_s"):
            codec.encode_latents(latents)
    print("case: z fails", h_s_fails, flush=True)
    with pytest.raises(CoderInputError):
        fast.decompress([y_payload, bad], out["shape"])
    with pytest.raises(CoderInputError):
        codec.encode_latents(nan_z)
    codec._params = params
    again = fast.compress(x)["strings"]
    assert [p.to_bytes() for p in again] == [p.to_bytes() for p in out["strings"]]
    assert torch.equal(fast.decompress(out["strings"], out["shape"])["x_hat"], good)


def test_calls_in_and_out_of_inference_mode(gpu_device):
    model = make_hyperprior(mean_scale=True).to(gpu_device)
    codec = fast_compressai.accelerate(model, P=4, device=str(gpu_device))._coder
    x = torch.rand(1, 3, 64, 64, device=gpu_device)
    # the first call makes this stream's words
    gaans._state(0, torch.cuda.current_stream(gpu_device).cuda_stream).slots.clear()
    got = []
    for mode in (True, False, True):
        with torch.inference_mode(mode), torch.no_grad():
            out = codec.encode_latents(codec.analyze(x))
            y_hat = codec.decode_latents(out["strings"], out["shape"])
            got.append([p.to_bytes() for p in out["strings"]] + [y_hat.cpu().numpy().tobytes()])
    assert got[0] == got[1] == got[2]
