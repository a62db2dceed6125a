"""z of the hyperpriors coded without a wait before ``h_s`` and y: z_hat as the
encode kernel writes it, and whose error is raised when z and y both fail."""

import threading

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


# one lane; less than a step; whole steps; a ragged last step in chunks of two
# units; 16-step blocks (2 units of 384 and 192 steps).  Every 7th value lies outside its
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


def test_strided_z(gpu_device):
    model = make_hyperprior(mean_scale=True).to(gpu_device)
    codec = fast_compressai.accelerate(model, P=4, device=str(gpu_device))._coder
    z = torch.randn(2, 8, 5, 7, device=gpu_device) * 3
    print("case: strided z", flush=True)
    with torch.no_grad():
        finish, z_hat = codec._z_encode(z)
        finish_s, z_hat_s = codec._z_encode(z.contiguous(memory_format=torch.channels_last))
    assert finish().to_bytes() == finish_s().to_bytes()
    assert torch.equal(z_hat, z_hat_s) and z_hat_s.stride() != z_hat.stride()


def changed(payload, at, device):
    blob = bytearray(payload.to_bytes())
    blob[at] ^= 0x55
    return WarpDivPayload._from_encoder(
        packed=torch.frombuffer(blob, dtype=torch.uint8).to(device),
        header_bytes=payload.header_bytes, chunk_len=payload.chunk_len,
        p_ch=payload.p_ch, batch=payload.batch,
        symbols_per_batch=payload.symbols_per_batch, cdf_count=payload.cdf_count,
        coding_fingerprint=payload.coding_fingerprint, channels=payload.channels,
        segments=payload.segments)


def error_of(call, kind=CoderInputError):
    with pytest.raises(kind) as e:
        call()
    return str(e.value)


# what fails besides z: nothing of its own (y sees the z_hat of a failed z), h_s,
# or y with another error than z's
@pytest.mark.parametrize("also", ["nothing", "h_s", "y"])
def test_error_of_z_is_raised_first(gpu_device, also):
    model = make_hyperprior(mean_scale=True).to(gpu_device)
    x = torch.rand(1, 3, 64, 64, device=gpu_device)
    fast = fast_compressai.accelerate(model, P=4, device=str(gpu_device))
    out = fast.compress(x)
    shape = out["shape"]
    good = fast.decompress(out["strings"], shape)["x_hat"]
    y_payload, z_payload = out["strings"]
    # the last unit's words: its final state no longer fits
    bad_z = changed(z_payload, -1, gpu_device)
    codec = fast._coder
    latents = codec.analyze(x)
    nan_z = torch.full_like(latents[1], float("nan"))
    z_decode = error_of(lambda: codec._z_decode(bad_z, shape)[0]())
    z_encode = error_of(lambda: codec._z_encode(nan_z)[0]())
    params, p_ch = codec._params, codec.p_ch
    y = y_payload
    print("case: z fails, and", also, flush=True)
    if also == "h_s":
        def fail(z_hat):
            raise RuntimeError("h_s")
        codec._params = fail
        assert error_of(lambda: codec.encode_latents(latents), RuntimeError) == "h_s"
    elif also == "y":
        y = changed(y_payload, 0, gpu_device)  # the header's magic number
        assert error_of(lambda: fast.decompress([y, z_payload], shape)) != z_decode
    assert error_of(lambda: codec.decode_latents([y, bad_z], shape)) == z_decode
    if also == "y":
        codec.p_ch = latents[0].size(1) + 1  # z's is at most its own channel count
        assert error_of(lambda: codec.encode_latents(latents)) != z_encode
    assert error_of(lambda: codec.encode_latents((latents[0], nan_z))) == z_encode
    codec._params, codec.p_ch = params, p_ch
    again = fast.compress(x)["strings"]
    assert [p.to_bytes() for p in again] == [p.to_bytes() for p in out["strings"]]
    assert torch.equal(fast.decompress(out["strings"], shape)["x_hat"], good)


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


# two host threads on the default stream and two on streams of their own, z of
# each in flight while its y, or another thread's z, is enqueued
def test_threads_and_streams(gpu_device):
    model = make_hyperprior(mean_scale=True).to(gpu_device)
    codec = fast_compressai.accelerate(model, P=4, device=str(gpu_device))._coder
    with torch.no_grad():
        latents = [codec.analyze(torch.rand(1 + i % 2, 3, 64, 64 << i % 2, device=gpu_device))
                   for i in range(4)]
    want = []
    for pair in latents:
        out = codec.encode_latents(pair)
        want.append([p.to_bytes() for p in out["strings"]]
                    + [codec.decode_latents(out["strings"], out["shape"]).cpu()])
    torch.cuda.synchronize()
    streams = [torch.cuda.current_stream(gpu_device)] * 2 + [torch.cuda.Stream(gpu_device)
                                                             for _ in range(2)]
    wrong = []

    def work(i):
        try:
            with torch.cuda.stream(streams[i]):
                for _ in range(20):
                    out = codec.encode_latents(latents[i])
                    y_hat = codec.decode_latents(out["strings"], out["shape"]).cpu()
                    got = [p.to_bytes() for p in out["strings"]]
                    if got != want[i][:2] or not torch.equal(y_hat, want[i][2]):
                        wrong.append((i, "other results"))
        except Exception as e:  # shown by the assertion below
            wrong.append((i, repr(e)))

    print("case: threads and streams", flush=True)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []
