"""Calls on a device with little memory left: the batched projections take the
scratch of their fastest plan only where it is there, and run with less, or with
none, where it is not."""
import contextlib

import numpy as np
import pytest
import torch

import torchburn_amd as tb
from torchburn_amd import synth
from torchburn_amd.decoder import decoder_from_weights

pytestmark = pytest.mark.gpu

MB = 1 << 20


@contextlib.contextmanager
def left(cuda, mb):
    """All but about mb MB of the device's memory held by someone else."""
    torch.cuda.synchronize()
    hold = []
    for size in (16384, 1024, 64):
        while torch.cuda.mem_get_info(cuda)[0] > (mb + size) * MB:
            hold.append(torch.empty(size * MB, dtype=torch.uint8, device=cuda))
    try:
        yield
    finally:
        hold.clear()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()


def normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def int4(g, n, k, gs):
    return (torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device="cuda", generator=g),
            torch.rand((n, k // gs), device="cuda", generator=g) * 0.01 + 0.001)


def same(call, cuda, mb):
    """call() with the device's memory free, then, its workspace released, with mb MB."""
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        want = call()
    torch.cuda.synchronize()
    tb.release_stream_workspace(s)
    with torch.cuda.stream(s):
        spare = torch.empty_like(want)   # the result's memory, in the allocator's cache
    del spare
    with left(cuda, mb):
        with torch.cuda.stream(s):
            got = call()
        torch.cuda.synchronize()
    tb.release_stream_workspace(s)
    err = ((got - want).norm() / want.norm()).item()
    assert err < 1e-6, err


def test_int4_linear(cuda):
    m, n, k, gs = 3210, 5191, 10816, 32   # 450 MB of scratch at its fastest, 67 at the least
    print(f"case short memory w4 linear m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    x, (w, s) = normal(g, m, k), int4(g, n, k, gs)
    same(lambda: tb.w4a32_grouped_linear(x, w, s, None, group_size=gs), cuda, 300)


def test_int4_mlp(cuda):
    m, k, inter, gs = 1959, 14144, 12768, 32   # h 95 MB, scratch 680 and 190 MB
    print(f"case short memory w4 mlp m={m} k={k} inter={inter}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = normal(g, m, k)
    (gw, gs_), (uw, us), (dw, ds) = (int4(g, n, kk, gs)
                                     for n, kk in ((inter, k), (inter, k), (k, inter)))
    same(lambda: tb.fused_swiglu_mlp_w4a32(x, gw, gs_, None, uw, us, None, dw, ds, None,
                                           group_size=gs), cuda, 480)


def test_int8_mlp(cuda):
    """h has to be there; the batched projections' scratch does not."""
    m, k, inter = 640, 8192, 16384   # h 40 MB, scratch 80
    print(f"case short memory w8 mlp m={m} k={k} inter={inter}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = normal(g, m, k)
    w = [torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)
         for shape in ((inter, k), (inter, k), (k, inter))]
    s = [torch.rand(n, device="cuda", generator=g) * 1e-3 for n in (inter, inter, k)]
    same(lambda: tb.fused_swiglu_mlp_w8a32(x, w[0], s[0], None, w[1], s[1], None, w[2], s[2],
                                           None), cuda, 110)


@pytest.mark.parametrize("wkind,mb,n", [
    (4, 300, 700),   # an arena and the buffers of 256 rows would fit, not those of 1024
    (4, 190, 700), (8, 60, 40)])   # ... 256 rows, or fewer than a chunk: step by step
def test_prompt_and_verify(cuda, wkind, mb, n):
    print(f"case short memory prompt wkind={wkind} left={mb} n={n}", flush=True)
    cfg = dict(num_layers=1, hidden=4096, intermediate=14336, num_heads=32, num_kv_heads=8,
               head_dim=128, vocab=1000, eps=1e-6, rope_theta=1e6, qkv_bias=True)
    w = synth.decoder_weights(cfg, 95, wkind, wkind, 32)
    g = np.random.default_rng(95)
    warm, toks = ([int(t) for t in g.integers(0, cfg["vocab"], k)] for k in (2, n))

    def run(dec):
        dec.prefill_tokens(toks, 0)
        return np.array(dec.get_logits()), np.array(dec.verify_tokens(n, toks[:5]))

    out = []
    for mem in (None, mb):
        dec = decoder_from_weights(w, cfg, group_size=32, max_seq_len=n + 8)
        for i, t in enumerate(warm):
            dec._step(t, i, True)
        with left(cuda, mem) if mem else contextlib.nullcontext():
            out.append(run(dec))
        dec.close()
    for want, got in zip(*out):
        assert np.abs(got - want).max() / np.abs(want).max() < 2e-4
