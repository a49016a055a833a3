"""Batched projections on rows whose elements span more than two f16 limbs hold:
one or more channels 1e3 to 1e30 times the rest (and the lowest f32), where the
weights' codes are zero, so that the outputs are sums of the small elements
alone.  Against float64 within f32's own bound, (K / 32 + 16) 2^-24 sum |w x|, in
which the large channels have no part; and the rows around them as ever."""
import numpy as np
import pytest
import torch

import torchburn_amd as tb
from torchburn_amd import synth
from test_gpu_qgemm import check, deq4

pytestmark = pytest.mark.gpu

ONE, RUN = 5, slice(64, 96)   # channels of zero codes: a single one, a group of 32


def close(y, x, w):
    """check(), and every row's 2-norm within 3.5 times what f32 sums show (1.4e-7 at
    K = 14336, measured with and without large channels)."""
    check(y, x, w)
    ref = x.astype(np.float64) @ w.T
    assert (np.linalg.norm(y - ref, axis=1) <= 5e-7 * np.linalg.norm(ref, axis=1)).all()


def wide_rows(g, m, k):
    x = synth.activations(g, m, k)
    x[5 % m] = 0.0        # two elements, eight orders apart
    x[5 % m, (7, ONE)] = (1.0, 1e8)
    x[6 % m, ::3] = 0.0   # a sparse row, not a wide one
    if m > 13:
        x[13] *= np.exp(-20.0 * g.random(k)).astype(np.float32)   # of every size, no gap
    x[0, ONE] = 1e3
    x[1 % m, ONE] = 1e4
    x[2 % m, ONE] = 1e6
    x[3 % m, RUN] *= np.float32(1e8)
    x[4 % m, ONE] = np.finfo(np.float32).min
    for i, big in enumerate((5e4, 1e5, 2e5, 4e5, 8e5)):   # around the line of the wide form
        if 7 + i < m:
            x[7 + i, ONE] = big
    x[m - 1, ONE] = 1e30
    return x


@pytest.mark.parametrize("m,n,k,gs,v2", [
    (5, 33, 96, 32, False), (8, 130, 992, 32, False),      # limbs built in the blocks
    (40, 300, 1152, 64, True), (6, 130, 1024, 0, False),
    (100, 8200, 992, 32, False), (33, 8200, 2080, 32, False),   # records: 32-row tiles
    (33, 8200, 4096, 64, False), (33, 8200, 1600, 64, True),    # 64 rows
    (130, 8200, 4160, 32, False), (500, 8200, 4160, 32, False)])   # 64 and 128 rows, two columns
def test_w4_wide_rows(cuda, m, n, k, gs, v2):
    print(f"case wide w4 m={m} n={n} k={k} gs={gs} v2={v2}", flush=True)
    g = synth.rng(101, m, n, k)
    x = wide_rows(g, m, k)
    w, s = synth.int4_weight(g, n, k, gs or k)
    w[:, ONE // 2] = (w[:, ONE // 2] & 15) | 0x80
    w[:, RUN.start // 2:RUN.stop // 2] = 0x88
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    if gs == 0:
        s = s.reshape(-1)
        y = tb.w4a32_linear(T(x), T(w), T(s))
    elif v2:
        s = s.astype(np.float16).astype(np.float32)
        y = tb.w4a32_grouped_linear_v2(T(x), tb.pack_rows_w4a32_group64_v1_to_v2(T(w), T(s), k))
    else:
        y = tb.w4a32_grouped_linear(T(x), T(w), T(s), None, group_size=gs)
    close(y.cpu().numpy(), x, deq4(w, s, gs or k))


@pytest.mark.parametrize("m,n,k", [
    (4, 33, 160), (8, 300, 992), (6, 40, 16416), (100, 8200, 992), (130, 4128, 1600),
    (500, 515, 4160)])
def test_w8_wide_rows(cuda, m, n, k):
    print(f"case wide w8 m={m} n={n} k={k}", flush=True)
    g = synth.rng(102, m, n, k)
    x = wide_rows(g, m, k)
    w, s = synth.int8_weight(g, n, k)
    w[:, ONE] = 0
    w[:, RUN] = 0
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    y = tb.w8a32_linear(T(x), T(w), T(s))
    close(y.cpu().numpy(), x, w.astype(np.float64) * s.astype(np.float64)[:, None])


@pytest.mark.parametrize("m,k,inter", [
    (8, 992, 1056), (200, 992, 2080),   # the second in chunks of 12 groups
    (130, 4096, 4128)])
@pytest.mark.parametrize("bits", [4, 8])
def test_swiglu_wide_rows(cuda, m, k, inter, bits):
    print(f"case wide mlp m={m} k={k} inter={inter} bits={bits}", flush=True)
    g = synth.rng(103, m, k, inter, bits)
    x = wide_rows(g, m, k)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    make = (lambda n, kk: synth.int4_weight(g, n, kk, 32)) if bits == 4 else \
        (lambda n, kk: synth.int8_weight(g, n, kk))
    wts = [make(n, kk) for n, kk in ((inter, k), (inter, k), (k, inter))]
    for w, _ in wts[:2]:
        if bits == 4:
            w[:, ONE // 2] = (w[:, ONE // 2] & 15) | 0x80
            w[:, RUN.start // 2:RUN.stop // 2] = 0x88
        else:
            w[:, ONE] = 0
            w[:, RUN] = 0
    (gw, gs), (uw, us), (dw, ds) = wts
    if bits == 4:
        y = tb.fused_swiglu_mlp_w4a32(T(x), T(gw), T(gs), None, T(uw), T(us), None, T(dw), T(ds),
                                      None, group_size=32)
        D = lambda w, s: deq4(w, s, 32)
    else:
        y = tb.fused_swiglu_mlp_w8a32(T(x), T(gw), T(gs), None, T(uw), T(us), None, T(dw), T(ds),
                                      None)
        D = lambda w, s: w.astype(np.float64) * s.astype(np.float64)[:, None]
    a, u = x.astype(np.float64) @ D(gw, gs).T, x.astype(np.float64) @ D(uw, us).T
    ref = (a / (1 + np.exp(-a)) * u) @ D(dw, ds).T
    err = np.abs(y.cpu().numpy() - ref).max(1) / np.abs(ref).max(1)
    assert err.max() < 2e-6, (err.argmax(), err.max())
