"""The two forms of each device quantizer, four elements per load and one, bit
for bit against the oracle: sizes around a block's 4096 elements, weights at an
address that is no multiple of 16 bytes, and rows with infinities and NaN (both
forms alike)."""
import numpy as np
import pytest
import torch

import torchburn_amd as tb
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def on_gpu(w, cuda, shifted):
    """w on the GPU, 4 bytes past a 16-byte boundary when shifted."""
    buf = torch.empty(w.size + 4, dtype=torch.float32, device=cuda)
    t = buf[1 if shifted else 0:][:w.size].reshape(w.shape)
    t.copy_(torch.from_numpy(w))
    return t


@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("n,k,gs", [(1, 32, 32), (1, 64, 64), (43, 96, 32), (16, 256, 64),
                                    (33, 4160, 64), (5, 8224, 32)])
def test_int4_groups(cuda, n, k, gs, shifted):
    print(f"case quantize int4 n={n} k={k} gs={gs} shifted={shifted}", flush=True)
    w = np.random.default_rng(n + k).standard_normal((n, k)).astype(np.float32)
    w[n // 2, :gs] = 0.0
    q, s = tb.quantize_weight_int4_grouped(on_gpu(w, cuda, shifted), group_size=gs)
    qr, sr = O.quantize_int4_grouped(w, gs)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr)


@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("n,k", [(3, 4), (5, 30), (7, 4096), (4, 4100), (2, 9000)])
def test_int8_rows(cuda, n, k, shifted):
    print(f"case quantize int8 n={n} k={k} shifted={shifted}", flush=True)
    w = np.random.default_rng(n + k).standard_normal((n, k)).astype(np.float32)
    w[n - 1] = 0.0
    q, s = tb.quantize_weight_int8(on_gpu(w, cuda, shifted))
    qr, sr = O.quantize_int8(w)
    assert np.array_equal(q.cpu().numpy(), qr) and np.array_equal(s.cpu().numpy(), sr)


def test_nonfinite_weights_alike(cuda):
    w = np.random.default_rng(5).standard_normal((6, 512)).astype(np.float32)
    w[0, 3], w[1, 70], w[2, :64], w[3, 100] = np.inf, -np.inf, np.nan, np.nan
    for f in (lambda t: tb.quantize_weight_int4_grouped(t, group_size=64),
              lambda t: tb.quantize_weight_int4_grouped(t, group_size=32), tb.quantize_weight_int8):
        a, b = f(on_gpu(w, cuda, False)), f(on_gpu(w, cuda, True))
        assert torch.equal(a[0], b[0])
        assert torch.equal(a[1].nan_to_num(7.0), b[1].nan_to_num(7.0))
