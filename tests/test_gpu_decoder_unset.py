"""A decoder one of whose layers was never set refuses every way to run it:
steps, prompts of any length (stepped or batched) and verify_tokens, for INT4
and INT8 layers, and runs once the layer is there."""
import ctypes as C

import numpy as np
import pytest

from torchburn_amd import decoder as D
from torchburn_amd import _lib

pytestmark = pytest.mark.gpu

H, I, HEADS, HD, V, GS = 64, 128, 1, 64, 96, 32


def layer(g, bits):
    """The 13 tensors of a layer in tb_decoder_set_layer's order."""
    def proj(n, k):
        if bits == 4:
            return [g.integers(0, 256, (n, k // 2), dtype=np.uint8),
                    np.full((n, k // GS), 0.01, np.float32)]
        return [g.integers(-127, 128, (n, k)).astype(np.int8), np.full(n, 0.001, np.float32)]
    one = np.ones(H, np.float32)
    return [one, *proj(3 * HD, H), *proj(H, HD), one, *proj(I, H), *proj(I, H), *proj(H, I), None]


@pytest.mark.parametrize("bits", [4, 8])
def test_unset_layer_is_refused(cuda, bits):
    print(f"case unset layer bits={bits}", flush=True)
    L = D._bind()
    g = np.random.default_rng(5)
    embed = g.normal(0, 1, (V, H)).astype(np.float32)
    lm = g.normal(0, 0.1, (V, H)).astype(np.float32)
    cfg = D._Config(2, H, I, HEADS, HEADS, HD, V, GS, 64, 1e-6, 1e4, bits, 32)
    h = C.c_void_p()
    norm = np.ones(H, np.float32)
    _lib.check(L.tb_decoder_create(C.byref(cfg), embed.ctypes.data, norm.ctypes.data,
                                   lm.ctypes.data, None, C.byref(h)))
    def set_layer(i):
        t = layer(g, bits)
        _lib.check(L.tb_decoder_set_layer(h, i, *[None if a is None else a.ctypes.data for a in t]))

    def runs():
        out, am, end = np.empty((20, V), np.float32), C.c_int64(), C.c_int64()
        yield "step", L.tb_decoder_step(h, 1, 0, out.ctypes.data, C.byref(am))
        for n in (2, 3, 20):
            toks = np.arange(n, dtype=np.int64)
            yield f"prompt {n}", L.tb_decoder_prefill(h, toks.ctypes.data, n, 0, C.byref(end))
            yield f"verify {n}", L.tb_decoder_verify(h, 0, toks.ctypes.data, n, out.ctypes.data)

    set_layer(0)
    for what, rc in runs():
        assert rc == _lib.TB_ERR_VALUE, what
        assert "layer 1 was never set" in _lib.lib().tb_last_error().decode(), what
    set_layer(1)
    for what, rc in runs():
        assert rc == _lib.TB_OK, what
    _lib.check(L.tb_decoder_destroy(h))
