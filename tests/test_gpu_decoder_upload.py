"""A decoder built from device tensors whose producing kernels are still queued
on the caller's stream: the uploads, the binary16 rounding of group-64 scales
and the cache's clearing all take effect before its first step, whatever is
queued.  Against the decoder of the same weights from host arrays, bit for bit."""
import numpy as np
import pytest
import torch

from torchburn_amd import synth
from torchburn_amd.decoder import decoder_from_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gs,lmkind", [(64, 4), (64, 32), (32, 4)])
def test_build_behind_queued_work(cuda, gs, lmkind):
    print(f"case decoder upload gs={gs} lmkind={lmkind}", flush=True)
    cfg = dict(num_layers=2, hidden=1024, intermediate=1024, num_heads=16, num_kv_heads=4,
               head_dim=64, vocab=1024, eps=1e-6, rope_theta=1e6, qkv_bias=True)
    w = synth.decoder_weights(cfg, 81, 4, lmkind, gs)
    toks = [int(t) for t in np.random.default_rng(81).integers(0, cfg["vocab"], 9)]

    def logits(weights):
        dec = decoder_from_weights(weights, cfg, group_size=gs, max_seq_len=64)
        dec.prefill_tokens(toks[:-1], 0)
        out = dec.decode_step(toks[-1], len(toks) - 1).numpy().copy()
        dec.close()
        return out

    want = logits(w)
    src = {k: torch.from_numpy(v).to(cuda) for k, v in w.items() if isinstance(v, np.ndarray)}
    layers = [{k: torch.from_numpy(v).to(cuda) for k, v in lw.items()} for lw in w["layers"]]
    a = torch.randn((4096, 4096), device=cuda)
    for _ in range(3):
        for _ in range(20):
            a = (a @ a).clamp_(-1, 1)   # some milliseconds on the default stream
        late = {k: v.clone() for k, v in src.items()}
        late["lm_head_s"] = late.get("lm_head_s")
        late["layers"] = [{k: v.clone() for k, v in lw.items()} for lw in layers]
        assert np.array_equal(logits(late), want)
