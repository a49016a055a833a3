"""Batched prompts against the CPU oracle's steps where the batch changes form:
INT8 layers (GEMV passes and the batched kernel, by rows), prompts of 2 to 6
tokens around the shortest batch, a second chunk after 1024 rows, buffers that
grow with a longer prompt, and INT8 verify_tokens with every lm_head."""
import numpy as np
import pytest

from oracle import oracle as O
from torchburn_amd import synth
from torchburn_amd._lib import UnsupportedOpError
from torchburn_amd.decoder import decoder_from_weights

pytestmark = pytest.mark.gpu

TOL = 2e-4   # max|d| / max|ref|, as for the decoder's steps


def pair(seed, wkind, lmkind, max_seq, **kw):
    cfg = dict(num_layers=2, hidden=256, intermediate=512, num_heads=4, num_kv_heads=2,
               head_dim=64, vocab=1000, eps=1e-6, rope_theta=1e6, qkv_bias=True)
    cfg.update(kw)
    w = synth.decoder_weights(cfg, seed, wkind, lmkind, 32)
    ref = O.Decoder(w, dict(num_layers=cfg["num_layers"], hidden=cfg["hidden"],
                            intermediate=cfg["intermediate"], num_heads=cfg["num_heads"],
                            num_kv_heads=cfg["num_kv_heads"], head_dim=cfg["head_dim"],
                            vocab=cfg["vocab"], group_size=32, max_seq=max_seq,
                            rope_theta=cfg["rope_theta"], eps=cfg["eps"], wkind=wkind,
                            lmkind=lmkind))
    return ref, decoder_from_weights(w, cfg, group_size=32, max_seq_len=max_seq), cfg


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


@pytest.mark.parametrize("wkind,lmkind,lengths", [
    (8, 8, (2, 3, 6)), (8, 32, (40, 70)), (4, 4, (2, 3, 5)), (4, 4, (5, 300, 1030)), (8, 8, (520,))])
def test_prompts_one_after_another(cuda, wkind, lmkind, lengths):
    print(f"case prompts wkind={wkind} lmkind={lmkind} lengths={lengths}", flush=True)
    ref, dec, cfg = pair(91, wkind, lmkind, sum(lengths) + 8)
    g = np.random.default_rng(91)
    pos = 0
    for n in lengths:
        toks = [int(t) for t in g.integers(0, cfg["vocab"], n)]
        for i, t in enumerate(toks):
            lo = ref.step(t, pos + i)
        assert dec.prefill_tokens(toks, pos) == pos + n
        assert rel(dec.get_logits(), lo) < TOL
        pos += n
    for i in range(3):   # steps over the cache that the batches wrote
        t = O.argmax(lo)
        lo = ref.step(t, pos + i)
        lg, am = dec._step(t, pos + i, True)
        assert rel(lg, lo) < TOL and am == O.argmax(lo)
    ref.close()
    dec.close()


@pytest.mark.parametrize("wkind", [4, 8])
def test_same_prompt_same_bits(cuda, wkind):
    """A prompt's logits do not depend on the prompts before it: 70 rows, whose
    gate/up plan takes more scratch than any of 256 rows, before and after 700."""
    print(f"case same prompt wkind={wkind}", flush=True)
    cfg = dict(num_layers=2, hidden=512, intermediate=2048, num_heads=8, num_kv_heads=2,
               head_dim=64, vocab=1000, eps=1e-6, rope_theta=1e6, qkv_bias=True)
    dec = decoder_from_weights(synth.decoder_weights(cfg, 93, wkind, wkind, 32), cfg,
                               group_size=32, max_seq_len=800)
    g = np.random.default_rng(93)
    short, long = ([int(t) for t in g.integers(0, cfg["vocab"], k)] for k in (70, 700))

    def logits(toks):
        dec.reset_kv_cache()
        dec.prefill_tokens(toks, 0)
        return np.array(dec.get_logits())

    first = logits(short)
    logits(long)
    assert np.array_equal(logits(short), first)
    dec.close()


@pytest.mark.parametrize("lmkind,n", [(8, 2), (8, 7), (8, 70), (32, 5)])
def test_int8_verify_rows(cuda, lmkind, n):
    print(f"case int8 verify lmkind={lmkind} n={n}", flush=True)
    ref, dec, cfg = pair(92, 8, lmkind, 128)
    g = np.random.default_rng(92)
    pre, toks = ([int(t) for t in g.integers(0, cfg["vocab"], k)] for k in (9, n))
    for i, t in enumerate(pre):
        ref.step(t, i)
    dec.prefill_tokens(pre, 0)
    want = np.stack([ref.step(t, 9 + i).copy() for i, t in enumerate(toks)])
    assert rel(dec.verify_tokens(9, toks), want) < TOL
    ref.close()
    dec.close()


@pytest.mark.parametrize("wkind,refused,taken", [(4, (3, 15), (16,)), (8, (3, 16), ())])
def test_layers_without_steps(cuda, wkind, refused, taken):
    """Layers wider than a GEMV pass, whose steps are refused: so are the prompts
    and verify_tokens that steps stand for."""
    print(f"case wide layers wkind={wkind}", flush=True)
    cfg = dict(num_layers=1, hidden=256, intermediate=16416, num_heads=4, num_kv_heads=2,
               head_dim=64, vocab=1000, eps=1e-6, rope_theta=1e6, qkv_bias=True)
    dec = decoder_from_weights(synth.decoder_weights(cfg, 94, wkind, wkind, 32), cfg,
                               group_size=32, max_seq_len=64)
    with pytest.raises(UnsupportedOpError, match="K <= 16384"):
        dec._step(1, 0, True)
    for n in refused:
        with pytest.raises(UnsupportedOpError, match="K <= 16384"):
            dec.prefill_tokens(list(range(n)), 0)
    for n in taken:
        assert dec.prefill_tokens(list(range(n)), 0) == n
    if wkind == 8:
        with pytest.raises(UnsupportedOpError, match="K <= 16384"):
            dec.verify_tokens(0, [1, 2, 3, 4])
    else:
        assert np.isfinite(dec.verify_tokens(0, [1, 2, 3, 4])).all()
    dec.close()
