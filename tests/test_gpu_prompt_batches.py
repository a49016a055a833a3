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


def test_short_prompt_of_large_layers_is_no_less_exact(cuda):
    """9 tokens through layers of more than 2^24 weights, as a batch and as steps:
    the batch's error against float64 is not the larger one (one layer, one output:
    1.5e-7 and 6e-7 of the result; on the fixed-point projections 1.1e-6)."""
    H, I = 2048, 8320
    cfg = dict(num_layers=1, hidden=H, intermediate=I, num_heads=16, num_kv_heads=4, head_dim=128,
               vocab=1024, eps=1e-6, rope_theta=1e6, qkv_bias=False)
    w = synth.decoder_weights(cfg, 96, 4, 32, 32)
    for lw in w["layers"]:   # large channels, and outputs of about unit size
        lw["post_norm"][::128] = 12.0
        for t in ("qkv_s", "o_s", "gate_s", "up_s", "down_s"):
            lw[t] *= 0.1
    dec = decoder_from_weights(w, cfg, group_size=32, max_seq_len=32)
    toks = [int(t) for t in np.random.default_rng(96).integers(0, cfg["vocab"], 9)]
    dec.prefill_tokens(toks, 0)
    batch = np.array(dec.get_logits(), np.float64)
    dec.reset_kv_cache()
    for i, t in enumerate(toks):
        steps, _ = dec._step(t, i, True)
    dec.close()

    f = lambda a: np.asarray(a, np.float64)
    deq = lambda p, s: (np.stack((p & 15, p >> 4), -1).reshape(p.shape[0], -1) - 8.0) * \
        np.repeat(f(s), 32, 1)
    rms = lambda v, n: v / np.sqrt((v * v).mean(1, keepdims=True) + cfg["eps"]) * f(n)
    y, x, n, hd = w["layers"][0], f(w["embed"])[toks], len(toks), 128
    qkv = rms(x, y["in_norm"]) @ deq(y["qkv_w"], y["qkv_s"]).T
    ang = np.arange(n)[:, None] / cfg["rope_theta"] ** (np.arange(0, hd, 2) / hd)
    cos, sin = (np.tile(fn(ang), (1, 2))[:, None] for fn in (np.cos, np.sin))
    turn = lambda v: v * cos + np.concatenate((-v[..., hd // 2:], v[..., :hd // 2]), -1) * sin
    q, k, v = (a.reshape(n, -1, hd) for a in np.split(qkv, (H, H + 4 * hd), 1))
    q, k, v = turn(q), np.repeat(turn(k), 4, 1), np.repeat(v, 4, 1)
    s = np.einsum("ihd,jhd->hij", q, k) / np.sqrt(hd) + np.triu(np.full((n, n), -np.inf), 1)
    p = np.exp(s - s.max(-1, keepdims=True))
    a = np.einsum("hij,jhd->ihd", p / p.sum(-1, keepdims=True), v).reshape(n, -1)
    x = x + a @ deq(y["o_w"], y["o_s"]).T
    xn = rms(x, y["post_norm"])
    g, u = (xn @ deq(y[t + "_w"], y[t + "_s"]).T for t in ("gate", "up"))
    x = x + (g / (1 + np.exp(-g)) * u) @ deq(y["down_w"], y["down_s"]).T
    ref = (rms(x, w["final_norm"]) @ f(w["lm_head_w"]).T)[-1]
    err = [np.linalg.norm(f(t) - ref) / np.linalg.norm(ref) for t in (batch, steps)]
    print(f"case short prompt errors: batch {err[0]:.2e}, steps {err[1]:.2e}", flush=True)
    assert err[0] <= 1.02 * err[1]
