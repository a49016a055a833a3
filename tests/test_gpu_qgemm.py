"""The batched f16-limb projection (INT4 from 5 rows, INT8 from 4, or 3 on 32 Mi
weights) at the edges of its tiles: rows around 32 and 64, column blocks of 128 and
256, K that is no whole number of 128-element stages, K splits, every scale form,
and rows of extreme or non-finite activations.  Against float64; the bound follows the kernel: two f16
limbs hold an activation to 2^-22, and every sum is f32, one addition per 32
elements of K plus the splits', so an output is off by at most
(K / 32 + 16) 2^-24 sum |w x|."""
import numpy as np
import pytest
import torch

import torchburn_amd as tb
from torchburn_amd import _lib, synth

pytestmark = pytest.mark.gpu


def deq4(w, s, gs):
    q = np.stack((w & 15, w >> 4), -1).reshape(w.shape[0], -1).astype(np.float64) - 8
    return q * (np.repeat(s.astype(np.float64), gs, 1) if s.ndim == 2 else s.astype(np.float64)[:, None])


def check(y, x, w, bias=None, res=None):
    """y against x w^T (+ bias) (+ res) within the bound above, row by row where finite."""
    xd = x.astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = xd @ w.T
        mag = np.abs(xd) @ np.abs(w).T
    for t in (bias, res):
        if t is not None:
            ref = ref + t.astype(np.float64)
            mag = mag + np.abs(t)
    bound = (x.shape[1] / 32 + 16) * 2.0 ** -24 * mag + 1e-37
    fin = np.isfinite(x).all(1)
    assert np.isfinite(y[fin]).all()
    assert (np.abs(y[fin] - ref[fin]) <= bound[fin]).all()
    assert not np.isfinite(y[~fin]).any()
    assert (np.isnan(y[~fin]) == np.isnan(ref[~fin])).all()
    inf = ~np.isnan(ref[~fin])
    assert (y[~fin][inf] == ref[~fin][inf].astype(np.float32)).all()


@pytest.mark.parametrize("m,n,k,gs,v2", [
    (17, 33, 160, 32, False), (32, 128, 128, 64, False), (33, 257, 2080, 32, False),
    (64, 300, 4096, 128, False), (65, 130, 96, 32, False), (130, 515, 1600, 64, False),
    (19, 70, 224, 0, False), (48, 129, 64, 64, True), (200, 65, 1600, 64, True),
    (500, 2050, 4128, 32, False)])   # 128 record blocks: 4 rows each
def test_w4_projection_edges(cuda, m, n, k, gs, v2):
    print(f"case qgemm w4 m={m} n={n} k={k} gs={gs} v2={v2}", flush=True)
    g = synth.rng(71, m, n, k)
    x = synth.activations(g, m, k)
    x[:, 3::37] *= 50.0
    b = synth.activations(g, n)
    w, s = synth.int4_weight(g, n, k, gs or k)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    if gs == 0:
        s = s.reshape(-1)
        y = tb.w4a32_linear(T(x), T(w), T(s), T(b))
    elif v2:
        s = s.astype(np.float16).astype(np.float32)
        y = tb.w4a32_grouped_linear_v2(T(x), tb.pack_rows_w4a32_group64_v1_to_v2(T(w), T(s), k), T(b))
    else:
        y = tb.w4a32_grouped_linear(T(x), T(w), T(s), T(b), group_size=gs)
    check(y.cpu().numpy(), x, deq4(w, s, gs or k), b)


@pytest.mark.parametrize("m,n,k,per_row", [
    (3, 8200, 4096, True),   # 32 Mi weights: from 3 rows
    (5, 33, 160, True), (32, 129, 992, False), (33, 300, 2080, True), (130, 260, 4160, True),
    (497, 2050, 2080, True),   # 128 record blocks: 4 rows each
    (6, 40, 16416, True)])   # K past the streaming GEMV's range
def test_w8_projection_edges(cuda, m, n, k, per_row):
    print(f"case qgemm w8 m={m} n={n} k={k}", flush=True)
    g = synth.rng(74, m, n, k)
    x = synth.activations(g, m, k)
    x[:, 3::37] *= 50.0
    x[m - 1, 5] = np.inf
    b = synth.activations(g, n)
    w, s = synth.int8_weight(g, n, k)
    w[:, 5] = np.where(w[:, 5] == 0, 1, w[:, 5])   # inf * w has one sign or the other
    s = s if per_row else s[:1]
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    y = tb.w8a32_linear(T(x), T(w), T(s), T(b))
    check(y.cpu().numpy(), x, w.astype(np.float64) * s.astype(np.float64)[:, None], b)


@pytest.mark.parametrize("m,k,inter", [(5, 96, 160), (40, 992, 1056), (130, 256, 4128)])
def test_w8_mlp_rows(cuda, m, k, inter):
    print(f"case qgemm w8 mlp m={m} k={k} inter={inter}", flush=True)
    g = synth.rng(75, m, k, inter)
    x, r = synth.activations(g, m, k), synth.activations(g, m, k)
    wts = [synth.int8_weight(g, n, kk) for n, kk in ((inter, k), (inter, k), (k, inter))]
    gb, ub, db = (synth.activations(g, n) for n in (inter, inter, k))
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    (gw, gs), (uw, us), (dw, ds) = wts
    us = us[:1]
    y = tb.fused_swiglu_mlp_w8a32(T(x), T(gw), T(gs), T(gb), T(uw), T(us), T(ub), T(dw), T(ds),
                                  T(db), residual=T(r)).cpu().numpy()
    D = lambda w, s: w.astype(np.float64) * s.astype(np.float64)[:, None]
    a, u = x.astype(np.float64) @ D(gw, gs).T + gb, x.astype(np.float64) @ D(uw, us).T + ub
    ref = (a / (1 + np.exp(-a)) * u) @ D(dw, ds).T + db + r
    assert np.abs(y - ref).max() / np.abs(ref).max() < 2e-6


def test_w4_extreme_and_nonfinite_rows(cuda):
    m, n, k, gs = 40, 130, 1152, 32
    g = synth.rng(72, m)
    x = synth.activations(g, m, k)
    x[1] *= 2.0 ** 100
    x[2] *= 2.0 ** -110
    x[3] = 0.0
    x[4, :k // 2] *= 2.0 ** 60
    x[33, 7] = np.inf
    x[34, 100] = -np.inf
    x[34, 1100] = np.inf
    x[35, 64] = np.nan
    w, s = synth.int4_weight(g, n, k, gs)
    r = synth.activations(g, m, n)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    y = tb.w4a32_grouped_linear_residual(T(x), T(w), T(s), T(r), group_size=gs)
    check(y.cpu().numpy(), x, deq4(w, s, gs), res=r)


@pytest.mark.parametrize("m,k,inter,gs", [
    (40, 2048, 4096, 32),    # limbs and partials within the scratch the entry point counts
    (20, 4128, 64, 32)])     # limbs larger than that count: a plan that fits the rest
def test_noalloc_mlp_at_17_rows_or_more(cuda, m, k, inter, gs):
    print(f"case qgemm noalloc m={m} k={k} inter={inter}", flush=True)
    g = synth.rng(73, m, k)
    x, r = synth.activations(g, m, k), synth.activations(g, m, k)
    wts = [synth.int4_weight(g, n, kk, gs) for n, kk in ((inter, k), (inter, k), (k, inter))]
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    t = [T(a) for p in wts for a in p]
    dx, dr = T(x), T(r)
    P = lambda a: a.data_ptr()
    outs = []
    for name in ("tb_fused_swiglu_mlp_w4a32_noalloc", "tb_fused_swiglu_mlp_w4a32"):
        out = torch.empty((m, k), device=cuda)
        _lib.check(getattr(_lib.lib(), name)(
            P(dx), P(t[0]), P(t[1]), None, P(t[2]), P(t[3]), None, P(t[4]), P(t[5]), None, P(dr),
            P(out), m, k, inter, k, gs, torch.cuda.current_stream(cuda).cuda_stream))
        outs.append(out.cpu().numpy())
    gw, uw, dw = (deq4(w, s, gs) for w, s in wts)
    a, u = x.astype(np.float64) @ gw.T, x.astype(np.float64) @ uw.T
    ref = (a / (1 + np.exp(-a)) * u) @ dw.T + r
    for o in outs:
        assert np.abs(o - ref).max() / np.abs(ref).max() < 2e-6


@pytest.mark.parametrize("m,n,k", [(5, 300, 4096), (70, 515, 2080)])
def test_w8_graphs_of_one_stream_run_side_by_side(cuda, m, n, k):
    """A captured INT8 projection uses no workspace: two graphs captured on one
    stream replay on two others at a time, beside eager calls on the first."""
    print(f"case qgemm w8 graphs m={m} n={n} k={k}", flush=True)
    g = synth.rng(79, m, n, k)
    x = [synth.activations(g, m, k) for _ in range(3)]
    w = g.integers(-127, 128, (n, k)).astype(np.int8)
    s = (0.001 + 0.01 * g.random(n)).astype(np.float32)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    dx, dw, ds = [T(a) for a in x], T(w), T(s)
    torch.cuda.synchronize()
    cap, graphs, ys = torch.cuda.Stream(), [], []
    for i in range(2):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[i], stream=cap):
            ys.append(tb.w8a32_linear(dx[i], dw, ds))
    st = [torch.cuda.Stream(), torch.cuda.Stream()]
    for rep in range(3):
        for y in ys:
            y.zero_()
        torch.cuda.synchronize()
        for i in range(2):
            with torch.cuda.stream(st[i]):
                graphs[i].replay()
        with torch.cuda.stream(cap):
            ye = tb.w8a32_linear(dx[2], dw, ds)
        torch.cuda.synchronize()
        for i, y in enumerate(ys + [ye]):
            check(y.cpu().numpy(), x[i], w * s.astype(np.float64)[:, None])


def graph_us(f, n=20):
    """Microseconds of one call of f inside a captured graph of n."""
    f()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        for _ in range(n):
            f()
    best = float("inf")
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        g.replay()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / n)
    return best


@pytest.mark.parametrize("n,k", [(4096, 4096), (4096, 14336), (896, 4864), (1024, 512)])
def test_captured_w8_is_no_slower_than_passes_of_two_rows(cuda, n, k):
    """Without scratch the batched kernel and GEMV passes of 2 rows (4 us at the
    least, and the weights read again) are both there: the faster one runs, within a
    half (the batched kernel alone takes up to 7 times the passes at these rows)."""
    g = synth.rng(105, n, k)
    w, s = synth.int8_weight(g, n, k)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)
    dw, ds = T(w), T(s)
    xs = {m: synth.activations(g, m, k) for m in (2, 4, 8, 32)}
    two = graph_us(lambda x=T(xs[2]): tb.w8a32_linear(x, dw, ds))
    for m in (4, 8, 32):
        x = T(xs[m])
        us = graph_us(lambda: tb.w8a32_linear(x, dw, ds))
        print(f"case w8 captured m={m} n={n} k={k}: {us:.1f} us, a pass {two:.1f}", flush=True)
        assert us < 1.5 * two * m / 2
    out = {}
    gr = torch.cuda.CUDAGraph()
    dx = {m: T(x) for m, x in xs.items()}
    with torch.cuda.graph(gr, stream=torch.cuda.Stream()):
        for m, x in dx.items():
            out[m] = tb.w8a32_linear(x, dw, ds)
    for _ in range(3):
        gr.replay()
        torch.cuda.synchronize()
        for m, y in out.items():
            check(y.cpu().numpy(), xs[m], w.astype(np.float64) * s.astype(np.float64)[:, None])
            y.zero_()
