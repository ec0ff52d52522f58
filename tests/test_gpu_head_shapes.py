"""The resident-h head kernel's shapes: tiles per wave, waves per block and record sizes follow the
head's size; both sides of its lines for tiles per wave and for one or two blocks a CU run here, at a
short depth (deeper heads and more than 13 waves a CU: test_gpu_head_depth.py), against the
oracle's scalar head (the reference kernel test's 1e-3 tolerance) and, for the tokens, against the
oracle's selection on the device's own logits (exact)."""
import numpy as np
import pytest

from helpers import hidden_bf16, twd, wsb_bytes

pytestmark = pytest.mark.gpu
CAP = 30.0
D = 384  # three chunks: an odd count, so the padding chunk is there

# 256 CUs: one tile per wave up to 4,096 tiles, two up to 8,192, four past that; one block per CU up
# to 12 waves, two blocks of half past that
SIZES = [
    16 * 3 + 5,            # fewer tiles than one block's waves
    49_152, 49_153,        # 12 waves per CU | 13: two blocks of 7
    65_536, 65_537,        # one | two tiles per wave
    131_072, 131_075,      # two | four tiles per wave
]


@pytest.fixture(scope="module", params=SIZES)
def head(request, oracle):
    import torch
    t = twd()
    dev = torch.device("cuda:0")
    V = request.param
    W, S, B = oracle.gen_lm_head(V, V, D)
    h = t.LMHead(torch.from_numpy(wsb_bytes(W, S, B)).to(dev), V, D, CAP)
    yield torch, dev, t, h, V, (W, S, B)
    h.close()


def _close(got, want):
    assert np.all(np.abs(got - want) <= 1e-3 + 1e-3 * np.abs(want))


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_greedy_shapes(head, oracle, M):
    torch, dev, t, h, V, (W, S, B) = head
    hb = hidden_bf16(7 * M + V, M, D)
    hid = torch.from_numpy(np.ascontiguousarray(hb).view(np.int16)).to(dev)
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    for _ in range(2):  # the second launch finds the counters as the first left them
        tok = h.greedy(hid, logits=logits).cpu().numpy()
    lg = logits.cpu().numpy()
    assert np.array_equal(h.logits(hid).cpu().numpy().view(np.uint32), lg.view(np.uint32))
    hf = (hb.astype(np.uint32) << 16).view(np.float32)
    for m in range(M):
        assert tok[m] == oracle.argmax(lg[m])
    for m in {0, M - 1}:
        _close(lg[m], oracle.lm_head(W, S, B, hf[m], D, softcap=CAP))


@pytest.mark.parametrize("M", [1, 4, 5, 8])
def test_rmsnorm_shapes(head, oracle, M):
    torch, dev, t, h, V, (W, S, B) = head
    rng = np.random.default_rng(M + V)
    x = (5.0 * rng.standard_normal((M, D))).astype(np.float32)
    wb = hidden_bf16(3, 1, D)[0]
    wf = (wb.astype(np.uint32) << 16).view(np.float32)
    xd = torch.from_numpy(x).to(dev)
    wd = torch.from_numpy(np.ascontiguousarray(wb).view(np.int16)).to(dev)
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    tok = h.greedy_rmsnorm(xd, wd, 1e-6, logits=logits).cpu().numpy()
    lg = logits.cpu().numpy()
    for m in range(M):
        assert tok[m] == oracle.argmax(lg[m])
    for m in {0, M - 1}:
        hn = (x[m].astype(np.float64) / np.sqrt(np.mean(x[m].astype(np.float64) ** 2) + 1e-6) * wf).astype(np.float32)
        _close(lg[m], oracle.lm_head(W, S, B, hn, D, softcap=CAP))


@pytest.mark.parametrize("M,norm", [(1, False), (4, True), (5, False), (8, True)])
def test_sample_shapes(head, oracle, M, norm):
    # the records hold 16, 32 or 64 rows by shape; history ids on record and block edges
    torch, dev, t, h, V, _ = head
    rng = np.random.default_rng(11 * M + V)
    n = 96
    hist = rng.integers(0, V, M * n)
    edges = np.array([0, 15, 16, 63, 64, 111, 112, V - 1], dtype=np.int64)
    hist[:8] = edges[edges < V][np.arange(8) % (edges < V).sum()]
    hist = hist.astype(np.int32)
    hd = torch.from_numpy(hist).to(dev)
    prm = [t.RowParams(0.9, 0.95 if m % 2 else 1.0, 30 + 40 * (m % 3), 1.2, float(np.float32(rng.uniform(0, 0.999))),
                       CAP, m * n, n) for m in range(M)]
    if norm:
        x = torch.from_numpy((5.0 * rng.standard_normal((M, D))).astype(np.float32)).to(dev)
        w = torch.from_numpy(np.ascontiguousarray(hidden_bf16(4, 1, D)[0]).view(np.int16)).to(dev)
        raw = h.logits_rmsnorm(x, w).cpu().numpy()
        tok, lg = h.sample_rmsnorm(x, w, prm, history=hd)
    else:
        hid = torch.from_numpy(np.ascontiguousarray(hidden_bf16(M + V, M, D)).view(np.int16)).to(dev)
        raw = h.logits(hid).cpu().numpy()
        tok, lg = h.sample(hid, prm, history=hd)
    tok, lg = tok.cpu().numpy(), lg.cpu().numpy()
    for m, p in enumerate(prm):
        pen = oracle.apply_repetition_penalty(raw[m], hist[m * n:(m + 1) * n], p.repetition_penalty, CAP)
        assert np.array_equal(lg[m].view(np.uint32), pen.view(np.uint32))
        assert int(tok[m]) & 0xFFFFFFFF == oracle.sample_token(pen, p.temperature, p.top_p, p.top_k, u=p.uniform)
