"""Captured selections with top_k > 256, and the scratch they hold: other calls on the same selector
between the replays, with other top_k or more such rows, leave a captured call's scratch where it is;
a selector warmed up at one top_k is captured at another; a first call inside a capture that allows
allocation. Every replay against the eager ids of the same rows, those against the oracle."""
import numpy as np
import pytest

from helpers import twd

pytestmark = pytest.mark.gpu

V = 50000


@pytest.fixture(scope="module")
def env():
    import torch
    yield torch, torch.device("cuda:0"), twd()


def params(t, top_k, rows):
    return [t.RowParams(0.8, 0.95, top_k, 1.0, float(np.float32((0.11 + 0.37 * i) % 1.0)), 0.0, 0, 0)
            for i in range(rows)]


def fill(torch, dev, lg, seed):
    z = (3.0 * np.random.default_rng(seed).standard_normal(tuple(lg.shape))).astype(np.float32)
    lg.copy_(torch.from_numpy(z).to(dev))
    return z


def capture(torch, t, sel, lg, p, tok, mode="global"):
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s, capture_error_mode=mode):
        sel.select(lg, p, tokens=tok, stream=s.cuda_stream)
    torch.cuda.synchronize()
    return g


def replay_and_check(torch, dev, oracle, g, lg, p, tok, seed):
    z = fill(torch, dev, lg, seed)
    tok.zero_()
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    want = [oracle.sample_token(z[i], q.temperature, q.top_p, q.top_k, u=q.uniform) for i, q in enumerate(p)]
    assert (tok.cpu().numpy().astype(np.int64) & 0xFFFFFFFF).tolist() == want, seed


def eager_and_check(torch, dev, oracle, sel, t, top_k, rows, seed):
    lg = torch.empty(rows, V, dtype=torch.float32, device=dev)
    z = fill(torch, dev, lg, seed)
    p = params(t, top_k, rows)
    got = sel.select(lg, p).cpu().numpy().astype(np.int64) & 0xFFFFFFFF
    assert got.tolist() == [oracle.sample_token(z[i], q.temperature, q.top_p, q.top_k, u=q.uniform)
                            for i, q in enumerate(p)], (top_k, rows, seed)


@pytest.mark.parametrize("warm, captured, others", [
    (1000, 1000, [(5000, 2), (300, 2)]),           # another top_k, as many rows
    (1000, 5000, [(1000, 2), (4096, 1)]),          # captured at a longer shortlist than any before
    (5000, 300, [(1000, 5), (5000, 9), (300, 16)]),  # more rows: the scratch grows past the captured one
])
def test_replays_between_other_calls(env, oracle, warm, captured, others):
    torch, dev, t = env
    sel = t.Selector(V, 16)
    eager_and_check(torch, dev, oracle, sel, t, warm, 2, 1)
    lg = torch.zeros(2, V, dtype=torch.float32, device=dev)
    tok = torch.zeros(2, dtype=torch.int32, device=dev)
    p = params(t, captured, 2)
    g = capture(torch, t, sel, lg, p, tok)
    junk = []
    for rep in range(4):
        replay_and_check(torch, dev, oracle, g, lg, p, tok, 10 + rep)
        top_k, rows = others[rep % len(others)]
        eager_and_check(torch, dev, oracle, sel, t, top_k, rows, 20 + rep)
        junk.append(torch.full((1 << 20,), -1, dtype=torch.int64, device=dev))  # over memory that was given back
    for x in junk:
        assert bool((x == -1).all())
    del g
    sel.close()


@pytest.mark.parametrize("top_k", [300, 5000])
def test_first_call_inside_a_capture(env, oracle, top_k):
    # allocation is legal in a relaxed capture; an eager call before the first replay finds the
    # scratch usable, though nothing of the capture has run
    torch, dev, t = env
    sel = t.Selector(V, 16)
    lg = torch.zeros(2, V, dtype=torch.float32, device=dev)
    tok = torch.zeros(2, dtype=torch.int32, device=dev)
    p = params(t, top_k, 2)
    g = capture(torch, t, sel, lg, p, tok, mode="relaxed")
    for rep in range(3):
        eager_and_check(torch, dev, oracle, sel, t, top_k, 2, 30 + rep)
        replay_and_check(torch, dev, oracle, g, lg, p, tok, 40 + rep)
    del g
    sel.close()
