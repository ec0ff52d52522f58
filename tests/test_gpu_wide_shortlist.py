"""Shortlists of 257 to 4,096 entries, finished by one block per row: every way it can go -- records
that bound the shortlist, records too few to (every entry a candidate), the gather overfull, its last
fine bin overfull too (ties), a bin too full to rank by counting, dead entries, prefixes exactly on a
threshold, and the lengths on both sides of its limit. Ids are compared with the oracle's sample_token
on the same row, exactly."""
import numpy as np
import pytest

from helpers import twd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    t = twd()
    sel = t.Selector(262144, 16)
    yield torch, torch.device("cuda:0"), t, sel
    sel.close()


def row_of(kind, n, seed):
    rng = np.random.default_rng(seed)
    z = (3.6 * rng.standard_normal(n)).astype(np.float32)
    if kind == "ties":          # some 40 distinct values
        return (np.round(z * 2) / 2).astype(np.float32)
    if kind == "equal":
        return np.full(n, 1.25, np.float32)
    if kind == "steps":         # three values: the last fine bin holds a third of the row
        return rng.integers(0, 3, n).astype(np.float32)
    if kind == "masked":        # 300 live entries, the rest one large negative number
        out = np.full(n, -1e9, np.float32)
        at = rng.choice(n, min(n, 300), replace=False)
        out[at] = z[at]
        return out
    if kind == "minus_inf":     # 120 live entries, the rest -inf
        out = np.full(n, -np.inf, np.float32)
        at = rng.choice(n, min(n, 120), replace=False)
        out[at] = z[at]
        return out
    if kind == "close":         # a span of a few ulps
        return (np.float32(20.0) + rng.integers(0, 4000, n).astype(np.float32) * np.float32(2e-6)).astype(np.float32)
    if kind == "outlier":       # one value far above: the others share few bins
        z[n // 3] = 500.0
        return z
    return z


KINDS = ["normal", "ties", "equal", "steps", "masked", "minus_inf", "close", "outlier"]


def check(env, oracle, rows, params, V):
    torch, dev, t, sel = env
    lg = torch.from_numpy(np.stack(rows)).to(dev)
    got = sel.select(lg, params).cpu().numpy().astype(np.int64) & 0xFFFFFFFF
    for i, p in enumerate(params):
        want = oracle.sample_token(rows[i], p.temperature, p.top_p, p.top_k, u=p.uniform)
        assert int(got[i]) == want, (V, i, p.top_k, p.top_p, p.temperature)


@pytest.mark.ties
@pytest.mark.parametrize("V", [300, 4097, 8193, 32003, 262144])
@pytest.mark.parametrize("k", [257, 1000, 4095, 4096, 4097])
def test_kinds_of_rows(env, oracle, V, k):
    t = env[2]
    rng = np.random.default_rng(V + k)
    rows, params = [], []
    for i, kind in enumerate(KINDS):
        for p in (0.93, 1.0):
            rows.append(row_of(kind, V, 100 * i + k))
            params.append(t.RowParams(float(rng.choice([0.5, 0.9, 1.7])), p, k, 1.0,
                                      float(np.float32(rng.uniform(0, 0.9999))), 0.0, 0, 0))
    check(env, oracle, rows, params, V)


@pytest.mark.ties
def test_prefixes_on_the_thresholds(env, oracle):
    # equal entries: every weight is 1, so u = j / 2048 puts r exactly on a running sum, and
    # p = i / 4096 of V = 4,096 equal entries puts p on (or an ulp from) a top-p prefix
    t = env[2]
    V = 4096
    rows, params = [], []
    for j in (1, 2, 700, 2047):
        rows.append(row_of("equal", V, 0))
        params.append(t.RowParams(0.7, 1.0, 2048, 1.0, j / 2048, 0.0, 0, 0))
    for i in (1, 3, 512, 1365, 2048):
        rows.append(row_of("equal", V, 0))
        params.append(t.RowParams(0.7, i / 4096, 3000, 1.0, 0.999, 0.0, 0, 0))
    check(env, oracle, rows, params, V)


def test_odd_temperatures_and_draws(env, oracle):
    # NaN and infinite temperatures (weights NaN or 1), u = 0, and rows with a NaN
    torch, dev, t, sel = env
    V = 32003
    rows = [row_of("normal", V, 1), row_of("normal", V, 2), row_of("minus_inf", V, 3), row_of("normal", V, 4)]
    params = [t.RowParams(float("nan"), 0.95, 700, 1.0, 0.3, 0.0, 0, 0),
              t.RowParams(float("inf"), 0.99, 700, 1.0, 0.6, 0.0, 0, 0),
              t.RowParams(float("inf"), 1.0, 700, 1.0, 0.6, 0.0, 0, 0),
              t.RowParams(1.0, 0.9, 700, 1.0, 0.0, 0.0, 0, 0)]
    check(env, oracle, rows, params, V)
    bad = row_of("normal", V, 5)
    bad[7] = np.nan
    tok = sel.select(torch.from_numpy(bad[None]).to(dev), [t.RowParams(1.0, 0.9, 700, 1.0, 0.5, 0.0, 0, 0)])
    assert int(tok.item()) & 0xFFFFFFFF == t.TOKEN_DEGENERATE


@pytest.mark.ties
@pytest.mark.parametrize("V", [100003, 262144, 500000])
@pytest.mark.parametrize("k", [257, 4096])
def test_overfull_lists(env, oracle, V, k):
    # lists gathered again whose last fine bin is overfull too. "deep": that bin holds the whole row, in
    # a thousandth of its range of values, so its counting by parts of the range takes three rounds;
    # "deep_ties": the same over three values, the last round by index; "two" and "zeros": one value,
    # -0 equal to +0
    torch, dev, t, _ = env
    rng = np.random.default_rng(V + k)

    def row(kind):
        if kind == "two":
            return rng.integers(0, 2, V).astype(np.float32)
        if kind == "zeros":
            z = np.where(rng.random(V) < 0.5, np.float32(-0.0), np.float32(0.0)).astype(np.float32)
            z[rng.choice(V, 100, replace=False)] = 3.5
            return z
        low = np.float32(1.0) + (rng.random(V).astype(np.float32) * np.float32(1e-3) if kind == "deep" else
                                 rng.integers(0, 3, V).astype(np.float32) * np.float32(2.0 ** -23))
        z = low.astype(np.float32)
        z[rng.choice(V, 100, replace=False)] = -5.0
        z[V // 3] = 600.0
        return z

    sel = t.Selector(V, 16)
    rows, params = [], []
    for kind in ("two", "zeros", "deep", "deep_ties"):
        for p, temp in ((1.0, 1.7), (0.9, 0.8), (1.0, 500.0)):
            rows.append(row(kind))
            params.append(t.RowParams(temp, p, k, 1.0, float(np.float32(rng.uniform(0, 0.9999))), 0.0, 0, 0))
    check((torch, dev, t, sel), oracle, rows, params, V)
    sel.close()


@pytest.mark.ties
@pytest.mark.parametrize("V", [257, 300, 513, 1500, 3000, 8193])
def test_small_vocabularies_taken_whole(env, oracle, V):
    # shortlists that reach past the records' range, sorted by bins over the list's own: a finite range,
    # an infinite one (-inf entries that a draw of 1 keeps), the widest finite one, equal entries
    t = env[2]
    rows, params = [], []
    for kind in ("normal", "ties", "equal", "minus_inf", "outlier"):
        for u in (0.42, 0.9999, 1.0):
            rows.append(row_of(kind, V, V + len(rows)))
            params.append(t.RowParams(1.1, 0.999, min(V, 4096), 1.0, u, 0.0, 0, 0))
    wide = row_of("normal", V, 5)
    wide[1::3] = np.finfo(np.float32).min
    rows.append(wide)
    params.append(t.RowParams(float("inf"), 1.0, min(V, 4096), 1.0, 0.8, 0.0, 0, 0))
    check(env, oracle, rows, params, V)


@pytest.mark.ties
@pytest.mark.parametrize("V", [50_000, 100_000, 140_001])
def test_overfull_lists_from_the_fused_pass(env, oracle, V):
    # records of 16, 32 and 64 entries; weights of few rows differ from zero, so nearly all logits are equal
    torch, dev, t, _ = env
    d = 128
    W = np.zeros((V, d // 8), np.uint32)
    S = np.full((V, d // 64), 0x3F80, np.uint16)  # 1.0
    B = np.zeros((V, d // 64), np.uint16)
    rng = np.random.default_rng(V)
    some = rng.choice(V, 40, replace=False)
    W[some] = rng.integers(0, 2 ** 32, (40, d // 8), dtype=np.uint64).astype(np.uint32)
    wsb = np.concatenate([W.reshape(-1).view(np.uint8), S.reshape(-1).view(np.uint8), B.reshape(-1).view(np.uint8)])
    head = t.LMHead(torch.from_numpy(wsb).to(dev), V, d, 30.0)
    bits = np.full((3, d), 0x3C00, np.uint16)  # 2^-7
    bits[1] = 0xBC00  # -2^-7: the 40 rows lie below the others
    h = torch.from_numpy(bits.view(np.int16)).to(dev)
    prm = [t.RowParams(0.9, 0.97, k, 1.0, u, 30.0, 0, 0) for k, u in ((300, 0.7), (1000, 0.31), (4096, 0.999))]
    tok, lg = head.sample(h, prm)
    tok, lg = tok.cpu().numpy(), lg.cpu().numpy()
    for m, p in enumerate(prm):
        assert int(tok[m]) & 0xFFFFFFFF == oracle.sample_token(lg[m], p.temperature, p.top_p, p.top_k, u=p.uniform)
    head.close()
