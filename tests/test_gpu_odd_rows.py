"""The record pass on rows that start at any float's address: odd vocabularies, odd strides and a base
pointer off 16 bytes, with and without the record words (few rows, long shortlists). Tokens are
compared with the oracle's sample_token on the same rows, exactly. Also the vocabularies at which the
merge changes the number of records that a thread holds."""
import numpy as np
import pytest

from helpers import twd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,pad,off", [(5003, 0, 0), (5003, 2, 1), (4099, 1, 3), (2050, 0, 2), (64, 3, 1), (63, 0, 3)])
@pytest.mark.parametrize("rows,k", [(3, 40), (11, 40), (11, 0)])
def test_rows_at_any_alignment(oracle, V, pad, off, rows, k):
    import torch
    t = twd()
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(V + rows + k)
    x = (3.0 * rng.standard_normal((rows, V))).astype(np.float32)
    buf = torch.full((off + rows * (V + pad),), float("nan"), dtype=torch.float32, device=dev)
    lg = buf[off:].view(rows, V + pad)[:, :V]
    lg.copy_(torch.from_numpy(x))
    sel = t.Selector(V, rows)
    prm = [t.RowParams(0.8, 0.9 if m % 2 else 1.0, k, 1.0, float(np.float32(rng.uniform(0, 0.999))), 0.0, 0, 0)
           for m in range(rows)]
    got = sel.select(lg, prm).cpu().numpy().astype(np.int64) & 0xFFFFFFFF
    sel.close()
    want = [oracle.sample_token(x[m], p.temperature, p.top_p, p.top_k, u=p.uniform) for m, p in enumerate(prm)]
    assert got.tolist() == want


# records of 64 entries, 1,024 threads: 1, 2, 4 and 8 records a thread up to these sizes and past them
@pytest.mark.parametrize("V", [65536, 65537, 131072, 131073, 262144, 262145])
@pytest.mark.parametrize("rows,k", [(2, 40), (9, 0)])
def test_rows_where_a_thread_takes_more_records(oracle, V, rows, k):
    import torch
    t = twd()
    rng = np.random.default_rng(V + rows)
    x = (3.0 * rng.standard_normal((rows, V))).astype(np.float32)
    x[:, -1] += 9.0  # the last record's entry among the likely ones
    prm = [t.RowParams(0.8 if m else 0.0, 0.95 if m % 2 else 1.0, k, 1.0, float(np.float32(rng.uniform(0, 0.999))),
                       0.0, 0, 0) for m in range(rows)]
    sel = t.Selector(V, rows)
    got = sel.select(torch.from_numpy(x).cuda(), prm).cpu().numpy().astype(np.int64) & 0xFFFFFFFF
    sel.close()
    want = [oracle.sample_token(x[m], p.temperature, p.top_p, p.top_k, u=p.uniform) for m, p in enumerate(prm)]
    assert got.tolist() == want


# both sides of the record words' line for many rows: shortlists of mean 128 and 256, and mixed ones
@pytest.mark.parametrize("V,rows", [(32003, 9), (262144, 48)])
@pytest.mark.parametrize("ks", [(127,), (128,), (256,), (40, 250, 1)])
def test_many_rows_with_and_without_words(oracle, V, rows, ks):
    import torch
    t = twd()
    rng = np.random.default_rng(V + rows + sum(ks))
    x = (3.0 * rng.standard_normal((rows, V))).astype(np.float32)
    prm = [t.RowParams(0.8, 0.97 if m % 2 else 1.0, ks[m % len(ks)], 1.0, float(np.float32(rng.uniform(0, 0.999))),
                       0.0, 0, 0) for m in range(rows)]
    sel = t.Selector(V, rows)
    got = sel.select(torch.from_numpy(x).cuda(), prm).cpu().numpy().astype(np.int64) & 0xFFFFFFFF
    sel.close()
    want = [oracle.sample_token(x[m], p.temperature, p.top_p, p.top_k, u=p.uniform) for m, p in enumerate(prm)]
    assert got.tolist() == want
