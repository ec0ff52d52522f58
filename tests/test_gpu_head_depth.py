"""The head kernels over depth: heads whose h passes through the streamed kernel's two buffers several
times and whose weights go round the resident kernel's ring, at two and four tiles per wave, and the
logits' error against 64 bits in every form up to 16 rows."""
import ctypes

import numpy as np
import pytest

from helpers import hidden_bf16, twd

pytestmark = pytest.mark.gpu
CAP = 30.0

# rows of the vocabulary and depth: 8, 9 (a padding chunk), 10 and 20 chunks, which are two to five
# windows of four with the last one full or half full; two tiles per wave past 65,536 rows, four past
# 131,072, more than one round of blocks past 262,144
SIZES = [(65_553, 1024), (65_553, 1280), (131_089, 1152), (131_089, 1280), (200_003, 2560), (300_005, 1280)]


def make(seed, V, d):
    """A head of synthetic weights and its [V, d] float64 matrix by blocks of rows."""
    import torch
    t = twd()
    dev = torch.device("cuda:0")
    buf = torch.empty(t.head_bytes(V, d), dtype=torch.uint8, device=dev)
    t.generate_head(buf, V, d, seed)
    head = t.LMHead(buf, V, d, CAP)
    w_bytes, s_bytes = V * d // 2, V * (d // 64) * 2
    W = buf[:w_bytes].view(torch.int32).view(V, d // 8)
    S = buf[w_bytes:w_bytes + s_bytes].view(torch.bfloat16).view(V, d // 64)
    B = buf[w_bytes + s_bytes:].view(torch.bfloat16).view(V, d // 64)
    return torch, dev, t, head, (W, S, B)


def exact(torch, wsb, h):
    """The softcapped logits of float64 rows h [M, d] in 64 bits."""
    W, S, B = wsb
    V, d = W.shape[0], h.shape[1]
    shift = torch.arange(0, 32, 4, dtype=torch.int32, device=W.device)
    out = torch.empty(h.shape[0], V, dtype=torch.float64, device=W.device)
    for r0 in range(0, V, 16384):
        n = min(16384, V - r0)
        q = ((W[r0:r0 + n, :, None] >> shift) & 15).view(n, d // 64, 64)
        w = q.double() * S[r0:r0 + n].double()[..., None] + B[r0:r0 + n].double()[..., None]
        out[:, r0:r0 + n] = torch.mm(h, w.view(n, d).t().contiguous())
    return CAP * torch.tanh(out / CAP)


def bf16_rows(torch, dev, bits):
    return torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).to(dev)


def norm_rows(torch, dev, seed, M, d):
    """x, the norm's weight, and x normalised in 64 bits."""
    rng = np.random.default_rng(seed)
    x = torch.from_numpy((5.0 * rng.standard_normal((M, d))).astype(np.float32)).to(dev)
    w = bf16_rows(torch, dev, hidden_bf16(seed + 1, 1, d)[0])
    xd = x.double()
    return x, w, xd / torch.sqrt(xd.square().mean(1, keepdim=True) + 1e-6) * w.view(torch.bfloat16).double()


def error(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.fixture(scope="module", params=SIZES)
def sized(request):
    V, d = request.param
    made = make(V + d, V, d)
    yield made + (V, d)
    made[3].close()


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_windows_and_rings(sized, oracle, M):
    torch, dev, t, head, wsb, V, d = sized
    h = bf16_rows(torch, dev, hidden_bf16(M + d, M, d))
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    for _ in range(2):  # the second launch finds the finish state as the first left it
        tok = head.greedy(h, logits=logits).cpu().numpy()
    assert torch.equal(head.logits(h).view(torch.int32), logits.view(torch.int32))
    assert error(logits, exact(torch, wsb, h.view(torch.bfloat16).double())) < BOUND
    lg = logits.cpu().numpy()
    assert [int(x) for x in tok] == [int(oracle.argmax(lg[m])) for m in range(M)]


@pytest.mark.parametrize("M", [1, 4, 5, 8])
def test_windows_and_rings_rmsnorm(sized, oracle, M):
    torch, dev, t, head, wsb, V, d = sized
    x, w, h = norm_rows(torch, dev, M + d, M, d)
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    tok = head.greedy_rmsnorm(x, w, 1e-6, logits=logits).cpu().numpy()
    assert error(logits, exact(torch, wsb, h)) < BOUND_NORM
    lg = logits.cpu().numpy()
    assert [int(v) for v in tok] == [int(oracle.argmax(lg[m])) for m in range(M)]


# 2-norm of the logits' error over that of the logits. Every form's sums are fp32, of exact products, in
# another order: 1.4e-6 to 1.9e-6 measured here for bf16 rows, 2.8e-6 to 3.2e-6 with the norm, whose h is
# itself two bf16 halves (2^-18). With the groups' 128 X and their bias summed apart to the end, five rows
# and more lie 3.0e-6 to 7.6e-6 away, and the norm's 4.4e-6 to 6.7e-6: the bounds tell the two apart.
BOUND, BOUND_NORM = 2.5e-6, 3.8e-6


@pytest.fixture(scope="module", params=[32_003, 262_144])
def deep(request):
    made = make(11, request.param, 5376)
    yield made
    made[3].close()


@pytest.mark.parametrize("M", [1, 4, 5, 7, 8, 9, 12, 16])
def test_deep_head_error(deep, oracle, M):
    torch, dev, t, head, wsb = deep
    V, d = wsb[0].shape[0], 5376
    h = bf16_rows(torch, dev, hidden_bf16(40 + M, M, d))
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    tok = head.greedy(h, logits=logits)
    assert error(logits, exact(torch, wsb, h.view(torch.bfloat16).double())) < BOUND
    assert torch.equal(tok.long(), logits.argmax(1))


# at this depth 5 and 6 rows are resident (10 and 12 rows of h in LDS), 7 and 8 stream
@pytest.mark.parametrize("M", [1, 4, 5, 6, 7, 8])
def test_deep_head_error_rmsnorm(deep, oracle, M):
    torch, dev, t, head, wsb = deep
    V, d = wsb[0].shape[0], 5376
    x, w, h = norm_rows(torch, dev, 50 + M, M, d)
    logits = torch.empty(M, V, dtype=torch.float32, device=dev)
    tok = head.greedy_rmsnorm(x, w, 1e-6, logits=logits)
    assert error(logits, exact(torch, wsb, h)) < BOUND_NORM
    assert torch.equal(tok.long(), logits.argmax(1))


@pytest.mark.parametrize("M", [4, 5, 8])
def test_deep_head_sample_and_verify_rmsnorm(deep, oracle, M):
    # 8 rows: prep launch, streamed kernel, then the selection that follows plain logits; 5 rows: the
    # fused pass
    torch, dev, t, head, wsb = deep
    V, d = wsb[0].shape[0], 5376
    x, w, _ = norm_rows(torch, dev, 60 + M, M, d)
    lg = head.logits_rmsnorm(x, w, 1e-6).cpu().numpy()
    arg = [int(oracle.argmax(lg[m])) for m in range(M)]
    drafts = arg[:M - 2] + [(arg[M - 2] + 1) % V]
    res = t.decode_verify(head.verify_greedy_rmsnorm(x, w, torch.tensor(drafts, dtype=torch.int32, device=dev), 1e-6))
    assert res["tokens"] == arg[:M - 1] and res["num_accepted"] == M - 2
    rng = np.random.default_rng(M)
    hist = rng.integers(0, V, M * 64).astype(np.int32)
    prm = [t.RowParams(0.9, 0.95, 40 + m, 1.2, float(np.float32(0.1 + 0.1 * m)), CAP, 64 * m, 64) for m in range(M)]
    tok, got = head.sample_rmsnorm(x, w, prm, history=torch.from_numpy(hist).to(dev))
    tok, got = tok.cpu().numpy(), got.cpu().numpy()
    for m, p in enumerate(prm):
        pen = oracle.apply_repetition_penalty(lg[m], hist[64 * m:64 * m + 64], p.repetition_penalty, CAP)
        assert np.array_equal(got[m].view(np.uint32), pen.view(np.uint32))
        assert int(tok[m]) & 0xFFFFFFFF == oracle.sample_token(pen, p.temperature, p.top_p, p.top_k, u=p.uniform)


def test_greedy_after_group_counters_left_nonzero(oracle):
    # a small head's blocks count in by groups first: what a launch that stopped part-way would leave in
    # their counters, other epochs' counts, all ones and zero
    torch, dev, t, head, wsb = make(5, 32_003, 512)
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    state = t.twd.lib.twd_head_finish_state(head.handle)
    line = 16 * 8  # a counter's line; the launch's counter first, after 64 maxima
    groups = [state + 64 * 8 + line * (1 + g) for g in range(16)]
    h = bf16_rows(torch, dev, hidden_bf16(3, 5, 512))
    want = head.logits(h).argmax(1)
    cur = ctypes.c_uint64()
    for garbage in (lambda e: (7 << 32) | (e - 1), lambda e: (3 << 32) | (e + 1000), lambda e: 2 ** 64 - 1, lambda e: 0):
        assert torch.equal(head.greedy(h).long(), want)
        torch.cuda.synchronize()
        for i, at in enumerate(groups):
            assert hip.hipMemcpy(ctypes.byref(cur), at, 8, 2) == 0
            epoch = cur.value & 0xFFFFFFFF
            assert cur.value >> 32 == 0 and epoch > 0, i  # armed for the next launch
            if i % 3 != 1:  # some groups only
                v = ctypes.c_uint64(garbage(epoch))
                assert hip.hipMemcpy(at, ctypes.byref(v), 8, 1) == 0
        for _ in range(3):
            assert torch.equal(head.greedy(h).long(), want)
    head.close()
