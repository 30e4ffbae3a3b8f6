"""Rows split over workgroups (nls_rowsplit.hip): softmaxInPlace, logProb,
topTokens and perplexity's term at the sizes where the split starts and ends,
on rows whose running sum is hard to predict or to keep, against the oracle
and against the one-launch kernels (the same calls without a workspace)."""
import ctypes
import math
import sys

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def torch():
    import torch

    assert torch.cuda.is_available(), "no GPU"
    return torch


def _rows(V, seed):
    """Named rows of V logits."""
    rng = np.random.default_rng(seed)
    f = np.float32
    n = rng.standard_normal(V)
    r = {
        "normal": n * 2.5,
        "wide": n * 12.0,                                      # terms down to e^-104 and zeros
        "quarter steps": np.round(n * 8) / 4,                  # many equal values
        "equal": np.full(V, 1.75),                             # every term 1: all ties and crossings exact
        "first half -inf": np.where(np.arange(V) < V // 2, -np.inf, n * 2),
        "every other -inf": np.where(np.arange(V) % 2 == 0, -np.inf, n),
        "largest last": np.where(np.arange(V) == V - 1, 70.0, n),   # tiny sums until the end
        "largest last, far": np.where(np.arange(V) == V - 1, 100.0, n * 3),
        "largest first": np.where(np.arange(V) == 0, 14.0, n),
        "just below 2": np.where(np.arange(V) == 0, 0.0, np.log((1.0 - 2.0**-20) / V)),
        "ties of 1": np.where(np.arange(V) == 0, 0.0, -24 * math.log(2.0)),  # about u / 2 each
        "falling": -np.arange(V) * (100.0 / V),
        "rising": np.arange(V) * (100.0 / V),
        "small": n * 1e-3,                                     # probabilities tied by rounding
    }
    x = n.copy()
    x[V // 2] = np.nan
    r["NaN inside"] = x
    x = np.where(np.arange(V) < V // 2, -np.inf, n)
    x[V // 4] = np.nan
    r["NaN among -inf"] = x
    x = n.copy()
    x[V // 3] = np.inf
    r["+inf inside"] = x
    r["all -inf"] = np.full(V, -np.inf)
    return list(r), np.stack([v.astype(f) for v in r.values()])


# below the split, its first size, ragged sizes, whole and nearly whole slices,
# real vocabularies, the last size of the split and the first past it
SIZES = [8191, 8192, 8193, 12287, 12288, 12289, 50001, 128256, 151936, 1 << 20, (1 << 20) + 1]


@pytest.mark.parametrize("V", SIZES)
def test_split_rows(pkg, torch, V):
    names, x = _rows(V, V)
    if V > 200000:
        keep = [0, 3, 6, 9, 14]
        names, x = [names[i] for i in keep], x[keep]
    R = len(names)
    say(f"[rowsplit] V={V}, {R} rows")
    big = torch.empty(R * V + 1, device="cuda")
    t = np.random.default_rng(V + 1).integers(0, V, size=R).astype(np.int32)
    t[0] = int(np.argmax(x[0]))
    dt = torch.from_numpy(t).cuda()
    vp = ctypes.c_void_p
    for off in (0, 1):  # rows on 16 bytes where V allows it, and 4 bytes past
        d = big[off:off + R * V].view(R, V)
        d.copy_(torch.from_numpy(x))
        say(f"  offset {off}: softmax")
        sm = pkg.softmax_device(d).cpu().numpy()
        d2 = d if off else d.clone()
        prob, logp = (q.cpu().numpy() for q in pkg.log_prob_device(d, dt))
        nll = pkg.row_nll_device(d, dt).cpu().numpy()
        tops = {n: [q.cpu().numpy() for q in pkg.top_tokens_device(d, n)] for n in (1, 5, 20, 64)}
        one = torch.empty(R, V, device="cuda")
        pkg.check(pkg.lib().nls_softmax_rows(vp(d.data_ptr()), R, V, vp(one.data_ptr()), None), "one launch")
        torch.cuda.synchronize()
        one = one.cpu().numpy()
        in_place = pkg.softmax_device(d2, out=d2).cpu().numpy()
        for i, name in enumerate(names):
            want = O.softmax(x[i])
            nan = np.isnan(want)
            for got in (sm[i], one[i], in_place[i]):
                assert np.array_equal(np.isnan(got), nan), (V, off, name)
                bad = np.flatnonzero(got.view(np.uint32)[~nan] != want.view(np.uint32)[~nan])
                assert bad.size == 0, (V, off, name, bad[:4], got[~nan][bad[:4]], want[~nan][bad[:4]])
            wp = want[t[i]]
            assert (prob[i] == wp) or (np.isnan(wp) and np.isnan(prob[i])), (V, off, name, prob[i], wp)
            if wp > 0:
                # the device's float64 log: within 1 ulp of the C library's
                assert abs(logp[i] - math.log(float(wp))) <= 2 * np.spacing(abs(math.log(float(wp)))), (V, off, name)
            ref = O.row_nll(x[i], int(t[i]))
            if math.isfinite(ref):
                # (pairwise sums: the oracle's own, in index order, may be V 2^-53 off)
                d64 = (x[i] - np.fmax.reduce(x[i])).astype(np.float64)
                ref = math.log(float(np.exp(d64).sum())) - float(d64[t[i]])
                # trees over 2^20 terms: 20 + 2 roundings of 2^-53, the exponential and log a few ulps each
                assert abs(nll[i] - ref) <= 1e-12 * max(1.0, abs(ref)), (V, off, name, nll[i], ref)
            else:
                assert nll[i] == ref or (np.isnan(nll[i]) and np.isnan(ref)), (V, off, name, nll[i], ref)
            if nan.any():
                continue  # no order among NaN probabilities
            order = np.argsort(-want, kind="stable")
            for n, (ids, pr) in tops.items():
                m = min(n, V)
                assert np.array_equal(ids[i], order[:m]), (V, off, name, n, ids[i][:8], order[:8])
                assert np.array_equal(pr[i], want[order[:m]]), (V, off, name, n)


def test_split_in_a_graph(pkg, torch):
    """The split calls captured once and replayed on changing logits, with
    eager calls between the replays."""
    R, V = 3, 50001
    say("[rowsplit] captured")
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(R, V, generator=g, device="cuda")
    t = torch.zeros(R, dtype=torch.int32, device="cuda")

    def calls():
        return [pkg.softmax_device(x), *pkg.log_prob_device(x, t), pkg.row_nll_device(x, t),
                *pkg.top_tokens_device(x, 5)]

    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = calls()
    for k in range(4):
        x.copy_(torch.randn(R, V, generator=g, device="cuda") * (1 + k))
        t.fill_(7 * k)
        want = [q.clone() for q in calls()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b), k


def test_workspace_rule(pkg):
    """A short, odd or missing workspace runs the one-launch kernels; the
    sizes the split covers ask for one."""
    L = pkg.lib()
    assert L.nls_rows_workspace(1, 4, 8191, 0) == 0
    assert L.nls_rows_workspace(1, 4, 8192, 0) > 0
    assert [L.nls_rows_workspace(0, r, v, 0) > 0 for r, v in
            [(4, 12287), (4, 12288), (193, 12288), (256, 14336), (257, 8192)]] == [False, True, False, True, True]
    assert [L.nls_rows_workspace(3, r, v, 0) > 0 for r, v in
            [(4, 40959), (4, 40960), (160, 50000), (161, 50000)]] == [False, True, True, False]
    assert L.nls_rows_workspace(2, 4, 8192, 33) == 0
    assert L.nls_rows_workspace(2, 4, 8192, 32) > L.nls_rows_workspace(1, 4, 8192, 0)
    assert L.nls_rows_workspace(0, 0, 8192, 0) == 0
    assert L.nls_rows_workspace(0, 1, (1 << 20) + 1, 0) == 0
    assert L.nls_rows_workspace(9, 1, 50000, 0) == 0
