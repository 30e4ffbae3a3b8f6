"""Rows split over workgroups (nls_rowsplit.hip): softmaxInPlace, logProb,
topTokens and perplexity's term at the sizes where the split starts and ends,
on rows whose running sum is hard to predict or to keep, against the oracle
and against the one-launch kernels (the same calls without a workspace); the
workspace's bounds."""
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


def _one_launch(pkg, torch, d, targets, ns=(1, 5, 20, 64)):
    """log_prob, row_nll and top_tokens of d by the calls without a workspace."""
    R, V = d.shape
    L = pkg.lib()

    def p(q):
        return ctypes.c_void_p(q.data_ptr())

    prob, logp = torch.empty(R, device="cuda"), torch.empty(R, dtype=torch.float64, device="cuda")
    pkg.check(L.nls_log_prob(p(d), R, V, p(targets), p(prob), p(logp), None), "nls_log_prob")
    nll = torch.empty(R, dtype=torch.float64, device="cuda")
    pkg.check(L.nls_row_nll(p(d), R, V, p(targets), p(nll), None), "nls_row_nll")
    tops = {}
    for n in ns:
        ids, pr = torch.empty(R, n, dtype=torch.int32, device="cuda"), torch.empty(R, n, device="cuda")
        pkg.check(L.nls_top_tokens(p(d), R, V, n, p(ids), p(pr), None), "nls_top_tokens")
        tops[n] = (ids, pr)
    torch.cuda.synchronize()
    return prob, logp, nll, tops


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
        one = one.cpu().numpy()
        # the same calls without a workspace: the one-launch kernels
        prob1, logp1, nll1, tops1 = (q.cpu().numpy() if torch.is_tensor(q) else
                                     {n: [w.cpu().numpy() for w in p] for n, p in q.items()}
                                     for q in _one_launch(pkg, torch, d, dt))
        in_place = pkg.softmax_device(d2, out=d2).cpu().numpy()
        for i, name in enumerate(names):
            want = O.softmax(x[i])
            nan = np.isnan(want)
            for got in (sm[i], one[i], in_place[i]):
                assert np.array_equal(np.isnan(got), nan), (V, off, name)
                bad = np.flatnonzero(got.view(np.uint32)[~nan] != want.view(np.uint32)[~nan])
                assert bad.size == 0, (V, off, name, bad[:4], got[~nan][bad[:4]], want[~nan][bad[:4]])
            wp = want[t[i]]
            for pr, lp in ((prob, logp), (prob1, logp1)):
                assert (pr[i] == wp) or (np.isnan(wp) and np.isnan(pr[i])), (V, off, name, pr[i], wp)
                if wp > 0:
                    # the device's float64 log: within 1 ulp of the C library's
                    assert abs(lp[i] - math.log(float(wp))) <= 2 * np.spacing(abs(math.log(float(wp)))), (V, off, name)
            assert nll[i] == nll1[i] or (np.isnan(nll[i]) and np.isnan(nll1[i])), (V, off, name, nll[i], nll1[i])
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
            for n, (ids, pr) in [*tops.items(), *tops1.items()]:
                m = min(n, V)
                assert np.array_equal(ids[i], order[:m]), (V, off, name, n, ids[i][:8], order[:8])
                assert np.array_equal(pr[i], want[order[:m]]), (V, off, name, n)


@pytest.mark.parametrize("V", [12288, 50001, 131072])
def test_nan_rows_as_in_one_launch(pkg, torch, V):
    """Rows with NaN or infinite logits, NaNs of any sign and payload: every
    output is the one-launch kernels', bit for bit (topTokens orders NaN
    probabilities by their bits, so the sum's own NaN decides its ids)."""
    rng = np.random.default_rng(V + 9)
    nans = np.array([0x7FC00000, 0xFFC00000, 0x7FC00123, 0xFFC00123, 0x7F800001, 0xFF800007], np.uint32)
    rows = []
    for i in range(18):
        x = rng.standard_normal(V).astype(np.float32)
        k = [1, 2, 60, 400][i % 4]
        x.view(np.uint32)[rng.choice(V, k, replace=False)] = nans[i % 6] if i < 6 else rng.choice(nans, k)
        if i % 5 == 4:
            x[rng.integers(0, V, size=3)] = np.inf
        rows.append(x)
    for at in (0, 1023, 1024, V - 1):  # the edges of the 1024 logits a wave sums
        x = rng.standard_normal(V).astype(np.float32)
        x.view(np.uint32)[at] = 0xFFC00123
        rows.append(x)
    x = rng.standard_normal(V).astype(np.float32)
    x[V // 2] = np.inf
    rows.append(x)
    x = np.full(V, -np.inf, np.float32)
    x.view(np.uint32)[V // 2] = 0x7FC00123
    rows += [x, np.full(V, -np.inf, np.float32), np.full(V, np.inf, np.float32)]
    R = len(rows)
    say(f"[rowsplit] NaN rows V={V}, {R} rows")
    d = torch.from_numpy(np.stack(rows)).cuda()
    t = torch.from_numpy(rng.integers(0, V, size=R).astype(np.int32)).cuda()
    vp = ctypes.c_void_p
    L = pkg.lib()

    def p(q):
        return vp(q.data_ptr())

    sm = torch.empty(R, V, device="cuda")
    pkg.check(L.nls_softmax_rows(p(d), R, V, p(sm), None), "one launch")
    prob = torch.empty(R, device="cuda")
    logp = torch.empty(R, dtype=torch.float64, device="cuda")
    pkg.check(L.nls_log_prob(p(d), R, V, p(t), p(prob), p(logp), None), "one launch")
    got = pkg.log_prob_device(d, t)
    for g, w in ((pkg.softmax_device(d), sm), (got[0], prob)):
        bad = (g.view(torch.int32) != w.view(torch.int32)).reshape(R, -1).any(1).nonzero().reshape(-1).tolist()
        assert not bad, (V, bad)
    assert torch.equal(got[1].view(torch.int64), logp.view(torch.int64))
    for n in (1, 5, 48):
        ids = torch.empty(R, n, dtype=torch.int32, device="cuda")
        pr = torch.empty(R, n, device="cuda")
        pkg.check(L.nls_top_tokens(p(d), R, V, n, p(ids), p(pr), None), "one launch")
        gi, gp = pkg.top_tokens_device(d, n)
        assert torch.equal(gi, ids), (V, n, (gi != ids).any(1).nonzero().reshape(-1).tolist())
        assert torch.equal(gp.view(torch.int32), pr.view(torch.int32)), (V, n)


@pytest.mark.parametrize("V", [14337, 50001])
def test_softmax_of_masked_and_vanishing_terms(pkg, torch, V):
    """Terms around e^-104 (the last nonzero float32 exponential), subnormal
    quotients and masked logits (-inf, the lowest float), in runs and
    scattered: softmax against the oracle, bit for bit."""
    rng = np.random.default_rng(V)
    base = rng.standard_normal(V) * 2
    edge = rng.uniform(-104.5, -103.5, size=V)
    edge[::7] = -104.0
    edge[1::7] = np.nextafter(np.float32(-104), np.float32(0))
    rows = [np.where(rng.random(V) < 0.99, -np.inf, base), np.where(rng.random(V) < 0.99, -3.4028234663852886e38, base),
            np.where(np.arange(V) % 512 < 256, -np.inf, base), edge, rng.uniform(-106.0, -80.0, size=V),
            np.where(rng.random(V) < 0.5, edge, -np.inf), rng.uniform(-90.0, -86.0, size=V)]
    x = np.stack(rows).astype(np.float32)
    x[3:, 5] = 0.0
    x[4:, 11] = 0.5
    say(f"[rowsplit] masked V={V}")
    got = pkg.softmax_device(torch.from_numpy(x).cuda()).cpu().numpy()
    for r in range(len(x)):
        want = O.softmax(x[r])
        bad = np.flatnonzero(got[r].view(np.uint32) != want.view(np.uint32))
        assert bad.size == 0, (V, r, bad[:4], got[r][bad[:4]], want[bad[:4]], x[r][bad[:4]])


@pytest.mark.parametrize("V", [8192, 50001, 128256])
def test_top_tokens_list_of_rows_in_order(pkg, torch, V):
    """Rows whose largest logits lie side by side (rising, falling, in blocks)
    list few logits for topTokens' last launch, not thousands that would
    overflow the list; ids and probabilities against the oracle."""
    i = np.arange(V)
    rng = np.random.default_rng(V)
    n = rng.standard_normal(V)
    x = np.stack([-i * (20.0 / V), i * (20.0 / V), -np.abs(i - V // 2) * (20.0 / V), np.sort(n), -np.sort(n),
                  np.where((i > 3000) & (i < 4400), 9.0 + n / 8, n)]).astype(np.float32)
    R = len(x)
    say(f"[rowsplit] rows in order V={V}")
    d = torch.from_numpy(x).cuda()
    vp = ctypes.c_void_p
    L = pkg.lib()
    for m in (1, 5, 20, 32, 64):
        if m > V // 256:
            continue
        need = L.nls_rows_workspace(2, R, V, m)
        work = torch.zeros(need, dtype=torch.uint8, device="cuda")
        ids = torch.empty(R, m, dtype=torch.int32, device="cuda")
        pr = torch.empty(R, m, device="cuda")
        pkg.check(L.nls_top_tokens_ws(vp(d.data_ptr()), R, V, m, vp(ids.data_ptr()), vp(pr.data_ptr()),
                                      vp(work.data_ptr()), need, None), "nls_top_tokens_ws")
        torch.cuda.synchronize()
        # a row's record: two floats, the list's bound and its count, in 32 bytes
        count = work[:R * 32].view(torch.int32).view(R, 8)[:, 3].cpu().numpy()
        assert (count >= m).all() and (count <= (1024 if m <= 32 else 2048)).all(), (V, m, count)
        for r in range(R):
            want = O.softmax(x[r])
            order = np.argsort(-want, kind="stable")[:m]
            assert np.array_equal(ids[r].cpu().numpy(), order), (V, m, r)
            assert np.array_equal(pr[r].cpu().numpy(), want[order]), (V, m, r)


@pytest.mark.parametrize("V", [40960, 40961, 50000, 50001, 65537, 128256, 131072, 1 << 20])
def test_row_nll_has_one_sum(pkg, torch, V):
    """perplexity's term is the same to the bit with and without a workspace,
    so it does not depend on how many positions are scored together: full and
    ragged chunks, on 16 bytes and 4 past, every kind of row."""
    names, x = _rows(V, V + 1)
    R = len(names)
    say(f"[rowsplit] row_nll V={V}, {R} rows")
    big = torch.empty(R * V + 1, device="cuda")
    t = torch.from_numpy(np.random.default_rng(V).integers(0, V, size=R).astype(np.int32)).cuda()
    t[1] = -1
    t[2] = V
    vp = ctypes.c_void_p
    for off in (0, 1):
        d = big[off:off + R * V].view(R, V)
        d.copy_(torch.from_numpy(x))
        got = pkg.row_nll_device(d, t)
        one = torch.empty(R, dtype=torch.float64, device="cuda")
        pkg.check(pkg.lib().nls_row_nll(vp(d.data_ptr()), R, V, vp(t.data_ptr()), vp(one.data_ptr()), None), "one launch")
        same = (got.view(torch.int64) == one.view(torch.int64)) | (got.isnan() & one.isnan())
        assert same.all(), (V, off, [names[i] for i in (~same).nonzero().reshape(-1).tolist()])


def test_row_nll_of_many_long_rows(pkg, torch):
    """More rows than the split takes, at a real vocabulary: float64 terms
    against numpy's, within the roundings of a tree over 2^17 terms."""
    R, V = 170, 128256
    say(f"[rowsplit] row_nll {R} x {V}")
    rng = np.random.default_rng(11)
    x = (rng.standard_normal((R, V), dtype=np.float32) * np.float32(2.5))
    x[3, ::2] = -np.inf
    x[4] = 1.5
    t = rng.integers(0, V, size=R).astype(np.int32)
    t[3] = 5
    assert pkg.lib().nls_rows_workspace(3, R, V, 0) == 0
    got = pkg.row_nll_device(torch.from_numpy(x).cuda(), torch.from_numpy(t)).cpu().numpy()
    for r in range(R):
        d = (x[r] - x[r].max()).astype(np.float64)
        ref = math.log(float(np.exp(d).sum())) - float(d[t[r]])
        assert abs(got[r] - ref) <= 1e-12 * max(1.0, abs(ref)), (r, got[r], ref)


def test_row_nll_of_any_number_of_rows(pkg, torch):
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(200, 50001, generator=g, device="cuda") * 3
    t = torch.randint(0, 50001, (200,), generator=g, device="cuda", dtype=torch.int32)
    want = pkg.row_nll_device(x, t)
    for k in (1, 7, 160, 161):
        assert torch.equal(pkg.row_nll_device(x[:k], t[:k]), want[:k]), k


def test_every_form_of_the_exponential(pkg, torch):
    """The quick form (where it holds) and the estimate's bound on every float32
    from -0 down to -inf, against the exact exponential."""
    say("[rowsplit] forms of the exponential: 2.1e9 inputs")
    L = pkg.lib()
    step = 1 << 28
    for a in range(0x80000000, 0xFF800001, step):
        b = min(a + step, 0xFF800001)
        x = (torch.arange(a - (1 << 32), b - (1 << 32), dtype=torch.int64, device="cuda").to(torch.int32)).view(torch.float32)
        want = pkg.expf_device(x)
        got = torch.empty_like(x)
        vp = ctypes.c_void_p
        pkg.check(L.nls_expf_forms_device(vp(x.data_ptr()), vp(got.data_ptr()), x.numel(), None), "forms")
        assert torch.equal(got.view(torch.int32), want.view(torch.int32)), hex(a)


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


def test_no_room_for_a_workspace(pkg, torch):
    """A call whose workspace the memory has no room for runs without one, as it
    did before there was one (the limit is torch's own, set just above what it
    holds)."""
    x = torch.randn(4096, 8192, device="cuda")
    want = pkg.top_tokens_device(x, 5)
    need = pkg.lib().nls_rows_workspace(2, 4096, 8192, 5)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    room = need // 2
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / total)
    say(f"[rowsplit] no room: {need} bytes wanted, {room} left")
    try:
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device="cuda")
        got = pkg.top_tokens_device(x, 5)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_short_rows_ask_for_no_workspace(pkg):
    """The lengths below which the Python entry points don't ask for a
    workspace are the library's: none wanted there, one wanted from there on."""
    L = pkg.lib()
    for op, start in pkg._ROWS_WORK_FROM.items():
        rows = 300 if op == pkg._ROWS_SOFTMAX else 4  # (softmax of few rows splits from 12288 on)
        assert L.nls_rows_workspace(op, rows, start, 1) > 0, op
        for r in (1, 4, 160, 300, 5000):
            assert not any(L.nls_rows_workspace(op, r, v, 1) for v in range(1, start, 127)), (op, r)
            assert L.nls_rows_workspace(op, r, start - 1, 1) == 0, (op, r)


@pytest.mark.parametrize("op", ["softmax", "log_prob", "top_tokens", "row_nll"])
def test_workspace_contract(pkg, torch, op):
    """A call writes no byte past the workspace it asked for, and none at all
    into one that is a byte short, off 16 bytes, or missing: the same results
    either way."""
    R, V, n = 3, 50001, 7
    L, vp = pkg.lib(), ctypes.c_void_p
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(R, V, generator=g, device="cuda") * 3
    t = torch.tensor([5, V - 1, 77], dtype=torch.int32, device="cuda")
    code = ["softmax", "log_prob", "top_tokens", "row_nll"].index(op)
    need = L.nls_rows_workspace(code, R, V, n)
    assert need > 0
    say(f"[rowsplit] workspace of {op}: {need} bytes")

    def p(q):
        return vp(q.data_ptr())

    def call(work, size):
        if op == "softmax":
            outs = [torch.zeros(R, V, device="cuda")]
            rc = L.nls_softmax_rows_ws(p(x), R, V, p(outs[0]), work, size, None)
        elif op == "log_prob":
            outs = [torch.zeros(R, device="cuda"), torch.zeros(R, dtype=torch.float64, device="cuda")]
            rc = L.nls_log_prob_ws(p(x), R, V, p(t), p(outs[0]), p(outs[1]), work, size, None)
        elif op == "top_tokens":
            outs = [torch.zeros(R, n, dtype=torch.int32, device="cuda"), torch.zeros(R, n, device="cuda")]
            rc = L.nls_top_tokens_ws(p(x), R, V, n, p(outs[0]), p(outs[1]), work, size, None)
        else:
            outs = [torch.zeros(R, dtype=torch.float64, device="cuda")]
            rc = L.nls_row_nll_ws(p(x), R, V, p(t), p(outs[0]), work, size, None)
        assert rc == 0
        torch.cuda.synchronize()
        return outs

    guard = 4096
    buf = torch.full((guard + need + guard,), 0xAB, dtype=torch.uint8, device="cuda")
    at = buf.data_ptr() + guard
    want = call(None, 0)
    for work, size in ((at, need - 1), (at + 8, need), (at, 0), (None, need)):
        for a, b in zip(call(vp(work) if work else None, size), want):
            assert torch.equal(a, b), (op, work, size)
        assert (buf == 0xAB).all(), (op, work, size)
    for a, b in zip(call(vp(at), need), want):
        assert torch.equal(a, b), op
    assert (buf[:guard] == 0xAB).all() and (buf[guard + need:] == 0xAB).all(), op
    assert (buf[guard:guard + need] != 0xAB).any(), op  # the split ran


def test_workspace_rule(pkg):
    """The sizes the split covers ask for a workspace, the others for none."""
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
