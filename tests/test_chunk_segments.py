"""Prompt portions by the workgroups that take all columns of a head, long ones in segments (dgi/csrc/mix/chunk_segments.h), against a token loop in
64 bits: many heads (whole portions: lengths around a chunk and a pair of them, no rows at all), few heads (segments), one long portion beside decode rows of
more sequences than a wave has lanes, sizes around the column blocks; gates and values that send chunks token by token.

Tolerance: as test_chunk_scan.py's: sums of a few hundred products of factors with some 16 roundings each, 3e-5 of the largest."""
import pytest
import torch

import test_chunk_scan as base
from dgi.ops import linrec
from test_chunk_parts import where_finite
from test_scan_precision import compare, in_short_portions, of_kind

F64 = torch.float64
pytestmark = pytest.mark.gpu
EDGES = [63, 64, 65, 33, 31, 0, 1, 97, 300]
MIXED = [1] * 40 + [700] + [2] * 30 + [150, 17]
MANY = [1] * 500 + [700] + [2] * 30 + [1900, 17] + [1] * 600 + [300, 40, 0]      # more sequences than a workgroup has threads


def make(mode, lens, H, D, V, dtype, strong=False):
    d = base.make(mode if mode == "mlstm" else "light", lens, H, D, V, dtype, [3 * (i % 2) for i in range(len(lens))])
    d["mode"] = mode
    if mode == "gla":
        a = torch.sigmoid(torch.randn(sum(lens), H * D, generator=torch.Generator().manual_seed(5)) + 2) ** (1 / 16)
        if strong:                                               # products of 1e-20 within some chunks, a zero, one that grows and shrinks again
            a[40:60] *= 0.1
            a[100, 1], a[200, 2], a[201, 2] = 0., 1e18, 1e-18
        d["decay"] = a.float()
    elif strong:
        if mode == "mlstm":
            # an output's error is 1e-6 of the sum of |n q| over |n . q|, which with gates of e^15 nothing but n . q itself bounds: of one sign it is that sum
            d["q"], d["k"] = d["q"].abs(), d["k"].abs()
            d["a"][40:60] = 1e4
            d["b"][90:95] = -1e4
            d["a"][150] = float("-inf")
        else:
            d["par"] = (torch.linspace(0, 1, H),)
    return d


def call(d):
    if d["mode"] != "gla":
        return base.call(d)
    lens, H, D, V = d["lens"], d["H"], d["D"], d["V"]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()  # noqa: E731
    S = d["S"].clone().cuda()
    y = linrec.gla_scan(d["q"].cuda(), d["k"].cuda(), d["v"].cuda(), d["decay"].cuda(), S, i32([p + t for p, m in zip(d["past"], lens) for t in range(m)]),
                        i32([sum(lens[:i]) for i in range(len(lens) + 1)]), i32(list(range(len(lens), 0, -1))), H, D, V)
    return y.cpu(), S.cpu()


def oracle(d):
    if d["mode"] != "gla":
        return base.oracle(d)
    lens, H, D, V = d["lens"], d["H"], d["D"], d["V"]
    S, T, at = d["S"].to(F64), sum(d["lens"]), 0
    q, k, v, a = (d[x].to(F64).reshape(T, H, -1) for x in ("q", "k", "v", "decay"))
    y = torch.zeros(T, H, V, dtype=F64)
    for i, ln in enumerate(lens):
        s = S[len(lens) - i] * (1. if d["past"][i] > 0 else 0.)
        for t in range(at, at + ln):
            s = a[t][:, :, None] * s + k[t][:, :, None] * v[t][:, None, :]
            y[t] = (q[t][:, :, None] * s).sum(1) * D ** -0.5
        if ln:
            S[len(lens) - i] = s
        at += ln
    return y.reshape(T, -1), S


@pytest.mark.parametrize("mode", ["gla", "light", "mlstm"])
@pytest.mark.parametrize("lens,H,D,V,dtype", [
    (EDGES, 32, 64, 64, torch.bfloat16), (EDGES, 32, 48, 40, torch.float32), (EDGES, 16, 100, 128, torch.bfloat16), (EDGES, 16, 128, 72, torch.float32),
    ([1500], 6, 64, 64, torch.bfloat16), ([850, 1900], 3, 64, 100, torch.float32), ([1300, 40], 5, 128, 128, torch.bfloat16), ([1700], 4, 128, 48, torch.float32),
    (MIXED, 8, 64, 64, torch.bfloat16), (MIXED, 4, 64, 128, torch.float32), (MANY, 4, 48, 64, torch.bfloat16)], ids=lambda x: "x".join(map(str, x))[:12] if isinstance(x, list) else str(x))
def test_portions(mode, lens, H, D, V, dtype):
    d = make(mode, lens, H, D, V, dtype)
    got, want = call(d), oracle(d)
    has_rows = torch.tensor([0] + [int(n > 0) for n in reversed(lens)], dtype=torch.bool)
    base.check(got[:1] + tuple(x[has_rows] for x in got[1:]), want[:1] + tuple(x[has_rows] for x in want[1:]))
    assert torch.equal(got[1][~has_rows], d["S"][~has_rows])


@pytest.mark.parametrize("mode", ["gla", "light", "mlstm"])
@pytest.mark.parametrize("lens,H", [([1500], 6), ([70, 250], 96)], ids=["segments", "whole"])
def test_strong_gates(mode, lens, H):
    """Decays whose inverses leave fp32 and gates beyond any range: those chunks go token by token, within a segment and among the states between them."""
    d = make(mode, lens, H, 64, 64, torch.float32, strong=True)
    base.check(call(d), oracle(d))


@pytest.mark.parametrize("mode", ["gla", "light", "mlstm"])
def test_non_finite_values_stay_behind(mode):
    """An infinity, NaN or value too large for its parts reaches its own column from its token on, across segments, and nothing before it."""
    clean = make(mode, [1500], 6, 64, 64, torch.float32)
    want = call(clean)[0]
    for bad in (float("inf"), float("nan"), 3e38):
        d = make(mode, [1500], 6, 64, 64, torch.float32)
        d["v"][171, 3] = bad
        got = call(d)[0]
        cols = torch.arange(got.shape[1]) != 3
        for part in (slice(0, 171), slice(171, None)):
            a, b = (x[part][:, cols] if part.start else x[part] for x in (got, want))
            assert (a - b).abs().max() <= 1e-5 * want.abs().max()
        if bad != 3e38:
            assert not torch.isfinite(got[171, 3])


# more than sixteen chunks of one portion in segments; whole portions of many heads
STEPS = pytest.mark.parametrize("lens,H,cut", [([450], 6, True), ([130, 40, 170], 66, False)], ids=["segments", "whole"])


def loop(d):
    """The same tokens one by one: the matrix memory's loop takes rows off a four-element boundary, the others' steps of up to four rows."""
    return base.call(dict(d, pad=1)) if d["mode"] == "mlstm" else in_short_portions(d, 4, call)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mode", ["gla", "light", "mlstm"])
@pytest.mark.parametrize("what", ["q", "k", "v", "gate", "state", "large"])
@STEPS
def test_not_finite(lens, H, cut, what, mode, dtype):
    """Infinities and NaN in what a token brings, or in the state: the same results are finite as token by token.  Values too large for three parts."""
    if mode == "light" and what == "gate":
        pytest.skip("light layers have one decay a head")
    for bad in (float("inf"), float("nan")) if what != "large" else (3.39e38,):
        d = make(mode, lens, H, 64, 64, dtype)
        d["past"] = [3] * len(lens)
        if what == "state":
            d["S"][len(lens), 2, 3, 4] = bad
        elif what == "gate":
            d["decay" if mode == "gla" else "a"][71, 2] = bad
        else:
            d["k" if what == "large" else what][71, 5] = bad
        assert base.route(d) == (3, cut)
        where_finite(call(d)[:2], loop(d)[:2])


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float32), (128, torch.bfloat16), (128, torch.float32)])
@pytest.mark.parametrize("mode,kind", [("gla", "plain"), ("gla", "share"), ("light", "plain"), ("light", "slow")])
@pytest.mark.parametrize("lens,H,cut", [([800], 6, True), ([130, 40, 170], 66, False)], ids=["segments", "whole"])
def test_no_further_off_than_the_loop(lens, H, cut, mode, kind, D, dtype):
    """As test_scan_precision.py's."""
    d = of_kind(make(mode, lens, H, D, 64, dtype), kind, 3)
    d["past"] = [7] * len(lens)
    assert base.route(d) == (3, cut)
    compare(mode, call(d)[:2], loop(d)[:2], oracle(d)[:2])


@torch.inference_mode()      # as models run, and other tests capture
def test_captured_segments_replay():
    """The states between segments in a graph's memory: every replay gives the eager result, with eager steps between them."""
    d = make("gla", [1500], 6, 64, 64, torch.bfloat16)
    c = {x: d[x].cuda() for x in ("q", "k", "v", "decay")}
    S0 = d["S"].cuda()
    S = S0.clone()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()  # noqa: E731
    where = (torch.arange(3, 1503, dtype=torch.int32).cuda(), i32([0, 1500]), i32([1]))
    run = lambda: linrec.gla_scan(c["q"], c["k"], c["v"], c["decay"], S, *where, 6, 64, 64)  # noqa: E731
    want = run()
    after = S.clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = run()
    for _ in range(3):
        S.copy_(S0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(S, after)
        run()
        torch.cuda.synchronize()


def test_decays_off_their_pairs():
    """Decays that cannot be read two at a time stay with the other kernel."""
    lens, H = [300, 33], 64
    d = make("gla", lens, H, 64, 64, torch.float32)
    wide = torch.zeros(sum(lens), H * 64 + 3)
    wide[:, 1:-2] = d["decay"]
    d["decay"] = type("Rows", (), {"cuda": lambda self: wide.cuda()[:, 1:-2], "to": lambda self, t: wide[:, 1:-2].to(t)})()
    base.check(call(d), oracle(d))
