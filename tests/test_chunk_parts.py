"""Prompt portions in chunks of 32 tokens on the bf16 matrix cores (dgi/csrc/mix/chunk_parts.hip): lengths around a chunk and around the 64 tokens
whose gates are made together, key and value sizes around its tiles, state-space groups (what their heads share is prepared in a pass of its own), segments,
and values that are not finite, which leave the matrix cores and go token by token.

Tolerance: as test_chunk_scan's, 3e-5 of the largest output."""
import pytest
import torch

from test_chunk_scan import F64, call, check, make, oracle, route
from test_scan_precision import in_short_portions

pytestmark = pytest.mark.gpu


def run(d):
    return call(d, **({"chunked": True} if d["mode"] == "ssm" else {}))


def heads(mode, V):
    return 8 if mode == "ssm" else 400 // -(-V // 16) + 1 if mode == "light" else 4      # light: so many that most steps are chunk_segments.h's


@pytest.mark.parametrize("mode", ["mlstm", "light", "ssm"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,V", [(64, 64), (4, 16), (36, 17), (100, 48), (128, 33)])
@pytest.mark.parametrize("lens", [[97], [128, 65, 160, 31, 32, 33, 1], [95, 129]], ids=lambda x: "-".join(map(str, x)))
def test_sizes(mode, dtype, D, V, lens):
    if mode == "light":
        lens = [n + 96 if n > 90 else n for n in lens]
    d = make(mode, lens, heads(mode, V), D, V, dtype, [3 * (i % 2) for i in range(len(lens))], seed=D + V)
    check(run(d), oracle(d))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,V", [(64, 64), (4, 16), (20, 8), (36, 17), (64, 33), (68, 48), (100, 48), (128, 33), (128, 100)])
@pytest.mark.parametrize("lens", [[257], [288, 225, 320, 31, 32, 33, 1], [255, 289], [170, 166]], ids=lambda x: "-".join(map(str, x)))
def test_sizes_of_light(dtype, D, V, lens):
    """Few heads, so that these portions are this kernel's: the lengths of the other layers with five chunks more."""
    d = make("light", lens, 4, D, V, dtype, [3 * (i % 2) for i in range(len(lens))], seed=D + V)
    assert route(d) == 1
    check(call(d), oracle(d))


@pytest.mark.parametrize("lens,H,D,V", [([65], 70, 64, 64), ([257], 70, 64, 64), ([272, 273], 70, 64, 64), ([15, 400, 1], 50, 64, 64), ([1] * 9 + [17, 520, 300], 10, 128, 128),
                                        ([280, 284, 384, 260, 320, 256, 324, 264, 316], 17, 64, 64), ([280, 284, 384, 260, 320, 256, 324, 264, 316], 16, 48, 33),
                                        ([2000] + [68, 80, 72, 132, 76, 68, 84, 72], 17, 64, 64), ([280, 284, 384, 260, 320, 256, 324, 264, 316], 8, 60, 130)],
                         ids=lambda x: "-".join(map(str, x))[:16] if isinstance(x, list) else str(x))
def test_lengths_of_light(lens, H, D, V):
    """One block of value columns a workgroup and, of more than 256 workgroups, two; up to eight sequences in one launch, more in two."""
    d = make("light", lens, H, D, V, torch.bfloat16 if H in (16, 17) else torch.float32, [3 * (i % 2) for i in range(len(lens))], seed=len(lens) + V)
    assert route(d) == 1
    check(call(d), oracle(d))


@pytest.mark.parametrize("H,D,lens", [(8, 128, [1500, 40]), (8, 60, [700]), (12, 64, [600, 0, 70])])
def test_segments(H, D, lens):
    """Few heads: segments (of whole chunks) side by side, with the prepared parts shared by both passes."""
    for past in (0, 40):
        d = make("ssm", lens, H, D, 24, torch.bfloat16, [past or (0 if n else 4) for n in lens], seed=H + D)      # an empty sequence keeps its state
        check(run(d), oracle(d))


@pytest.mark.parametrize("D,V", [(128, 33), (100, 48), (68, 16)])
@pytest.mark.parametrize("lens", [[320], [333, 311], [319], [1027, 1, 0], [1025, 1]], ids=lambda x: "-".join(map(str, x)))
def test_ssm_pass(D, V, lens):
    """Long state-space steps of more than 64 channels: the parts come from a pass before, on either side of the lines from which they do; H = 8 in segments where one
    portion may have 512 rows, H = 72 in whole portions."""
    for H in (8, 72) if lens[0] > 1000 else (8,):
        d = make("ssm", lens, H, D, V, torch.bfloat16, [3 * (i % 2) if n else 4 for i, n in enumerate(lens)], seed=D + H)
        check(run(d), oracle(d))


def test_ssm_same_with_and_without_the_pass():
    """Beside an empty sequence the same 400 rows are a step without it: the same numbers, bit for bit."""
    d = make("ssm", [400], 8, 128, 64, torch.bfloat16, [5])
    y, S = run(d)
    y2, S2 = run(dict(d, lens=[400, 0], past=[5, 5], S=torch.cat([d["S"][:1], d["S"]])))
    assert torch.equal(y, y2) and torch.equal(S[1], S2[2])


def where_finite(got, want):
    """The same values are finite, and they agree."""
    for a, b in zip(got, want):
        fa, fb = torch.isfinite(a), torch.isfinite(b)
        assert torch.equal(fa, fb)
        if fb.any():
            assert (a[fa] - b[fb]).abs().max() <= 1e-4 * max(1.0, b[fb].abs().max().item())


@pytest.mark.parametrize("what", ["q", "k", "v", "gate", "state", "large"])
@pytest.mark.parametrize("mode", ["mlstm", "ssm"])
def test_not_finite(mode, what):
    """Infinities and NaN in what a token brings, or in the state: the same results are finite as row by row.  Values too large for three parts."""
    for bad in (float("inf"), float("nan")) if what != "large" else (3.39e38,):
        d = make(mode, [130], 8, 64, 32, torch.float32, [3])
        t = 71
        if mode == "ssm":
            G, x = d["G"], d["xbc"]
            at = {"v": 3, "k": 8 * 32 + 5, "q": 8 * 32 + G * 64 + 5, "large": 8 * 32 + 5}.get(what)
            if at is not None:
                x[t, at] = bad
        elif what in ("q", "k", "v", "large"):
            d["k" if what == "large" else what][t, 5] = bad
        if what == "gate":
            (d["dt"] if mode == "ssm" else d["a"])[t, 2] = bad
        if what == "state":
            d["S"][1, 2, 3, 4] = bad
        slow = call(d, chunked=False) if mode == "ssm" else call(dict(d, pad=1))
        where_finite(run(d)[:2], slow[:2])


@pytest.mark.parametrize("what", ["q", "k", "v", "gate", "state", "large"])
def test_ssm_pass_not_finite(what):
    """The same where the parts come from a pass before."""
    for bad in (float("inf"), float("nan")) if what != "large" else (3.39e38,):
        d = make("ssm", [330], 8, 128, 32, torch.float32, [3])
        at = {"v": 3, "k": 8 * 32 + 5, "q": 8 * 32 + d["G"] * 128 + 5, "large": 8 * 32 + 5}.get(what)
        if at is not None:
            d["xbc"][171, at] = bad
        elif what == "gate":
            d["dt"][171, 2] = bad
        else:
            d["S"][1, 2, 3, 4] = bad
        where_finite(run(d)[:2], call(d, chunked=False)[:2])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mode", ["mlstm", "light"])
@pytest.mark.parametrize("what", ["q", "k", "v", "state", "large"])
def test_not_finite_bf16(what, mode, D):
    """bf16 rows, and light layers; beside the loop, which light layers have for steps of up to four rows."""
    for dtype in (torch.bfloat16, torch.float32) if mode == "light" else (torch.bfloat16,):
        for bad in (float("inf"), float("nan")) if what != "large" else (3.39e38,):
            d = make(mode, [130], 8, D, 32, dtype, [3])
            if what == "state":
                d["S"][1, 2, 3, 4] = bad
            else:
                d["k" if what == "large" else what][71, 5] = bad
            assert route(d) == 1
            slow = call(dict(d, pad=1)) if mode == "mlstm" else in_short_portions(d, 4)
            where_finite(call(d)[:2], slow[:2])


def test_light_decays_that_are_none():
    """Decays of 0, below 0 and above 1 (whose powers may leave the fp32 range)."""
    d = make("light", [200], 104, 64, 32, torch.float32, [3])
    d["par"][0][:6] = torch.tensor([0.0, -0.5, 1.0, 1.01, 1e-30, 100.0])
    assert route(d) == 1
    got, want = run(d), oracle(d)
    for h in range(104):
        g, w = got[0].view(200, 104, 32)[:, h].to(F64), want[0].view(200, 104, 32)[:, h]
        for t in range(200):                                   # up to where a state of fp32 values would overflow
            if w[t].abs().max() > 1e30:
                break
            assert (g[t] - w[t]).abs().max() <= 3e-5 * max(1.0, w[: t + 1].abs().max().item())
