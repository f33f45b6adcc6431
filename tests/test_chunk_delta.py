"""Long prompt portions of the gated delta rule in chunks of 32 tokens (dgi/csrc/mix/chunk_delta.hip): lengths around a chunk, key and value sizes
around the tiles, heads that share q and k and heads that do not, sequences of unlike length, and values that are not finite, which leave the
matrix cores and go token by token.

Tolerance: as test_chunk_scan's, 3e-5 of the largest output."""
import pytest
import torch

from test_chunk_parts import where_finite
from test_chunk_scan import call, check, make, oracle
from test_scan_precision import taken

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [3, 4])                          # odd: every head has its own q and k
@pytest.mark.parametrize("D,V,dtype", [(64, 64, torch.float32), (64, 33, torch.bfloat16), (36, 17, torch.float32), (4, 16, torch.bfloat16),
                                       (100, 48, torch.bfloat16), (128, 32, torch.bfloat16)])
@pytest.mark.parametrize("lens", [[769], [800], [1500, 1, 831]], ids=lambda x: "-".join(map(str, x)))
def test_sizes(H, D, V, dtype, lens):
    d = make("delta", lens, H, D, V, dtype, [3 * (i % 2) for i in range(len(lens))], seed=D + V)
    check(call(d), oracle(d))


def test_repeated_keys_and_extreme_gates():
    """Equal keys at full write strength, where the inverse is as badly scaled as it gets; gates that close and open."""
    d = make("delta", [800], 4, 64, 64, torch.float32, [3])
    d["k"][:400] = d["k"][0]
    d["a"][:400], d["b"][:400] = 20.0, -20.0
    for i, (a, b) in enumerate(((40.0, 0.0), (-40.0, 0.0), (0.0, 40.0), (0.0, -40.0), (40.0, -40.0))):
        d["a"][417 + 9 * i], d["b"][418 + 9 * i] = a, b
    check(call(d), oracle(d))


@pytest.mark.parametrize("what", ["q", "k", "v", "a", "b", "S", "large"])
def test_not_finite(what):
    """Infinities and NaN in what a token brings, or in the state: the same results are finite as row by row.  Values too large for three parts."""
    for bad in (float("inf"), float("nan")) if what != "large" else (3.39e38,):
        d = make("delta", [800], 4, 64, 32, torch.float32, [3])
        if what == "S":
            d["S"][1, 2, 3, 4] = bad
        else:
            d["v" if what == "large" else what][71, 2] = bad
        where_finite(call(d)[:2], call(dict(d, pad=1))[:2])


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float32), (128, torch.bfloat16)])
@pytest.mark.parametrize("what", ["value", "state", "nan"])
def test_too_large_for_parts(what, D, dtype):
    """Finite values whose first bf16 part is an infinity, as x = beta (v - A k S) or by way of the state; and bf16 rows with a NaN.  What is finite row by row is
    finite here, and agrees (the products of the row loop overflow earlier in places)."""
    d = make("delta", [800], 4, D, 32, dtype, [3])
    big = 3.4e38 if dtype == torch.float32 else torch.finfo(dtype).max
    if what == "value":
        d["v"][71, 2] = big
        d["a"][71, 0] = 40.0
        x = torch.sigmoid(d["a"][71, 0]) * d["v"][71, 2].float()
        assert torch.isfinite(x)
        if dtype == torch.float32:
            assert not torch.isfinite(x.to(torch.bfloat16))
    elif what == "state":
        d["S"][1, 2, 3, 4] = 3.4e38
    else:
        for n in "qkv":
            d[n][71 + 90 * "qkv".index(n), 2] = float("nan")
    for got, want in zip(call(d), call(dict(d, pad=1))):
        ok = torch.isfinite(want)
        assert ok.any() and (got[ok] - want[ok]).abs().max() <= 1e-4 * max(1.0, want[ok].abs().max().item())
    if what == "nan":
        where_finite(call(d)[:2], call(dict(d, pad=1))[:2])


@pytest.mark.parametrize("H,D,V,dtype,lens", [(4, 64, 32, torch.bfloat16, [1, 16, 17, 0, 700, 801, 650, 700, 640]),
                                              (3, 128, 20, torch.bfloat16, [1, 16, 17, 0, 600, 801, 650, 700, 640]),
                                              (3, 64, 16, torch.bfloat16, [505, 1, 16, 17, 0] + [540] * 11 + [577]),
                                              (2, 36, 16, torch.float32, [1700, 1, 16, 17, 0, 1533, 2000, 1800, 64])], ids=lambda x: str(x)[:14])
def test_many_sequences(H, D, V, dtype, lens):
    """More than eight sequences: those of up to 16 rows in a launch of their own; more than sixteen: not ordered by length."""
    d = make("delta", lens, H, D, V, dtype, [3 * (i % 2) if n else 4 for i, n in enumerate(lens)], seed=D)
    assert taken(d) > 0
    check(call(d), oracle(d))
