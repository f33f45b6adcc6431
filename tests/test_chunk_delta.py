"""Long prompt portions of the gated delta rule in chunks of 32 tokens (dgi/csrc/mix/chunk_delta.hip): lengths around a chunk, key and value sizes
around the tiles, heads that share q and k and heads that do not, sequences of unlike length, and values that are not finite, which leave the
matrix cores and go token by token.

Tolerance: as test_chunk_scan's, 3e-5 of the largest output."""
import pytest
import torch

from test_chunk_parts import where_finite
from test_chunk_scan import call, check, make, oracle

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
