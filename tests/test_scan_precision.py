"""The fast forms of the matrix-state recurrences against the token loop they take the place of, both measured against 64 bits: a chunk
that regroups the sums (dgi/csrc/mix/chunk_scan.hip) and a kernel laid out for single rows (row_scan_kernel in linear_scan.hip)
are no further off than the loop, in results and in states.

The measure is the 2-norm of the difference over that of the result, over 2e5 to 5e5 values.  Errors of the two forms are independent
roundings, so the ratio of two such norms has a spread of under one per cent (a few per cent where a sequence's values share a factor): 1.05.
The quotient of a matrix memory is dominated by its few smallest denominators and varies by tens of per cent: it is not compared."""
import pytest
import torch

from dgi.ops import linrec
from test_chunk_scan import F64, call, make, oracle

pytestmark = pytest.mark.gpu


def errors(got, want):
    return [((a.to(F64) - b).norm() / b.norm()).item() for a, b in zip(got, want)]


def compare(mode, fast, loop, want, limit=1.05):
    names = ["y", "state", "normaliser", "maximum"]
    a, b = errors(fast, want), errors(loop, want)
    for n, x, y in list(zip(names, a, b))[1 if mode == "mlstm" else 0:3]:
        assert x <= limit * y, (n, x, y)


def in_short_portions(d, rows):
    """The same tokens, at most ``rows`` of a sequence per call."""
    at, done, outs = [0] * len(d["lens"]), [], [[] for _ in d["lens"]]
    cur = dict(d)
    first = [sum(d["lens"][:i]) for i in range(len(d["lens"]))]
    while True:
        take = [min(rows, n - a) for n, a in zip(d["lens"], at)]
        if sum(take) == 0:
            return (torch.cat([torch.cat(o) for o in outs]),) + tuple(done)
        idx = torch.cat([torch.arange(f + a, f + a + t) for f, a, t in zip(first, at, take)])
        cur.update(lens=take, past=[p + a for p, a in zip(d["past"], at)])
        for k in ("q", "k", "v", "a", "b", "xbc", "dt"):
            if k in d:
                cur[k] = d[k][idx]
        done = call(cur)
        for o, part in zip(outs, torch.split(done[0], take)):
            o.append(part)
        done = done[1:]
        cur.update(S=done[0], **({"n": done[1], "m": done[2]} if len(done) > 1 else {}))
        at = [a + t for a, t in zip(at, take)]


@pytest.mark.parametrize("mode", ["wkv", "delta", "mlstm", "ssm"])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float32), (128, torch.bfloat16)])
def test_chunks(mode, D, dtype):
    d = make(mode, [300, 212], 16, D, 64 if mode != "wkv" else D, dtype, [0, 7], seed=D)
    want = oracle(d)
    if mode == "ssm":
        fast, loop = call(d, chunked=True), call(d, chunked=False)
    elif mode == "wkv":
        fast, loop = call(d), in_short_portions(d, 40)
    else:
        fast, loop = call(d), call(dict(d, pad=1))              # rows off a four-element boundary stay with the loop
    compare(mode, fast, loop, want)


@pytest.mark.parametrize("mode", ["wkv", "delta", "mlstm", "light"])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (48, torch.float32), (128, torch.bfloat16)])
def test_single_rows(mode, D, dtype, monkeypatch):
    d = make(mode, [1] * 96, 32, D, D, dtype, [9] * 96, seed=D)
    d["S"] *= 0.3
    want = oracle(d)
    fast = call(d)
    # a state four bytes off a 16-byte boundary goes to the loop
    where = []

    def shifted(fn):
        def run(*a, **k):
            a = list(a)
            i = next(i for i, t in enumerate(a) if torch.is_tensor(t) and t.dim() == 4)
            off = torch.empty(a[i].numel() + 1, device="cuda")[1:].view(a[i].shape)
            off.copy_(a[i])
            own, a[i] = a[i], off
            y = fn(*a, **k)
            own.copy_(off)
            where.append(off.data_ptr() % 16)
            return y
        return run

    for n in ("wkv_scan", "delta_scan", "mlstm_scan", "lightning_scan"):
        monkeypatch.setattr(linrec, n, shifted(getattr(linrec, n)))
    loop = call(d)
    assert where == [4]
    compare(mode, fast, loop, want)


def test_delta_chunks_of_128_channels():
    """Sums over 128 channels of the read-out, on rows as a convolution leaves them (SiLU): 1.4e6 results, so the ratio has a spread of two
    per mille."""
    d = make("delta", [600, 500], 10, 128, 128, torch.float32, [0, 0], seed=1)
    for n in ("q", "k", "v"):
        d[n] = torch.nn.functional.silu(d[n])
    want = oracle(d)
    fast, loop = errors(call(d), want)[0], errors(call(dict(d, pad=1)), want)[0]      # rows off a four-element boundary stay with the loop
    assert fast <= 1.01 * loop, (fast, loop)
