"""The fast forms of the matrix-state recurrences against the token loop they take the place of, both measured against 64 bits: a chunk
that regroups the sums (dgi/csrc/mix/chunk_scan.hip) and a kernel laid out for single rows (row_scan_kernel in linear_scan.hip)
are no further off than the loop, in results and in states.

The measure is the 2-norm of the difference over that of the result, over 2e5 to 5e5 values.  Errors of the two forms are independent
roundings, so the ratio of two such norms has a spread of under one per cent (a few per cent where a sequence's values share a factor): 1.05.
The quotient of a matrix memory is dominated by its few smallest denominators and varies by tens of per cent: it is not compared."""
import ctypes

import pytest
import torch

import dgi.build
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


def in_short_portions(d, rows, call=call):
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
        for k in ("q", "k", "v", "a", "b", "xbc", "dt", "decay"):
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


def taken(d):
    """Floats of workspace that long portions of delta get: 0, and their chunks would have sixteen tokens."""
    lib = ctypes.CDLL(dgi.build.build(group="mix"))
    lib.dgi_linear_scan_parts.restype = ctypes.c_longlong
    row = 2 * d["G"] * d["D"] + d["H"] * d["V"]
    at = ctypes.c_void_p(4096)
    return lib.dgi_linear_scan_parts(1, d["D"], d["V"], d["H"], d["G"], len(d["lens"]), sum(d["lens"]), at, row, at, row, int(d["q"].dtype == torch.float32),
                                     ctypes.byref(ctypes.c_int()))


def of_kind(d, kind, seed):
    """Rows as a convolution leaves them (SiLU); rows that share a direction twice as large as what they differ in; decays near 1."""
    g = torch.Generator().manual_seed(seed)
    for n in "qkv":
        x = d[n].float()
        if kind == "silu":
            x = torch.nn.functional.silu(x)
        if "share" in kind and n != "v":
            x = x + 2 * torch.randn(1, x.shape[1], generator=g)
        d[n] = x.to(d[n].dtype)
    if "slow" in kind:
        if d["mode"] == "delta":
            d["par"] = (d["par"][0] - 5, d["par"][1])
        elif d["mode"] == "mlstm":
            d["b"] = d["b"] + 6
        else:
            d["par"] = (1 - torch.rand(d["H"], generator=g) * 1e-3,)
    return d


@pytest.mark.parametrize("D,dtype,rows", [(64, torch.float32, 800), (64, torch.bfloat16, 400), (128, torch.bfloat16, 400)])
@pytest.mark.parametrize("kind", ["plain", "silu", "share", "slow", "share slow"])
def test_long_portions_of_delta(kind, D, dtype, rows):
    """Chunks of 32 tokens with a prepared inverse (dgi/csrc/mix/chunk_delta.hip).  Where decays are near 1 the loop is five times further off (it rounds every
    decay); keys that share a direction make the inverse's terms large beside their sum: there states may be up to a quarter further off than the loop's."""
    d = of_kind(make("delta", [rows], 16, D, 64, dtype, [7], seed=D), kind, 3)
    assert taken(d) > 0
    want = oracle(d)
    a, b = errors(call(d), want), errors(call(dict(d, pad=1)), want)
    assert a[0] <= 1.05 * b[0] and a[1] <= (1.25 if kind == "share" else 1.05) * b[1], (a, b)
    if "slow" in kind:
        assert a[0] <= 0.4 * b[0] and a[1] <= 0.4 * b[1], (a, b)


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float32), (128, torch.bfloat16), (128, torch.float32)])
@pytest.mark.parametrize("kind", ["plain", "slow"])
def test_chunks_of_light(kind, D, dtype):
    """Light layers in chunks of 32 (dgi/csrc/mix/chunk_parts.hip) against the loop, which takes steps of up to four rows."""
    d = of_kind(make("light", [300], 16, D, 64, dtype, [7], seed=D), kind, 3)
    compare("light", call(d), in_short_portions(d, 4), oracle(d))


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float32), (128, torch.bfloat16)])
@pytest.mark.parametrize("kind", ["plain", "silu", "share", "slow"])
def test_outputs_of_a_matrix_memory(kind, D, dtype):
    """Its outputs by the geometric mean of the errors of tokens and heads, which a few small denominators do not decide (8192 of them: a spread of one per
    cent)."""
    d = of_kind(make("mlstm", [512], 16, D, 64, dtype, [7], seed=D), kind, 3)
    want = oracle(d)[0].view(512 * 16, 64)

    def mean(y):
        return ((y.to(F64).view_as(want) - want).norm(dim=1) / want.norm(dim=1)).clamp_min(1e-12).log().mean().exp().item()

    fast, loop = mean(call(d)[0]), mean(call(dict(d, pad=1))[0])
    assert fast <= 1.05 * loop, (fast, loop)
