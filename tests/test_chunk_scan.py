"""Prompt portions of the matrix-state recurrences in chunks of sixteen tokens (dgi/csrc/mix/chunk_scan.hip) against a token loop in
64 bits: lengths around the chunk and the pairs of chunks the loops take, key and value sizes around the tiles, several
sequences with and without a state, decode rows beside portions, segments, extreme decays, values that are not finite.

Tolerance: every output is a sum of at most a few hundred products whose factors carry relative errors of some 16 roundings (the
products of decays inside a chunk) of 6e-8, about 1e-6 of the sum of magnitudes; 3e-5 of the largest output, as the other tests of
these recurrences allow."""
import ctypes

import pytest
import torch

import dgi.build
from dgi.ops import linrec, recur

F64 = torch.float64
pytestmark = pytest.mark.gpu


def softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


def make(mode, lens, H, D, V, dtype, past, seed=0, pad=0):
    g = torch.Generator().manual_seed(seed + 17)
    T, n = sum(lens), len(lens)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    d = {"mode": mode, "lens": lens, "H": H, "D": D, "V": V, "pad": pad, "past": past, "S": rn(n + 1, H, V, D) if mode == "ssm" else rn(n + 1, H, D, V),
         "n": rn(n + 1, H, D), "m": rn(n + 1, H)}
    if mode == "ssm":
        G = d["G"] = 2 if H % 2 == 0 else 1
        d["xbc"], d["dt"] = rn(T, H * V + 2 * G * D), rn(T, H).to(dtype)
        d["par"] = (rn(H) * 0.5 - 1, rn(H) * 0.3 - 0.5, rn(H))
        return d
    G = d["G"] = H // 2 if mode == "delta" and H % 2 == 0 else H
    x = rn(T, 2 * G * D + H * V + pad).to(dtype)
    d["q"], d["k"], d["v"] = x[:, :G * D], x[:, G * D:2 * G * D], x[:, 2 * G * D:2 * G * D + H * V]
    if mode == "wkv":
        d["a"], d["par"] = rn(T, H * D) * 0.6, (rn(H * D) * 0.7 - 1.5, rn(H * D) * 0.3)
    elif mode == "delta":
        d["a"], d["b"], d["par"] = rn(T, H), rn(T, H), (rn(H) * 0.5 - 1, rn(H) * 0.5 - 1)
    elif mode == "mlstm":
        d["a"], d["b"] = rn(T, H) * 2, rn(T, H) * 2
    else:
        d["par"] = (torch.rand(H, generator=g) ** 0.1,)
    return d


def route(d):
    """The kernel that takes the step's portions: 0 the token loop, 1 chunk_scan.hip or those it passes steps on to (all of light: chunk_parts.hip),
    2 chunk_scan_decay.hip, 3 chunk_segments.h; with the last one, whether long portions are cut."""
    lib, floats, at = ctypes.CDLL(dgi.build.build(group="mix")), ctypes.c_longlong(), ctypes.c_void_p(4096)
    H, G, D, V, fp32 = d["H"], d.get("G", d["H"]), d["D"], d["V"], d["q"].dtype == torch.float32
    row = 2 * G * D + H * V + d["pad"]
    args = (["wkv", "delta", "mlstm", "gla", "light"].index(d["mode"]), D, V, H, G, len(d["lens"]), sum(d["lens"]), at, row,
            ctypes.c_void_p(4096 + G * D * (4 if fp32 else 2)), row, int(fp32), at, H * D)
    form = lib.dgi_linear_scan_form(*args)
    lib.dgi_linear_scan_segments(*args, ctypes.byref(floats))
    return (form, floats.value > 0) if form == 3 else form


def call(d, **kw):
    c = lambda t: t.cuda()  # noqa: E731
    lens, H, D, V = d["lens"], d["H"], d["D"], d["V"]
    pos = torch.tensor([p + t for p, m in zip(d["past"], lens) for t in range(m)], dtype=torch.int32).cuda()
    row0 = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32).cuda()
    slots = torch.arange(len(lens), 0, -1, dtype=torch.int32).cuda()
    S, n, m = c(d["S"].clone()), c(d["n"].clone()), c(d["m"].clone())
    where = (pos, row0, slots)
    if d["mode"] == "ssm":
        b, a, s = d["par"]
        y = recur.ssm_scan(c(d["xbc"]), c(d["dt"]), c(b), c(a), c(s), S, *where, H, V, D, d["G"], **kw)
        return y.cpu(), S.cpu()
    # rows stay strided views
    gd, hv = d["G"] * D, H * V
    base = c(torch.cat([d["q"], d["k"], d["v"], d["q"][:, :d["pad"]]], 1))
    q, k, v = base[:, :gd], base[:, gd:2 * gd], base[:, 2 * gd:2 * gd + hv]
    if d["mode"] == "wkv":
        y = linrec.wkv_scan(q, k, v, c(d["a"]), c(d["par"][0]), c(d["par"][1]), S, *where, H, D)
    elif d["mode"] == "delta":
        y = linrec.delta_scan(q, k, v, c(d["a"]), c(d["b"]), c(d["par"][0]), c(d["par"][1]), S, *where, H, d["G"], D, V)
    elif d["mode"] == "mlstm":
        y = linrec.mlstm_scan(q, k, v, c(d["a"]), c(d["b"]), 15.0, S, n, m, *where, H, D, V)
        return y.cpu(), S.cpu(), n.cpu(), m.cpu()
    else:
        y = linrec.lightning_scan(q, k, v, c(d["par"][0]), S, *where, H, D, V)
    return y.cpu(), S.cpu()


def oracle(d):
    lens, H, D, V, mode = d["lens"], d["H"], d["D"], d["V"], d["mode"]
    S, n, m = d["S"].to(F64), d["n"].to(F64), d["m"].to(F64)
    T = sum(lens)
    y = torch.zeros(T, H, V, dtype=F64)
    if mode == "ssm":
        x, G = d["xbc"].to(F64), d["G"]
        v = x[:, :H * V].view(T, H, V)
        k = x[:, H * V:H * V + G * D].view(T, G, D).repeat_interleave(H // G, 1)
        q = x[:, H * V + G * D:].view(T, G, D).repeat_interleave(H // G, 1)
        dt = softplus(d["dt"].to(F64) + d["par"][0].to(F64))
        dec = torch.exp(-torch.exp(d["par"][1].to(F64)) * dt)
    else:
        q, k, v = (d[x].to(F64).reshape(T, -1, D if x != "v" else V) for x in ("q", "k", "v"))
        rep = H // q.shape[1]
        q, k = q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1)
        if mode == "light":
            q, k, v = (torch.nn.functional.silu(t) for t in (q, k, v))
        if mode == "delta":
            unit = lambda t: t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k = unit(q) * D ** -0.5, unit(k)
            beta, dec = torch.sigmoid(d["a"].to(F64)), torch.exp(-torch.exp(d["par"][0].to(F64)) * softplus(d["b"].to(F64) + d["par"][1].to(F64)))
        if mode == "mlstm":
            q = q * D ** -0.5
            ig, fg = 15 * torch.tanh(d["a"].to(F64) / 15), -softplus(-15 * torch.tanh(d["b"].to(F64) / 15))
    at = 0
    for i, ln in enumerate(lens):
        slot = len(lens) - i
        old = d["past"][i] > 0
        s = (S[slot].transpose(1, 2) if mode == "ssm" else S[slot]) * (1.0 if old else 0.0)
        nn, mm = n[slot] * (1.0 if old else 0.0), m[slot] * (1.0 if old else 0.0)
        for t in range(at, at + ln):
            kv = k[t][:, :, None] * v[t][:, None, :]
            if mode == "wkv":
                w = torch.exp(-torch.exp(d["a"][t].to(F64) + d["par"][0].to(F64))).view(H, D, 1)
                y[t] = torch.einsum("hk,hkv->hv", q[t], s + d["par"][1].to(F64).view(H, D, 1) * kv)
                s = w * s + kv
                continue
            if mode == "delta":
                s = dec[t][:, None, None] * s
                s = s + k[t][:, :, None] * (beta[t][:, None] * (v[t] - torch.einsum("hk,hkv->hv", k[t], s)))[:, None, :]
            elif mode == "mlstm":
                new = torch.maximum(fg[t] + mm, ig[t])
                a, b = torch.exp(fg[t] + mm - new), torch.exp(ig[t] - new)
                s, nn, mm = a[:, None, None] * s + b[:, None, None] * kv, a[:, None] * nn + b[:, None] * k[t], new
            elif mode == "ssm":
                s = dec[t][:, None, None] * s + dt[t][:, None, None] * kv
            else:
                s = d["par"][0].to(F64)[:, None, None] * s + kv
            y[t] = torch.einsum("hk,hkv->hv", q[t], s)
            if mode == "mlstm":
                y[t] /= (torch.maximum((nn * q[t]).sum(-1).abs(), torch.exp(-mm)) + 1e-6)[:, None]
            if mode == "ssm":
                y[t] += d["par"][2].to(F64)[:, None] * v[t]
        S[slot] = s.transpose(1, 2) if mode == "ssm" else s
        n[slot], m[slot] = nn, mm
        at += ln
    return (y.reshape(T, -1), S) + ((n, m) if mode == "mlstm" else ())


def check(got, want):
    for a, b in zip(got, want):
        assert torch.isfinite(b).all()
        assert (a.to(F64) - b).abs().max() <= 3e-5 * max(1.0, b.abs().max().item())


MODES = ["wkv", "delta", "mlstm", "light", "ssm"]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("lens", [[65], [257], [272, 273], [15, 400, 1], [1] * 9 + [17, 520, 300]], ids=lambda x: "-".join(map(str, x))[:20])
def test_lengths(mode, lens):
    """Ends inside a chunk, at its edge and after an odd number of chunks; short sequences beside long ones in one launch (up to eight
    sequences) and in one of their own; every second sequence continues a state."""
    H = (200 if len(lens) < 3 else 70) if mode == "light" else 6        # light: enough workgroups (or rows) for either of its kernels
    d = make(mode, lens, H, 64, 64, torch.float32, [3 * (i % 2) for i in range(len(lens))])
    check(call(d, **({"chunked": True} if mode == "ssm" else {})), oracle(d))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("D,V", [(4, 16), (20, 8), (64, 33), (68, 48), (128, 100), (36, 17)])
def test_sizes(mode, D, V):
    """Key sizes below, at and above a 64-channel group, value sizes of one, two and three 16-column blocks and odd ones; bf16 rows."""
    if mode == "wkv":
        V = D
    light = mode == "light"
    H = 400 // -(-V // 16) + 1 if light else 4
    d = make(mode, [170, 166] if light else [70, 66], H, D, V, torch.bfloat16, [5, 0])
    check(call(d, **({"chunked": True} if mode == "ssm" else {})), oracle(d))


@pytest.mark.parametrize("D,V,pad", [(18, 10, 0), (20, 8, 1), (200, 32, 0)])
@pytest.mark.parametrize("mode", ["delta", "mlstm", "light", "ssm"])
def test_rows_the_chunks_do_not_take(mode, D, V, pad):
    """Key sizes that are no multiple of four or above 128 (ssm: 256, so 200 is one of its own) and rows off a four-element boundary: another
    kernel, the same result."""
    d = make(mode, [70, 66], 4, D, V, torch.bfloat16, [0, 5], pad=pad)
    check(call(d), oracle(d))


@pytest.mark.parametrize("H,n", [(2, [1500, 700, 5]), (1, [3000])])
def test_ssm_segments(H, n):
    """Few heads: portions in segments side by side, the last one short, beside a sequence of one segment."""
    for past in (0, 40):
        d = make("ssm", n, H, 128, 48, torch.bfloat16, [past] * len(n))
        check(call(d), oracle(d))


def test_wkv_decays_beyond_the_fp32_range():
    """Channels whose decays leave the fp32 range within half a chunk, beside ones that barely decay; decays of exactly zero."""
    d = make("wkv", [150, 90], 3, 68, 68, torch.float32, [0, 7])
    d["a"][20:60, ::3] = 3.0
    d["a"][45, 1::2] = 8.0
    d["a"][50:53, 0] = 60.0
    d["a"][70:, :5] = -9.0
    check(call(d), oracle(d))


def test_mlstm_and_delta_extreme_gates():
    for mode in ("mlstm", "delta"):
        d = make(mode, [200], 4, 64, 64, torch.float32, [3])
        for i, (a, b) in enumerate(((40.0, 0.0), (-40.0, 0.0), (0.0, 40.0), (0.0, -40.0), (40.0, -40.0))):
            d["a"][17 + 9 * i], d["b"][18 + 9 * i] = a, b
        check(call(d), oracle(d))


def test_delta_repeated_keys():
    """Equal keys and full write strength: the substitution inside a chunk is as badly scaled as it gets (entries of 1 below the diagonal)."""
    d = make("delta", [130], 4, 64, 64, torch.float32, [3])
    d["k"][:] = d["k"][0]
    d["a"][:], d["b"][:] = 20.0, -20.0
    check(call(d), oracle(d))


@pytest.mark.parametrize("mode", MODES)
def test_non_finite_values_stay_behind(mode):
    """An infinity or NaN in a token's value reaches that token's column from that token on, and nothing before it."""
    lens, t = [170 if mode == "light" else 130], 71      # inside a chunk
    H = 200 if mode == "light" else 4
    kw = {"chunked": True} if mode == "ssm" else {}
    clean = make(mode, lens, H, 64, 64, torch.float32, [0])
    want = call(clean, **kw)[0]
    for bad in (float("inf"), float("nan")):
        d = make(mode, lens, H, 64, 64, torch.float32, [0])
        (d["xbc"] if mode == "ssm" else d["v"])[t, 3] = bad
        got = call(d, **kw)[0]
        assert torch.equal(got[:t], want[:t]) or (got[:t] - want[:t]).abs().max() <= 1e-5 * want.abs().max()
        cols = torch.ones(got.shape[1], dtype=torch.bool)
        cols[3] = False
        assert torch.isfinite(got[:, cols]).all()
        assert not torch.isfinite(got[t, 3])


@pytest.mark.parametrize("D,V", [(132, 33), (200, 48), (256, 64), (256, 100)])
def test_ssm_large_states(D, V):
    """Key sizes of 129 to 256 (one column block per workgroup, so every wave beyond the roles of one would write another's columns):
    one, two and more blocks of columns, whole portions, segments, and short sequences in a launch of their own."""
    for lens in ([70, 66], [700, 33], [1] * 9 + [120]):
        d = make("ssm", lens, 2, D, V, torch.float32, [3 * (i % 2) for i in range(len(lens))], seed=D + V)
        check(call(d, chunked=True), oracle(d))


@pytest.mark.parametrize("lens", [[0, 577], [577, 0], [0, 0, 1500, 0], [600, 0, 70]])
def test_ssm_segments_beside_sequences_without_rows(lens):
    """Empty sequences leave a portion longer than rows - sequences + 1: its last rows and its state are there all the same, and the
    empty ones keep their states."""
    d = make("ssm", lens, 1, 128, 32, torch.bfloat16, [4 if n == 0 else 0 for n in lens], seed=len(lens))
    check(call(d, chunked=True), oracle(d))


def test_ssm_of_fp32_models_does_not_depend_on_the_step():
    """A sequence alone, beside others, and in two parts: the same numbers, bit for bit."""
    lens, cut = [300, 90, 700], 130
    d = make("ssm", lens, 8, 64, 64, torch.float32, [0, 5, 0])
    y, S = call(d)
    check((y, S), oracle(make("ssm", lens, 8, 64, 64, torch.float32, [0, 5, 0])))
    only = dict(d, lens=lens[:1], past=[0], xbc=d["xbc"][:300], dt=d["dt"][:300])
    y1, S1 = call(only)
    assert torch.equal(y1, y[:300]) and torch.equal(S1[1], S[3])
    y2, S2 = call(dict(only, lens=[cut], xbc=d["xbc"][:cut], dt=d["dt"][:cut]))
    y3, S3 = call(dict(only, lens=[300 - cut], past=[cut], S=S2, xbc=d["xbc"][cut:300], dt=d["dt"][cut:300]))
    assert torch.equal(torch.cat([y2, y3]), y[:300]) and torch.equal(S3[1], S[3])


@pytest.mark.parametrize("q,k", [(1e17, 1e-17), (1e-17, 1e17), (1e-15, 1e-3), (1e16, 1e-3)])
def test_wkv_scales_beside_strong_decays(q, k):
    """Half a chunk's decays near the edge of what the scaled operands allow, q and k far from 1: scaled they would leave the fp32 range
    (an overflow, or keys that vanish), the results do not."""
    d = make("wkv", [130, 40], 3, 64, 64, torch.float32, [0, 7])
    d["a"][:], d["par"] = 0.0, (torch.full_like(d["par"][0], 2.04), d["par"][1])      # half a chunk: about 1e-27
    d["a"][:, 1::2] = -6.0
    d["q"] *= q
    d["k"] *= k
    d["S"] *= k
    y, S = call(d)
    wy, wS = oracle(d)
    assert torch.isfinite(wy.float()).all() and torch.isfinite(wS.float()).all()
    assert (y.to(F64) - wy).abs().max() <= 3e-5 * wy.abs().max()
    assert (S.to(F64) - wS).abs().max() <= 3e-5 * wS.abs().max()
    # the strongly decayed channels by themselves: their own sums, not hidden behind the others'
    d["q"][:, 1::2] = 0.0
    y, wy = call(d)[0], oracle(d)[0]
    assert (y.to(F64) - wy).abs().max() <= 3e-5 * wy.abs().max()


@pytest.mark.parametrize("mode,H,D,line", [("wkv", 52, 16, 136), ("wkv", 310, 16, 224), ("wkv", 11, 68, 104), ("ssm", 2, 20, 48), ("ssm", 14, 20, 112),
                                           ("ssm", 28, 20, 144), ("ssm", 14, 20, 88)])
def test_portions_around_the_line_between_the_launches(mode, H, D, line):
    """Among more than eight sequences portions of at most ``line`` rows go in a launch of their own; the line depends on the number of
    workgroups (and, wkv, on the key size).  One row to either side of it, on average near it, and decode rows beside one long portion."""
    V = D if mode == "wkv" else 17
    for lens, H in (([line, line + 1, line - 1, 1, line, 2 * line + 200, line + 1, 15, line + 7, line + 16], H),
                    ([1] * 30 + [line + 1, 700, line], -(-10 * H // 33))):
        d = make(mode, lens, H, D, V, torch.bfloat16, [3 * (i % 2) for i in range(len(lens))], seed=H)
        if mode == "ssm":
            assert recur.scan_chunks(sum(lens), len(lens), H, V, torch.bfloat16)
        check(call(d), oracle(d))


@pytest.mark.parametrize("lens", [[90, 70], [1500, 40]])
def test_ssm_takes_only_position_zero_as_a_start(lens):
    """A portion at any other position reads its state, whole or in segments: the same as row by row."""
    d = make("ssm", lens, 1, 64, 32, torch.bfloat16, [-2000, 0], seed=4)
    want = call(d, chunked=False)
    check(call(d, chunked=True), [t.to(F64) for t in want])
    assert not torch.allclose(want[0][:4], call(dict(d, past=[0, 0]), chunked=False)[0][:4])


@pytest.mark.parametrize("mode,dtype", [("delta", torch.bfloat16), ("delta", torch.float32), ("mlstm", torch.bfloat16), ("mlstm", torch.float32),
                                        ("light", torch.bfloat16), ("light", torch.float32)])
@pytest.mark.parametrize("D,V", [(64, 64), (48, 33), (64, 72), (60, 130)])
@pytest.mark.parametrize("lens", [[70, 71, 96, 65, 80, 64, 81, 66, 79],             # four column blocks a workgroup (delta of up to 64 channels)
                                  [500] + [17, 20, 18, 33, 19, 17, 21, 18],         # two: one portion is most of the step
                                  [1, 300, 1, 1, 17, 290, 1, 16, 1, 310, 305, 1, 1, 1, 1, 299]])      # decode rows beside portions
def test_more_workgroups_than_units(mode, dtype, D, V, lens):
    """Steps of more than 256 workgroups, which take two blocks of value columns each, or four, longest sequences first."""
    if mode == "light":
        lens = [n * 5 if n > 16 else n for n in lens]           # its chunks are taken from up to 112 rows a sequence on
    H = 16 if len(lens) * 16 * -(-V // 32) > 256 else 32
    d = make(mode, lens, H, D, V, dtype, [0 if i % 3 else 40 for i in range(len(lens))], seed=len(lens) + V, pad=8)
    check(call(d), oracle(d))
