"""Steps of single rows of the matrix-state recurrences (row_scan_kernel in dgi/csrc/mix/linear_scan.hip) against a token loop in
64 bits: sizes around the column and channel groups, fresh sequences whose slot holds no numbers, sequences without and with
several rows in a step of as many rows as sequences."""
import pytest
import torch

from test_chunk_scan import call, check, make, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["wkv", "delta", "mlstm", "light"])
@pytest.mark.parametrize("D,V", [(64, 64), (48, 48), (4, 4), (65, 60), (100, 64), (64, 68), (128, 128), (17, 124)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_single_rows(mode, D, V, dtype):
    if mode == "wkv":
        V = D
    if V % 4:
        V = V // 4 * 4 if mode != "wkv" else V
    past = [5, 0, 700, 1, 0]
    d = make(mode, [1] * 5, 4, D, V, dtype, past, seed=D + V)
    want = oracle(d)
    got = call(d)
    check(got, want)
    # a fresh sequence reads nothing of its slot
    for i, p in enumerate(past):
        if p == 0:
            d["S"][5 - i] = float("nan")
            d["n"][5 - i] = float("nan")
            d["m"][5 - i] = float("nan")
    check(call(d), want)


@pytest.mark.parametrize("mode", ["wkv", "delta", "mlstm", "light"])
def test_rows_unlike_sequences(mode):
    d = make(mode, [3, 0, 1, 0, 2, 0], 4, 64, 64, torch.float32, [2, 9, 0, 4, 7, 1], seed=3)      # sequences without rows keep their state
    check(call(d), oracle(d))
