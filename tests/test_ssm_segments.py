"""How the state-space scan cuts a step into segments (dgi_ssm_segments, host code): whatever the portions, no row lies behind the last.
And which steps go in chunks at all."""
import ctypes
import os

import pytest

import dgi.build
from dgi.ops import recur


def segments(n_seq, heads, dv, rows):
    import torch  # noqa: F401  the library links against torch's
    lib = ctypes.CDLL(dgi.build.build(group="mix"))
    each = ctypes.c_int(-1)
    return lib.dgi_ssm_segments(n_seq, heads, dv, rows, ctypes.byref(each)), each.value


@pytest.mark.parametrize("n_seq", [1, 2, 3, 17, 64])
@pytest.mark.parametrize("heads,dv", [(1, 16), (1, 32), (3, 48), (16, 64), (64, 64)])
def test_segments_cover_a_step_of_one_portion(n_seq, heads, dv):
    """All rows may be one sequence's: the others are empty."""
    for rows in (1, 511, 512, 513, 577, 639, 640, 1535, 1536, 1537, 4096, 100003):
        segs, each = segments(n_seq, heads, dv, rows)
        assert 1 <= segs <= 24
        if segs > 1:
            assert each % 16 == 0 and each >= 64 and segs * each >= rows


def test_which_steps_go_in_chunks(monkeypatch):
    import torch
    f32, bf16 = torch.float32, torch.bfloat16
    assert recur.scan_chunks(4096, 2, 64, 64, bf16) and not recur.scan_chunks(4096, 2, 64, 64, f32)
    assert not recur.scan_chunks(64, 64, 64, 64, bf16)
    assert recur.scan_chunks(10, 1, 1, 16, f32, True) and not recur.scan_chunks(4096, 2, 64, 64, bf16, False)
    # the switches: a number of workgroups from which steps go row by row (0: all), and off, also for calls that ask for chunks
    monkeypatch.setattr(recur, "SCAN_CHUNK_BELOW", 512)
    assert not recur.scan_chunks(4096, 2, 64, 64, bf16) and recur.scan_chunks(4096, 1, 64, 64, bf16)
    assert recur.scan_chunks(4096, 2, 64, 64, bf16, True)
    monkeypatch.setattr(recur, "SCAN_CHUNK", 0)
    assert not recur.scan_chunks(4096, 1, 64, 64, bf16) and not recur.scan_chunks(4096, 1, 64, 64, bf16, True)
