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


def test_short_portions_need_no_pass():
    """Steps of short portions, and of up to 64 channels, have no launch before the one that does the work; with more than 64 workgroups only portions that may
    have 1024 rows are cut."""
    import torch  # noqa: F401
    lib = ctypes.CDLL(dgi.build.build(group="mix"))
    lib.dgi_ssm_parts_floats.restype = ctypes.c_longlong
    chunks = ctypes.c_int()

    def floats(dk, heads, groups, rows, n_seq):
        return lib.dgi_ssm_parts_floats(dk, heads, groups, rows, n_seq, ctypes.byref(chunks))

    for rows, n_seq in ((65, 1), (319, 1), (640, 8), (1030, 12), (530, 24)):
        assert floats(128, 16, 2, rows, n_seq) == 0 and floats(64, 16, 2, rows, n_seq) == 0
    for rows, n_seq in ((320, 1), (8192, 2), (2032, 33), (616, 17)):
        assert floats(128, 16, 2, rows, n_seq) > 0 and floats(64, 16, 2, rows, n_seq) == 0
    assert floats(128, 6, 2, 8192, 2) == 0 and floats(132, 16, 2, 8192, 2) == 0
    assert lib.dgi_ssm_whole(8, 8, 64, 64, 1, 520, 9) and not lib.dgi_ssm_whole(8, 8, 64, 64, 1, 2007, 9)
    assert not lib.dgi_ssm_whole(1, 8, 64, 64, 1, 600, 10) and not lib.dgi_ssm_whole(8, 8, 64, 64, 4, 520, 9)
    assert lib.dgi_ssm_whole(2, 32, 64, 64, 1, 4000, 3) and not lib.dgi_ssm_whole(2, 24, 64, 64, 1, 4000, 5)
