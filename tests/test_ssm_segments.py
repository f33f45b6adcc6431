"""How the state-space scan cuts a step into segments (dgi_ssm_segments, host code): whatever the portions, no row lies behind the last."""
import ctypes
import os

import pytest

import dgi.build


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
