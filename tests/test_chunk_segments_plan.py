"""Which steps the kernel of whole heads takes (dgi/csrc/mix/chunk_segments.hip), and what workspace its segments have: the plan is a host function, so
it runs here without a GPU."""
import ctypes
import random

import pytest
import torch  # noqa: F401  (the library's own dependencies)

import dgi.build

MODES = {"mlstm": 2, "gla": 3, "light": 4}


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(dgi.build.build(group="mix"))


def plan(lib, mode, H, n_seq, rows, D=64, V=None, fp32=False):
    """(rows of a segment: 0 not here, 1 << 29 whole portions; floats of workspace)"""
    floats, at, row = ctypes.c_longlong(), ctypes.c_void_p(4096), 3 * H * D
    each = lib.dgi_linear_scan_segments(MODES[mode], D, V or D, H, H, n_seq, rows, at, row, at, row, int(fp32), at, H * D, ctypes.byref(floats))
    return each, floats.value


def test_workspace_does_not_grow_with_the_sequences(lib):
    """A place for each segment of a portion that is cut, and they fill the chip once: 20 MB at most, whatever the step."""
    rng, cut = random.Random(1), 0
    for _ in range(20000):
        mode, H, D = rng.choice(sorted(MODES)), rng.choice([1, 2, 5, 8, 16, 32, 64, 128]), rng.choice([16, 48, 64, 100, 128])
        n = int(2 ** rng.uniform(0, 12))
        each, floats = plan(lib, mode, H, n, n + int(2 ** rng.uniform(0, 15)), D, rng.choice([D, 64, 200]), rng.random() < 0.5)
        assert 4 * floats <= 20 << 20, (mode, H, D, n, each)
        cut += floats > 0
    assert cut > 1000
    # decode rows beside four portions of 2000 rows in all
    for n in (4, 68):
        each, floats = plan(lib, "light", 64, n, n + 2000, 128)
        assert 0 < 4 * floats <= 20 << 20


def segments_of(n, seg_rows, chunk=32, most=16):
    """As segments.h counts them."""
    k = max(1, min(most, (n + seg_rows // 3) // seg_rows))
    each = -(-(-(-n // k)) // chunk) * chunk
    return -(-n // each)


def test_places_and_workgroups_suffice():
    """Segments of cut portions within 6 / 5 rows / seg_rows, all of them within rows / seg_rows and the portions."""
    rng = random.Random(2)
    for _ in range(20000):
        seg = 32 * rng.randint(3, 40)
        lens = [int(2 ** rng.uniform(0, 12)) for _ in range(rng.randint(1, 40))]
        if rng.random() < 0.3:
            lens = [max(1, 5 * seg // 3 + rng.randint(-2, 2))] * rng.randint(1, 8)
        own = [segments_of(n, seg) for n in lens]
        assert sum(k for k in own if k > 1) <= 6 * sum(lens) // (5 * seg), (seg, lens)
        assert sum(own) <= sum(lens) // seg + len(lens)


# the steps named beside the rule: mode, heads, portions, rows in all, channels, fp32 rows
HERE = [("gla", 64, 3, 120, 64, 0), ("gla", 64, 16, 1120, 64, 0), ("gla", 64, 8, 2000, 64, 0), ("gla", 16, 16, 320, 64, 0), ("light", 64, 8, 2000, 64, 0),
        ("gla", 64, 8, 560, 128, 0), ("gla", 16, 8, 320, 128, 0), ("light", 64, 3, 300, 128, 0), ("gla", 16, 1, 2000, 64, 0), ("gla", 32, 2, 1000, 64, 0),
        ("light", 16, 1, 2000, 64, 0), ("light", 64, 2, 4096, 64, 0), ("gla", 64, 1, 300, 64, 0), ("gla", 16, 5, 1589, 64, 0), ("light", 16, 11, 3901, 64, 0),
        ("gla", 16, 4, 760, 64, 1), ("light", 16, 8, 4000, 64, 0), ("mlstm", 64, 3, 120, 64, 0), ("mlstm", 16, 8, 160, 64, 0), ("mlstm", 16, 16, 1000, 64, 0),
        ("mlstm", 64, 12, 900, 64, 1), ("mlstm", 64, 3, 300, 64, 0), ("mlstm", 32, 8, 664, 64, 0), ("mlstm", 64, 3, 900, 64, 1), ("mlstm", 64, 8, 4000, 64, 1),
        ("mlstm", 32, 1, 661, 64, 0), ("mlstm", 16, 1, 2000, 64, 0), ("mlstm", 32, 17, 2016, 64, 0), ("mlstm", 32, 3, 1377, 64, 0)]
THERE = [("gla", 16, 8, 160, 64, 0), ("gla", 4, 4, 912, 128, 1), ("gla", 16, 10, 100, 64, 0), ("gla", 16, 1, 300, 128, 0), ("gla", 16, 1, 250, 64, 0), ("light", 16, 3, 300, 64, 0),
         ("mlstm", 32, 5, 3000, 64, 0), ("mlstm", 64, 5, 3065, 64, 0), ("mlstm", 64, 67, 3232, 64, 0), ("mlstm", 16, 1, 2000, 128, 0), ("mlstm", 64, 2, 5438, 64, 1),
         ("mlstm", 32, 3, 1605, 64, 1), ("mlstm", 32, 94, 1639, 64, 1)]


@pytest.mark.parametrize("mode,H,n,rows,D,fp32", HERE + THERE)
def test_rule(lib, mode, H, n, rows, D, fp32):
    assert bool(plan(lib, mode, H, n, rows, D, fp32=bool(fp32))[0]) == ((mode, H, n, rows, D, fp32) in HERE)


def test_long_portions_are_cut(lib):
    """One portion that may have most of the rows gets a launch of its states; alike ones among few heads are cut fine enough to fill the chip."""
    for mode, H, n, rows, D in (("gla", 16, 1, 2000, 64), ("light", 16, 8, 4000, 64), ("light", 64, 8, 2000, 64), ("light", 32, 4, 758, 128), ("gla", 16, 500, 2754, 64),
                                ("mlstm", 32, 17, 2016, 64), ("gla", 64, 501, 4500, 64), ("light", 32, 4, 698, 128), ("light", 32, 10, 674, 128), ("light", 32, 6, 806, 64),
                                ("light", 64, 3, 900, 64), ("mlstm", 16, 7, 603, 64), ("mlstm", 32, 14, 750, 64)):
        each, floats = plan(lib, mode, H, n, rows, D)
        assert 0 < each <= max(128, rows * H // 256 + 31) and floats > 0
    for mode, H, n, rows, D in (("gla", 64, 3, 300, 64), ("gla", 64, 8, 560, 128), ("light", 64, 3, 480, 64), ("mlstm", 64, 3, 300, 64), ("gla", 64, 203, 3747, 128)):
        assert plan(lib, mode, H, n, rows, D) == (1 << 29, 0)
