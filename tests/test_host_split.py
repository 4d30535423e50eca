"""luma_split_plan, the rule that shares a small set out (LUMA_FLAG_SPLIT):
where medium tensors get a workgroup each and how far records are split, at
the sizes on both sides of its lines, and the limits that the kernels and the
workspace rely on."""

import ctypes
import random

import numpy as np
import pytest

from luma_amd import _lib as L
from luma_amd.optimizer import _Engine


@pytest.fixture(scope="module")
def lib():
    return L.load()


def plan(lib, records, medium, small, longest, c=16384):
    wide = ctypes.c_int32(7)
    shift = lib.luma_split_plan(records, medium, small, longest, c, ctypes.byref(wide))
    assert wide.value in (0, 1)
    return shift, wide.value


# (records, medium, small, longest) -> (shift, wide), where each was measured
# faster than the other forms (luma_split_plan's comment)
@pytest.mark.parametrize("of,want", [
    ((0, 30, 0, 8192), (3, 1)), ((0, 100, 0, 512), (2, 1)), ((0, 100, 0, 8192), (2, 1)),
    ((0, 120, 0, 8000), (2, 1)), ((0, 121, 0, 8000), (1, 1)), ((0, 204, 0, 8000), (1, 1)),
    ((0, 205, 0, 8000), (0, 1)), ((0, 400, 0, 512), (0, 1)), ((0, 500, 0, 8192), (0, 1)), ((0, 700, 0, 512), (0, 0)),
    ((0, 1200, 0, 4096), (0, 0)), ((0, 1200, 0, 8192), (0, 1)),
    ((0, 2000, 0, 512), (0, 0)), ((0, 2000, 0, 8192), (0, 0)),
    ((0, 431, 569, 700), (0, 0)),          # small tensors' workgroups count too
    ((100, 300, 0, 512), (2, 0)),          # short medium tensors: wavefronts beside the parts
    ((100, 300, 0, 8192), (0, 1)), ((100, 100, 0, 2048), (1, 1)),
    ((20, 300, 0, 2048), (3, 0)), ((60, 300, 0, 2048), (1, 0)),
    ((800, 300, 0, 2048), (0, 0)), ((800, 600, 0, 8192), (0, 1)),
    ((1500, 600, 0, 8192), (0, 0)),        # beyond the measured sets
    ((0, 0, 1000, 0), (0, 0)),
    # records alone: one round of workgroups
    ((13, 0, 0, 0), (3, 0)), ((48, 0, 0, 0), (3, 0)), ((49, 0, 0, 0), (2, 0)),
    ((192, 0, 0, 0), (2, 0)), ((193, 0, 0, 0), (1, 0)), ((408, 0, 0, 0), (1, 0)),
    ((409, 0, 0, 0), (0, 0)), ((500, 0, 0, 0), (0, 0)),
])
def test_rule(lib, of, want):
    assert plan(lib, *of) == want


def test_records_alone_and_unknown_longest(lib):
    for r in (0, 1, 48, 49, 192, 193, 408, 409, 5000):
        assert lib.luma_split_shift(r, 16384) == plan(lib, r, 0, 0, 0)[0]
    for r, m in ((0, 100), (0, 1200), (0, 2000), (800, 600)):
        assert plan(lib, r, m, 0, 0) == plan(lib, r, m, 0, L.MEDIUM_TENSOR)
    assert lib.luma_split_plan(5, 5, 5, 500, 16384, None) == plan(lib, 5, 5, 5, 500)[0]


def test_limits(lib):
    """The workspace has room for SPLIT_CHUNKS parts, and no part is shorter
    than the shortest chunk."""
    rng = random.Random(1)
    for _ in range(20000):
        r, m, s = (rng.choice([0, rng.randrange(1, 30), rng.randrange(1, 3000)]) for _ in range(3))
        c = 1 << rng.randrange(11, 18)
        shift, wide = plan(lib, r, m, s, rng.randrange(257, 8193), c)
        n = r + (m if wide else 0)
        assert shift == 0 or (0 < n << shift <= L.SPLIT_CHUNKS and c >> shift >= 2048)


def test_engine_plans_as_the_library_launches(lib):
    """summary_chunk derives the counts from the sizes as the chunk table has
    them."""
    eng = object.__new__(_Engine)
    eng.lib, eng.chunk_elems, eng.split = lib, 0, True
    eng.small_tensors = eng.medium_tensors = True
    for sizes in ([300, 9, 8192, 8193, 16385, 70000], [257] * 2000, [512] * 100 + [3] * 50,
                  [300000] * 20 + [400] * 300, [200]):
        numels = np.array(sizes, dtype=np.int64)
        c = eng.chunk_for(numels)
        _, ch, n_small, n_medium = eng.chunk_layout(numels, c)
        med = [n for n in sizes if L.SMALL_TENSOR < n <= L.MEDIUM_TENSOR]
        shift, _ = plan(lib, len(ch) - n_small - n_medium, n_medium, n_small, max(med, default=0), c)
        assert eng.summary_chunk(numels) == c >> shift
