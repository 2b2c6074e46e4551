"""Which prefill kernel a batch takes: the one measured faster on each side of every line (no GPU needed).

Each case gives the (context, new rows) of its multi-row sequences; the times
beside it are of one call with the narrow and the wide kernel forced (MI355X,
graph-replayed, us).
"""

from __future__ import annotations

import ctypes

import pytest

from nanoserve_amd import _lib
from tests._helpers import prefill_columns

D64, G16, D128, G8 = (14, 2, 64), (32, 2, 64), (28, 4, 128), (16, 2, 128)  # query heads, KV heads, head size


def _chunks(n, rows, context):
    return [(context * f // 100, rows) for f in {1: (100,), 2: (100, 75), 4: (100, 90, 80, 50)}[n]]


@pytest.mark.parametrize("seqs,heads,wide", [
    # Whole prompts, D = 128.
    ([(0, 2400)], D128, False),                                     # 99.9 / 107.2
    ([(0, 2600)], D128, False),                                     # 112.0 / 114.0
    ([(0, 3000)], D128, True),                                      # 139.0 / 125.9
    ([(0, 16000)], D128, True),
    ([(0, 4600)], G8, False),                                       # 169.8 / 179.1
    ([(0, 4800)], G8, False),                                       # 181.4 / 185.2
    ([(0, 5200)], G8, True),                                        # 211.3 / 201.0
    ([(0, 2450), (0, 150)], D128, False),                           # 97.5 / 104.5
    ([(0, 1400), (0, 1340)], D128, True),                           # 80.3 / 71.6
    ([(0, 700), (0, 640), (0, 669), (0, 693)], D128, True),         # 56.4 / 50.9
    ([(0, 3642), (0, 3718)], D128, True),                           # 421 / 337
    # Chunks behind a context, one round of wide blocks.
    (_chunks(1, 2048, 1000), D128, False),                          # 116.2 / 125.6
    (_chunks(1, 2300, 1000), D128, False),                          # 131.5 / 136.5
    (_chunks(1, 2048, 1300), D128, False),                          # 130.7 / 138.0
    (_chunks(1, 2048, 3000), D128, True),                           # 206.5 / 194.5
    (_chunks(1, 2048, 8000), D128, True),                           # 427.9 / 365.8
    (_chunks(1, 3584, 1750), G8, False),                            # 183.2 / 203.9
    (_chunks(1, 3584, 5250), G8, True),                             # 334.8 / 325.1
    (_chunks(2, 900, 500), D128, False),                            # 65.2 / 67.9
    (_chunks(2, 1540, 1225), G8, False),                            # 108.1 / 116.4
    (_chunks(2, 1024, 2000), D128, True),                           # 130.1 / 125.2
    (_chunks(4, 512, 700), D128, True),                             # 66.5 / 60.9
    (_chunks(1, 600, 8000), D128, False),                           # too few blocks
    # ... and past one round.
    (_chunks(1, 2450, 1000), D128, True),                           # 169.4 / 140.3
    (_chunks(1, 2600, 1000), D128, True),                           # 176.8 / 145.9
    (_chunks(2, 1300, 500), D128, True),                            # 108.0 / 85.5
    # Decode rows beside the chunks, D = 128.
    (_chunks(2, 1024, 4000) + [(1000, 1)] * 48, D128, True),        # 242.9 / 216.8
    ([(0, 2048)] + [(1000, 1)] * 48, D128, False),                  # 104.7 / 108.9
    # D = 64.
    ([(0, 8192)], D64, False),                                      # 216.9 / 265.1
    ([(0, 16000)], D64, True),                                      # 720.3 / 670.9
    ([(0, 1850 - 13 * i) for i in range(6)], D64, False),           # 97.3 / 104.3
    ([(0, 1850 - 13 * i) for i in range(10)], D64, True),           # 155.5 / 150.5
    (_chunks(1, 14100, 10000), D64, False),                         # 1398.5 / 1420.9
    (_chunks(1, 18000, 10000), D64, True),                          # 1840.8 / 1780.1
    (_chunks(1, 6800, 8000), G16, False),                           # 993.8 / 1029.6
    (_chunks(1, 7500, 8000), G16, True),                            # 1148.0 / 1094.0
    # The blocks of short chunks are mostly empty; decode rows alone have none.
    ([(100, 3)] * 200, D128, False),
    ([(100, 1)] * 64, D64, False),
])
def test_the_faster_width_is_taken(seqs, heads, wide):
    want = {64: (128, 384), 128: (128, 256)}[heads[2]][wide]
    assert prefill_columns(seqs, heads) == want


def test_more_sequences_than_the_schedule_lists_take_the_narrow_kernel():
    assert prefill_columns([(0, 64)] * 256, (128, 8, 128)) == 256
    assert prefill_columns([(0, 64)] * 257, (128, 8, 128)) == 128


def test_bad_arguments_are_refused():
    lib = _lib.load()
    one, two = (ctypes.c_int64 * 1)(5), (ctypes.c_int64 * 2)(0, 5)
    assert lib.ns_paged_prefill_columns(None, 1, two, 1, 1, 14, 2, 64) == _lib.NS_ERR_INVALID_ARG
    assert lib.ns_paged_prefill_columns(one, 1, None, 1, 1, 14, 2, 64) == _lib.NS_ERR_INVALID_ARG
    assert lib.ns_paged_prefill_columns(one, 1, two, 1, 1, 15, 2, 64) == _lib.NS_ERR_INVALID_ARG
    assert lib.ns_paged_prefill_columns(one, 1, two, 1, 1, 14, 2, 96) == _lib.NS_ERR_UNSUPPORTED
    assert lib.ns_paged_prefill_columns(one, 1, two, 1, 1, 64, 2, 64) == _lib.NS_ERR_UNSUPPORTED
