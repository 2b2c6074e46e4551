"""Which INT4 kernel a call takes: the one measured faster on each side of every line (no GPU needed).

The times beside a case are of the register kernel and of the one named
(MI355X, graph-replayed, weights from HBM, us), forced in turn.
"""

from __future__ import annotations

import ctypes

import pytest

from nanoserve_amd import _lib
from tests._helpers import INT4_STREAM_CASES, int4_kernel

REGISTER, STREAM, TILED = _lib.NS_INT4_REGISTER, _lib.NS_INT4_STREAM, _lib.NS_INT4_TILED


@pytest.mark.parametrize("N,K,M,want", [
    (4096, 896, 32, REGISTER),      # 5.50 / 6.55
    (4096, 1024, 32, REGISTER),     # 5.90 / 6.71
    (4096, 1024, 48, STREAM),       # 8.10 / 6.72
    (4864, 896, 48, REGISTER),      # 6.72 / 7.62
    (4864, 896, 64, STREAM),        # 8.25 / 7.66
    (4864, 1024, 32, STREAM),       # 8.16 / 6.68
    (6144, 896, 48, STREAM),        # 8.27 / 7.52
    (9728, 896, 16, REGISTER),      # 6.98 / 6.90 at best, slower below
    (9728, 896, 32, STREAM),        # 8.37 / 7.65
    (9728, 896, 48, STREAM),        # 10.43 / 9.92
    (9728, 896, 64, STREAM),        # 12.37 / 9.89
    (9728, 896, 128, STREAM),       # 30.45 / 18.41
    (11008, 896, 48, REGISTER),     # 11.99 / 13.60
    (14336, 896, 48, REGISTER),     # 14.07 / 14.90
    (14336, 896, 64, STREAM),       # 16.83 / 15.16
    (24576, 896, 48, REGISTER),     # 20.93 / 23.15
    (28672, 896, 48, REGISTER),     # 23.77 / 27.17
    (28672, 896, 64, STREAM),       # 29.61 / 27.46
    (28672, 1024, 48, STREAM),      # 30.36 / 27.48
    (1152, 896, 32, REGISTER),      # 3.95 / 5.97
    (1152, 896, 64, REGISTER),      # 4.98 / 6.47
    (1152, 896, 65, STREAM),        # 7.62 / 6.48
    (1152, 1024, 128, STREAM),      # 8.50 / 6.71
    (1152, 896, 129, REGISTER),     # the tiled GEMM fuses no norm, the stream holds 128 rows
])
def test_projections_behind_a_norm_take_the_faster_kernel(N, K, M, want):
    assert int4_kernel(M, N, K, norm=True)[0] == want


@pytest.mark.parametrize("N,K,M,want", [
    (512, 1152, 1, REGISTER),       # 3.48 / 3.81
    (12288, 1152, 1, REGISTER),     # 5.57 / 6.58
    (12288, 1152, 6, REGISTER),     # 6.08 / 6.58
    (12288, 1152, 12, STREAM),      # 7.05 / 6.70
    (16384, 1152, 1, STREAM),       # 8.54 / 7.98
    (1536, 1408, 1, REGISTER),      # 4.05 / 4.21
    (8192, 1664, 1, REGISTER),      # 5.92 / 6.34
    (512, 1920, 1, REGISTER),       # 3.89 / 4.16
    (512, 1536, 1, STREAM),         # 3.95 / 3.83
    (8192, 1536, 6, STREAM),        # 6.17 / 5.69
    (512, 2176, 1, STREAM),         # 5.99 / 4.31
    (896, 4864, 1, STREAM),
    (28672, 3584, 128, STREAM),
    (896, 4864, 129, TILED),
    (896, 896, 16, REGISTER),       # up to 1024 without a norm
])
def test_long_k_calls_take_the_faster_kernel(N, K, M, want):
    assert int4_kernel(M, N, K)[0] == want


@pytest.mark.parametrize("K,gs", [(4864, 64), (4864, 32), (4896, 32), (1280, 64)])
def test_small_groups_and_part_chunks_keep_the_register_kernel(K, gs):
    for M in (1, 16, 33, 128):
        assert int4_kernel(M, 896, K, gs)[0] == REGISTER


@pytest.mark.parametrize("N,K,M,tokens,features", [
    (1152, 896, 2600, 64, 64),      # 15.6; 128 x 64 16.5
    (1152, 896, 3600, 64, 64),      # 23.2; 128 x 64 26.6, 128 x 128 24.8
    (1024, 1024, 2800, 64, 64),     # 16.7; 128 x 64 17.8
    (1024, 1024, 3000, 64, 64),     # 17.0; 128 x 64 17.9
    (2048, 1024, 1400, 64, 64),     # 17.0; 128 x 64 18.0
    (2048, 1024, 2048, 128, 64),    # 18.7; 64 x 64 23.2
    (1536, 1536, 1200, 64, 64),     # 18.5; 128 x 64 19.5
    (1536, 1536, 2048, 64, 64),     # 23.0; 128 x 64 23.9
    (3072, 896, 1400, 64, 64),      # 24.7; 128 x 128 25.6
    (9728, 896, 2048, 128, 128),
    (1536, 8960, 1800, 128, 64),
])
def test_the_tiled_gemm_takes_the_faster_tiles(N, K, M, tokens, features):
    """Unsplit times per tile shape, us."""
    assert int4_kernel(M, N, K)[:3] == (TILED, tokens, features)


def test_the_stream_cases_take_every_shape_the_rule_can_pick():
    """The GPU tests run each of INT4_STREAM_CASES: they must take the shapes they
    stand for, and no layer may take a shape that is not among them."""
    for tile, (few, phases, split) in INT4_STREAM_CASES.items():
        for N, K, M in (few, phases):
            assert int4_kernel(M, N, K) == (STREAM, *tile, 1)
        N, K, M = split
        got = int4_kernel(M, N, K, workspace=True)
        assert got[:3] == (STREAM, *tile) and got[3] > 1
        assert phases[1] // 128 > 32
    taken = set()
    for K in (1152, 1280, 2048, 3584, 4864, 8192, 14336):
        for N in [*range(16, 2048, 48), *range(2048, 30000, 208), 65536, 151936]:
            for M in (1, 8, 16, 17, 32, 33, 48, 64, 65, 100, 128):
                for workspace in (False, True):
                    kind, *tile, _ = int4_kernel(M, N, K, workspace=workspace)
                    if kind == STREAM:
                        taken.add(tuple(tile))
    assert taken == set(INT4_STREAM_CASES)


def test_the_normed_stream_takes_two_to_five_feature_tiles():
    taken = {int4_kernel(M, N, K, norm=True)[1:3] for K in (896, 1024) for N in range(1152, 30000, 112)
             for M in (17, 32, 33, 48, 64, 65, 100, 128) if int4_kernel(M, N, K, norm=True)[0] == STREAM}
    assert taken == {(32, 32), (32, 48), (32, 64), (32, 80)}


def test_kernel_query_refuses_what_the_call_refuses():
    lib = _lib.load()
    t, f, s = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int32()
    out = (ctypes.byref(t), ctypes.byref(f), ctypes.byref(s))
    assert lib.ns_int4_linear_kernel(0, 896, 896, 128, 0, 0, *out) == _lib.NS_ERR_INVALID_ARG
    assert lib.ns_int4_linear_kernel(1, 896, 896, 128, 0, 0, None, *out[1:]) == _lib.NS_ERR_INVALID_ARG
    for N, K, gs, norm in ((24, 896, 128, 0), (896, 900, 100, 0), (896, 896, 48, 0), (896, 1152, 128, 1)):
        assert lib.ns_int4_linear_kernel(1, N, K, gs, norm, 0, *out) == _lib.NS_ERR_UNSUPPORTED
