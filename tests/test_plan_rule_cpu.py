"""The plan rule for shapes outside the dispatch table (host code only): every
plan is one the library accepts as an explicit configuration and resolves to
itself, and its split-K scratch fits the static scratch wherever one split's
does many times over."""

from __future__ import annotations

import ctypes
import random

import pytest

from kernels import _lib
from kernels._lib import GemmConfig

NONE, SILU = _lib.EPILOGUE_NONE, _lib.EPILOGUE_SILU_MUL


def _shapes(seed, count):
    rng = random.Random(seed)
    for _ in range(count):
        N = 2 * int(2 ** rng.uniform(0, 16))
        K = 8 * int(2 ** rng.uniform(0, 11.5))
        yield rng.choice([1, 2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 24, 32, 33, 48, 49, 64, 65, 128, 200]), N, K


@pytest.mark.parametrize("epi", [NONE, SILU])
def test_plans_resolve_to_themselves(epi):
    lib = _lib.load()
    for M, N, K in _shapes(5 + epi, 4000):
        plan, got = GemmConfig(), GemmConfig()
        assert lib.krk_gemm_plan(M, N, K, epi, ctypes.byref(plan)) == 0
        rc = lib.krk_gemm_resolve(M, N, K, epi, ctypes.byref(plan), ctypes.byref(got))
        assert rc == 0, (M, N, K, plan.as_dict(), _lib.last_error())
        assert got.as_dict() == plan.as_dict(), (M, N, K)
        c = plan.as_dict()
        ws = lib.krk_gemm_workspace_bytes(M, N, K, epi)
        assert (ws > 0) == (c["splits"] > 1), (M, N, K, c)
        assert c["splits"] <= max(1, -(-K // 256)), (M, N, K, c)


@pytest.mark.parametrize("M,N,K,epi,cfg", [
    (64, 10106, 8192, SILU, {"kernel": _lib.KERNEL_STREAM}),           # the plan is LDS-staged with K whole
    (200, 96224, 14336, NONE, {"kernel": _lib.KERNEL_STREAM, "unroll": 2}),
    (200, 96224, 14336, SILU, {"kernel": _lib.KERNEL_MFMA_LDS, "unroll": 3}),   # the plan has four weight tiles
    (13, 58940, 8192, SILU, {"kernel": _lib.KERNEL_MFMA_LDS, "k_chunk": 512, "m_tiles": 2}),
    (33, 73576, 992, NONE, {"kernel": _lib.KERNEL_MFMA_LDS, "k_chunk": 512, "splits": 4}),
    (12, 21042, 9728, SILU, {"channels": 8, "k_chunk": 512}),
    (12, 300, 88, NONE, {"k_chunk": 256}),                             # the plan is wave-sliced
    (4, 20, 4096, NONE, {"unroll": 5}),
    (128, 80648, 14336, SILU, {"unroll": 7, "splits": 7}),
    (5, 68, 14336, NONE, {"splits": 1, "n_tiles": 1}),                 # the plan splits K on the VALU kernel
    (32, 2528, 4176, NONE, {"splits": 5}),
    (64, 127376, 656, SILU, {"splits": 3}),                            # the plan is the stream kernel, of two K stages
    (128, 24400, 408, SILU, {"kernel": _lib.KERNEL_MFMA_LDS, "channels": 24, "splits": 2}),
])
def test_partial_configurations_are_completed(M, N, K, epi, cfg):
    """A configuration that names only some fields runs where some choice of
    the others does, whatever the plan's are, and keeps the named ones."""
    lib = _lib.load()
    given, got, again = GemmConfig.from_dict(cfg), GemmConfig(), GemmConfig()
    assert lib.krk_gemm_resolve(M, N, K, epi, ctypes.byref(given), ctypes.byref(got)) == 0, _lib.last_error()
    out = got.as_dict()
    assert {k: out[k] for k in cfg} == cfg
    assert lib.krk_gemm_resolve(M, N, K, epi, ctypes.byref(got), ctypes.byref(again)) == 0
    assert again.as_dict() == out


@pytest.mark.parametrize("M,N,K,epi,stream", [
    (44, 153720, 792, NONE, True), (51, 153320, 384, NONE, True), (49, 115344, 568, NONE, True),   # aligned rows of y
    (41, 2 * 34784, 352, SILU, True), (37, 2 * 52032, 816, SILU, True), (64, 2 * 31272, 760, SILU, True),
    (43, 2 * 53938, 968, SILU, True), (36, 2 * 26268, 488, SILU, True), (36, 2 * 26268, 512, SILU, True),   # others
    (35, 2 * 33174, 760, SILU, True), (45, 2 * 41095, 376, SILU, True), (49, 2 * 9943, 1016, SILU, True),
    (62, 2 * 48697, 256, SILU, False), (52, 2 * 14497, 576, SILU, False), (62, 2 * 26268, 488, SILU, False),
    (44, 144278, 200, NONE, False), (44, 65528, 792, NONE, False), (32, 153720, 792, NONE, False),
    (64, 2 * 9000, 1000, SILU, True), (49, 2 * 10016, 776, SILU, True),   # where the tile kernel is the other choice
    (60, 2 * 8200, 640, SILU, False), (49, 2 * 9047, 784, SILU, False), (48, 2 * 9000, 640, SILU, True),
])
def test_wide_shapes_of_a_short_k(M, N, K, epi, stream):
    """33-64 rows below K = 1024: the stream kernel where it measured faster."""
    plan = GemmConfig()
    assert _lib.load().krk_gemm_plan(M, N, K, epi, ctypes.byref(plan)) == 0
    assert plan.kernel == (_lib.KERNEL_STREAM if stream else _lib.KERNEL_MFMA_LDS), plan.as_dict()


@pytest.mark.parametrize("M,N,K,epi,splits", [
    (1, 600, 15752, SILU, 8), (1, 10, 9736, SILU, 20), (8, 48, 3504, SILU, 7), (7, 20, 2632, SILU, 6),
    (3, 2390, 14184, SILU, 3), (1, 300, 15880, NONE, 8), (5, 26, 13640, NONE, 27), (8, 36, 7888, NONE, 16),
    (3, 210, 14600, NONE, 12), (4, 16, 14704, NONE, 29),
    (1, 320, 12296, SILU, 15), (7, 400, 15528, NONE, 12), (3, 1550, 12656, SILU, 4),
    (1, 160, 12296, SILU, 1), (1, 300, 12296, NONE, 1), (3, 44, 9688, NONE, 1),
])
def test_few_channels_of_a_long_k(M, N, K, epi, splits):
    """Up to 8 rows: K is split where a few blocks would each walk all of it."""
    plan = GemmConfig()
    assert _lib.load().krk_gemm_plan(M, N, K, epi, ctypes.byref(plan)) == 0
    assert plan.splits == splits, plan.as_dict()
    assert splits == 1 or plan.kernel == _lib.KERNEL_VALU


@pytest.mark.parametrize("M,N,K,epi,depth", [
    (1, 1002, 11624, NONE, 7), (1, 1002, 10240, NONE, 10), (1, 1002, 9728, NONE, 19), (2, 1600, 10752, NONE, 7),
    (1, 1600, 10752, SILU, 7), (1, 1600, 10240, SILU, 10), (1, 2 * 8912, 8880, SILU, 5), (1, 2 * 8912, 10300 // 8 * 8, SILU, 7),
])
def test_depth_past_one_pass(M, N, K, epi, depth):
    plan = GemmConfig()
    assert _lib.load().krk_gemm_plan(M, N, K, epi, ctypes.byref(plan)) == 0
    assert plan.kernel == _lib.KERNEL_VALU and plan.unroll == depth, plan.as_dict()


@pytest.mark.parametrize("M,N,K,stream", [
    (72, 132988, 520, True), (45, 114926, 688, True), (83, 158058, 512, True), (64, 144730, 200, False), (64, 65522, 520, False),
])
def test_selecting_calls_plan_for_aligned_logits(M, N, K, stream):
    """The workspace's rows of logits are aligned, whatever N is; a call with
    N one short of a multiple of 8 runs the plan of that multiple."""
    lib, plan, whole = _lib.load(), GemmConfig(), GemmConfig()
    for k in (1, 8):
        assert lib.krk_gemm_select_plan(M, N, K, k, ctypes.byref(plan)) == 0
        assert (plan.kernel == _lib.KERNEL_STREAM) == stream, plan.as_dict()
        if stream:
            assert lib.krk_gemm_select_plan(M, -(-N // 8) * 8, K, k, ctypes.byref(whole)) == 0
            assert plan.as_dict() == whole.as_dict()
            assert lib.krk_gemm_select_fused(M, N, K, k, None) == lib.krk_gemm_select_fused(M, N, K, k, ctypes.byref(plan))


@pytest.mark.parametrize("M,N,K,sliced", [
    (18, 1536, 4224, True), (32, 3584, 4608, True), (24, 4096, 5120, True), (32, 2560, 5120, True),
    (32, 512, 4608, False), (24, 4352, 4608, False), (32, 2560, 5632, False),
    (32, 2838, 4512, True),
    (30, 8126, 3352, False), (32, 6992, 3384, False), (30, 8126, 3360, True), (30, 8126, 2712, True), (24, 8126, 3352, True),
    (24, 1540, 4232, True), (24, 3072, 5112, True), (25, 2560, 4408, False), (24, 3208, 5016, False),
])
def test_two_x_tiles_of_a_long_k(M, N, K, sliced):
    plan = GemmConfig()
    assert _lib.load().krk_gemm_plan(M, N, K, NONE, ctypes.byref(plan)) == 0
    assert plan.kernel == (_lib.KERNEL_SLICE if sliced else _lib.KERNEL_MFMA_LDS), plan.as_dict()


@pytest.mark.parametrize("M,N,K,waves,rows", [
    (6, 65536, 512, 4, 2), (8, 10240, 1536, 4, 2), (8, 65536, 1024, 8, 2), (4, 65536, 512, 8, 2),
    (3, 4432, 3160, 4, 1), (3, 16390, 3160, 8, 2), (3, 8982, 3584, 8, 2),
])
def test_waves_of_many_channels(M, N, K, waves, rows):
    plan = GemmConfig()
    assert _lib.load().krk_gemm_plan(M, N, K, NONE, ctypes.byref(plan)) == 0
    assert (plan.kernel, plan.waves, plan.n_tiles) == (_lib.KERNEL_VALU, waves, rows), plan.as_dict()


@pytest.mark.parametrize("M,N,K", [(34, 1654, 752), (33, 1024, 64), (48, 2048, 1536), (64, 4096, 3072), (100, 3126, 1344)])
def test_argmax_of_few_channels_is_fused(M, N, K):
    lib, plan = _lib.load(), GemmConfig()
    assert lib.krk_gemm_select_fused(M, N, K, 1, None) == 1
    assert lib.krk_gemm_select_plan(M, N, K, 1, ctypes.byref(plan)) == 0
    assert lib.krk_gemm_select_fused(M, N, K, 1, ctypes.byref(plan)) == 1
    if N >= 8:
        assert lib.krk_gemm_select_fused(M, N, K, 8, None) == 0


def test_splits_beyond_64_rows():
    """A plan for more than 64 rows is the 64-row plan but for its splits, which
    size the workspace for the tile kernel's sums; what runs in launches of 64
    rows (a selecting call, a configuration with other fields than the plan's)
    splits K as the 64-row plan does."""
    lib = _lib.load()
    shapes = [(130, 2560, 4096), (192, 2560, 9728), (66, 1938, 7896), (112, 536, 10008)] + list(_shapes(17, 2000))
    for M, N, K in shapes:
        M = 65 + M % 192
        plan, base, got = GemmConfig(), GemmConfig(), GemmConfig()
        for epi in (NONE, SILU):
            assert lib.krk_gemm_plan(M, N, K, epi, ctypes.byref(plan)) == 0
            assert lib.krk_gemm_plan(64, N, K, epi, ctypes.byref(base)) == 0
            p, b = plan.as_dict(), base.as_dict()
            assert dict(p, splits=0) == dict(b, splits=0) and p["splits"] >= b["splits"], (M, N, K, epi)
            need, need64 = lib.krk_gemm_workspace_bytes(M, N, K, epi), lib.krk_gemm_workspace_bytes(64, N, K, epi)
            assert need64 <= need <= max(need64, 4 << 20), (M, N, K, epi)
            for cfg, splits in (({}, p["splits"]), ({"kernel": p["kernel"]}, p["splits"]), (p, p["splits"])):
                given = GemmConfig.from_dict(cfg)
                assert lib.krk_gemm_resolve(M, N, K, epi, ctypes.byref(given), ctypes.byref(got)) == 0
                assert got.as_dict() == dict(p, splits=splits), (M, N, K, epi, cfg)
            other = GemmConfig.from_dict(dict(p, unroll=5 - p["unroll"] if p["kernel"] == _lib.KERNEL_MFMA_LDS else 2, splits=0))
            if lib.krk_gemm_resolve(M, N, K, epi, ctypes.byref(other), ctypes.byref(got)) == 0 and got.unroll != plan.unroll:
                assert got.splits == b["splits"], (M, N, K, epi, got.as_dict())
        if N >= 8:
            assert lib.krk_gemm_select_plan(M, N, K, 8, ctypes.byref(plan)) == 0
            assert lib.krk_gemm_select_plan(64, N, K, 8, ctypes.byref(base)) == 0
            assert plan.as_dict() == base.as_dict(), (M, N, K, "select")


def test_split_scratch_stays_small():
    """The rule splits only narrow shapes: partial sums of at most 4 MB less
    the counters, so the allocation-free call takes every plan but the VALU
    kernel's for an x slice that fills LDS."""
    lib = _lib.load()
    for M, N, K in _shapes(11, 4000):
        plan = GemmConfig()
        assert lib.krk_gemm_plan(M, N, K, NONE, ctypes.byref(plan)) == 0
        c = plan.as_dict()
        if c["splits"] > 1 and not (c["kernel"] == _lib.KERNEL_VALU and c["m_tiles"] * K * 2 > 65536):
            assert c["splits"] * min(M, 64) * N * 4 <= (4 << 20) - (64 << 10), (M, N, K, c)
