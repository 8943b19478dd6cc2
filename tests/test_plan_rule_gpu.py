"""GPU parity of the plan rule for shapes outside the dispatch table, on both
sides of each of its lines (rows, channels per CU, K) and at ragged sizes,
against the oracle."""

from __future__ import annotations

import pytest
import torch

from kernels import gemm as G
from oracle import gemm_ref as R
from test_gemm_gpu import _check_selection, assert_parity, check_gateup, check_linear, krk_select, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (1, 700, 3000), (1, 2562, 2504), (1, 4100, 4616), (2, 2050, 2560), (2, 300, 5640),   # VALU
    (3, 515, 1032), (3, 4097, 1032), (4, 8201, 2048), (6, 8200, 512), (8, 8203, 1536), (4, 2500, 3080), (8, 8300, 1000),  # VALU / wave-sliced
    (5, 255, 72), (12, 4096, 1416), (13, 4104, 1416), (16, 8192, 520), (32, 8200, 520), (8, 8300, 2056),
    (18, 1530, 4224), (32, 4096, 5120), (24, 1540, 4616), (17, 3072, 5112), (30, 8126, 3352),                # wave-sliced, two x tiles
    (9, 600, 6672), (17, 1800, 4104), (24, 3300, 4104), (32, 500, 5128),                   # LDS-staged, split
    (33, 1023, 1536), (33, 1024, 3072), (64, 2047, 2048), (48, 2048, 3080), (40, 5000, 1544), (64, 9000, 1528),
    (1, 1002, 11624), (2, 1600, 10256), (1, 3, 11272), (5, 26, 13640), (8, 36, 7888), (3, 210, 14600),  # few channels, long K
    (7, 400, 15528), (3, 4432, 3160), (4, 16390, 3160),
    (16, 16390, 1024), (33, 16400, 1000), (33, 65536, 264), (49, 65544, 1016),              # stream
])
def test_rule_plans(device, M, N, K):
    x, w = R.randn_bf16((M, K), 8100 + M + N), R.randn_bf16((N, K), 8200 + K, 0.02)
    check_linear(x, w, f"rule {G.plan(M, N, K)}")


@pytest.mark.parametrize("M,I,K", [
    (1, 1025, 2824), (2, 300, 5640), (4, 2100, 1544), (6, 310, 4104), (8, 1201, 2560),     # VALU
    (1, 300, 15752), (1, 5, 9736), (8, 24, 3504), (7, 10, 2632), (3, 1195, 14184),         # few channels, long K
    (1, 4100, 8880), (1, 4100, 10296), (8, 850, 7176),
    (9, 4097, 520), (16, 300, 2560), (17, 2050, 4096), (32, 1300, 3600), (32, 500, 1800),  # LDS-staged
    (33, 1200, 1000), (33, 1201, 1000), (64, 4500, 1032), (40, 8300, 1032),                # stream / LDS-staged
    (36, 8200, 264), (48, 8195, 512), (64, 8200, 776), (50, 10248, 264), (64, 8199, 1016),
])
def test_rule_gateup_plans(device, M, I, K):
    x, w = R.randn_bf16((M, K), 8300 + M + I), R.randn_bf16((2 * I, K), 8400 + K, 0.02)
    check_gateup(x, w, f"rule {G.plan(M, 2 * I, K, 1)}")


@pytest.mark.parametrize("M,N,K", [(33, 1024, 64), (40, 2047, 520), (64, 4095, 1536), (100, 1554, 3072), (49, 3009, 776)])
def test_fused_argmax_of_few_channels(device, M, N, K):
    """Argmax in the epilogue on half-padded weight tiles: the oracle's choice
    among the call's own logits, with equal maxima in one row and NaN in another,
    and the same without the logits."""
    x, w = R.randn_bf16((M, K), 8500 + M), R.randn_bf16((N, K), 8600 + N, 0.02)
    w[N - 1], w[17] = w[5], w[5]      # equal logits in every row
    x[M - 1, K - 1] = float("nan")
    assert G.select_fused(M, N, K, 1)
    say("fused argmax", M, N, K)
    idx, vals, logits = krk_select(x, w, 1)
    _check_selection(idx, vals, logits, 1, f"argmax M={M} N={N} K={K}")
    assert_parity(logits[:M - 1], R.linear_bf16(x[:M - 1], w), "logits")
    if M <= 64:  # the plain call's logits bit for bit
        plain = check_linear(x[:M - 1], w, "plain") if M - 1 > 32 else None
        assert plain is None or torch.equal(plain, logits[:M - 1])
    again, _, _ = krk_select(x, w, 1, logits=False)
    assert again.tolist() == idx.tolist()


@pytest.mark.parametrize("M,N,K,k", [(70, 65537, 264, 1), (33, 65541, 520, 8)])
def test_selection_with_unaligned_rows(device, M, N, K, k):
    """N not a multiple of 8: the stream kernel's logits in the aligned rows of
    the workspace and in the caller's unaligned ones select alike."""
    x, w = R.randn_bf16((M, K), 8700 + M), R.randn_bf16((N, K), 8800 + K, 0.02)
    say("selection, unaligned rows", M, N, K, k)
    idx, vals, logits = krk_select(x, w, k)
    _check_selection(idx, vals, logits, k, f"select M={M} N={N} K={K} k={k}")
    assert_parity(logits, R.linear_bf16(x, w), "logits")
    again, v2, _ = krk_select(x, w, k, logits=False)
    assert again.tolist() == idx.tolist() and v2.tolist() == vals.tolist()
