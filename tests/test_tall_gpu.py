"""GPU parity of calls of more than 64 rows, which run launches of up to 128
rows on the tile kernel (csrc/krk_tile.h): row counts at the edges of its
16-row tiles and of a launch, channels and K that fill no tile or stage,
split and whole K, strided operands, infinities and NaN, against the oracle.
The bar is the library's: |y - ref| <= 2e-2 + 1e-2·|ref|, and every plain
output a rounding of some fp32 sum of the exact products.
"""

from __future__ import annotations

import pytest
import torch

from kernels import _lib
from kernels import gemm as G
from oracle import gemm_ref as R
from test_gemm_gpu import assert_fp32_rounding, assert_parity, check_gateup, check_linear, krk, say

pytestmark = pytest.mark.gpu

NONE, SILU = _lib.EPILOGUE_NONE, _lib.EPILOGUE_SILU_MUL


@pytest.mark.parametrize("M,N,K", [
    (65, 96, 2560), (80, 250, 520), (96, 33, 136), (97, 2560, 4096), (128, 2560, 1416), (112, 6144, 264),
    (66, 40, 72), (128, 3, 8), (129, 100, 1000), (193, 18, 2568), (256, 21000, 128), (128, 2560, 9728),
    (104, 70, 9728), (128, 400, 9728), (97, 3500, 4104), (130, 1938, 7896),   # K splits of few channels
])
def test_rows_beyond_64(device, M, N, K):
    x = R.randn_bf16((M, K), 9100 + M)
    w = R.randn_bf16((N, K), 9200 + N, 0.02)
    check_linear(x, w, f"tall M={M} N={N} K={K}")


@pytest.mark.parametrize("M,I,K", [(65, 24, 2560), (96, 1, 40), (97, 333, 1000), (128, 1216, 2560), (130, 70, 136),
                                   (65, 33, 6144), (120, 307, 9600), (97, 2017, 4104)])  # K splits of few channels
def test_gateup_rows_beyond_64(device, M, I, K):
    x = R.randn_bf16((M, K), 9300 + M)
    wgu = R.randn_bf16((2 * I, K), 9400 + I, 0.02)
    check_gateup(x, wgu, f"tall gateup M={M} I={I} K={K}")


@pytest.mark.parametrize("M,N,K,epi", [(128, 4096, 7320, NONE), (100, 4040, 9728, NONE), (200, 2 * 2040, 7168, SILU)])
def test_long_k_beside_too_many_channels_to_split(device, M, N, K, epi):
    """Two K splits of whole tiles do not fit the scratch of these calls, and
    K is long: launches of 64 rows, which split it, are faster.  Their results
    are those of 64-row calls bit for bit (up to the last launch of 200 rows,
    whose 72 rows fit)."""
    say("launches of 64", M, N, K, epi)
    x, w = R.randn_bf16((M, K), 9260 + M).to(device), R.randn_bf16((N, K), 9360 + K, 0.02).to(device)
    make = (lambda m: G.SkinnyGateUp(m, N // 2, K, device)) if epi == SILU else (lambda m: G.SkinnyMatmul(m, N, K, device))
    assert G.plan(64, N, K, epi)["splits"] > 1
    y = make(M)(x, w)
    assert torch.equal(y[:64], make(64)(x[:64], w))
    if M <= 128:
        assert torch.equal(y[64:], make(64)(torch.cat([x[64:], x[:128 - M]]), w)[:M - 64])
    ref = R.gateup_bf16(x.cpu(), w.cpu()) if epi == SILU else R.linear_bf16(x.cpu(), w.cpu())
    assert_parity(y.cpu(), ref, "launches of 64")


@pytest.mark.parametrize("M,N,K,epi", [
    (49, 16385, 72, NONE), (64, 20480, 520, NONE), (63, 18000, 2568, NONE),
    (49, 2 * 8193, 136, SILU), (64, 2 * 10240, 264, SILU), (60, 2 * 9001, 2632, SILU),
])
def test_49_to_64_rows(device, M, N, K, epi):
    """The shapes that run on the tile kernel below 65 rows, at the ends of
    their ranges: 65-80 plain or 33-40 SwiGLU channels per CU under an LDS-staged
    plan with K whole."""
    plan, per_cu = G.plan(M, N, K, epi), -(-N // 256) / (2 if epi == SILU else 1)
    assert plan["kernel"] == _lib.KERNEL_MFMA_LDS and plan["splits"] == 1, plan
    assert (32 < per_cu <= 40) if epi == SILU else (64 < per_cu <= 80)
    x, w = R.randn_bf16((M, K), 9250 + M), R.randn_bf16((N, K), 9350 + N, 0.02)
    (check_gateup if epi == SILU else check_linear)(x, w, f"tile M={M} N={N} K={K}")


@pytest.mark.parametrize("M,N,K,ypad", [(100, 77, 520, 3), (128, 2560, 1024, 4), (70, 64, 264, 1)])
def test_strided_operands(device, M, N, K, ypad):
    """Row strides past the operands' widths; y with rows that are not 8-byte
    aligned.  Nothing outside y's rows may be written."""
    say("strided", M, N, K, ypad)
    x, w = R.randn_bf16((M, K), 9500 + M), R.randn_bf16((N, K), 9600 + N, 0.02)
    xd = torch.full((M, K + 24), float("nan"), dtype=torch.bfloat16, device=device)
    wd = torch.full((N, K + 8), float("nan"), dtype=torch.bfloat16, device=device)
    xd[:, :K], wd[:, :K] = x.to(device), w.to(device)
    yd = torch.full((M, N + ypad), 7.0, dtype=torch.bfloat16, device=device)
    nbytes = G.workspace_bytes(M, N, K)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=device) if nbytes else None
    G.gemm_into(xd[:, :K], wd[:, :K], yd[:, :N], NONE, ws)
    y = yd.cpu()
    assert torch.equal(y[:, N:], torch.full((M, ypad), 7.0, dtype=torch.bfloat16))
    assert_parity(y[:, :N].contiguous(), R.linear_bf16(x, w), "strided")
    assert_fp32_rounding(y[:, :N].contiguous(), x, w, "strided")


@pytest.mark.parametrize("K", [520, 4096])
def test_special_values_stay_in_their_rows_and_columns(device, K):
    """An infinite x element, a NaN x element and a NaN weight row reach only
    their own output row or column (K = 520 ends in a partial stage)."""
    M, N = 101, 70
    say("special values", K)
    x, w = R.randn_bf16((M, K), 9700), R.randn_bf16((N, K), 9701, 0.02)
    clean = krk(x, w)
    x[100, K - 1], x[33, 0], w[69, 5] = float("inf"), float("nan"), float("nan")
    y = krk(x, w)
    assert y[:, 69].isnan().all() and y[33].isnan().all()
    assert y[100, :69].isinf().all()
    keep = torch.ones(M, dtype=torch.bool)
    keep[[33, 100]] = False
    assert torch.equal(y[keep][:, :69], clean[keep][:, :69])


@pytest.mark.parametrize("M,N,K", [(100, 520, 2560), (64, 16400, 520), (72, 2560, 4096), (130, 70, 1032)])
def test_normed_rows_beyond_64(device, M, N, K):
    say("normed", M, N, K)
    x, d = R.randn_bf16((M, K), 9800), R.randn_bf16((M, K), 9801)
    wn = R.randn_bf16((K,), 9802, 0.1) + 1.0
    w = R.randn_bf16((N, K), 9803, 0.02)
    xout = torch.empty((M, K), dtype=torch.bfloat16, device=device)
    y = G.SkinnyMatmul(M, N, K, device)(x.to(device), w.to(device), norm=(d.to(device), wn.to(device), xout, 1e-6))
    ref_xout, ref = R.normed_linear_bf16(x, d, wn, 1e-6, w)
    assert torch.equal(xout.cpu(), ref_xout)
    assert_parity(y.cpu(), ref, "normed")


@pytest.mark.parametrize("M", [96, 128, 130, 192, 200])
def test_forms_of_the_call_agree(device, M):
    """A split plan (o_proj): repeated calls, the allocation-free call and the
    plan given as a configuration are bit-identical, the block counters end at
    zero (130 and 192 rows: the last launch, of 2 and 64, counts its splits
    there, in a workspace that the tile kernel's sums have passed through), and
    a configuration other than the plan runs in launches of 64."""
    N, K = 2560, 4096
    say("forms", M)
    x, w = R.randn_bf16((M, K), 9900).to(device), R.randn_bf16((N, K), 9901, 0.02).to(device)
    plan = G.plan(M, N, K)
    assert plan["splits"] > 1
    mm = G.SkinnyMatmul(M, N, K, device)
    first = mm(x, w).clone()
    blocks = -(-N // plan["channels"])
    for _ in range(3):
        assert torch.equal(mm(x, w), first)
    assert int(mm.workspace[:4 * blocks].max()) == 0
    assert torch.equal(G.SkinnyMatmul(M, N, K, device, config=plan)(x, w), first)
    assert torch.equal(G.gemm_noalloc(x, w, torch.full_like(first, float("nan"))), first)
    if M % 128 and M % 128 <= 64:  # the last launch: the 64-row plan
        tail = torch.cat([x[M // 128 * 128:], x[:64 - M % 128]])
        assert torch.equal(G.SkinnyMatmul(64, N, K, device)(tail, w)[:M % 128], first[M // 128 * 128:])
    other = G.SkinnyMatmul(M, N, K, device, config=dict(plan, splits=1))(x, w)
    assert_parity(other.cpu(), first.cpu(), "launches of 64 against the tile kernel")
