"""GPU parity of the MatMulNBits kernel for small batches, 8-bit weights and fp32 prompts
against the oracle's 64-bit product, at the edges of its tiles.

4-bit weights with fp16 or bf16 activations are rounded once to that type, as the
reference product here rounds them; in the other forms the codes enter the matrix cores
exactly. Every product is exact in fp32 either way, so the bound is that of fp32 accumulation, 2^-24 * (number of additions of one output, at
most 32 per chunk and piece, one per chunk and one per wave) * sum |a * w|, plus the
rounding of the output type."""

from __future__ import annotations

import numpy as np
import pytest
from test_gpu_ops import _mnb_inputs, dev, host

pytestmark = pytest.mark.gpu


def _run(ortmi, oracle, dt, M, K, N, bits, block, asym, edit=None):
    import torch

    tdt = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dt]
    rng = np.random.default_rng(M * 31 + K + N + bits)
    A, B, s, zp = _mnb_inputs(rng, M, N, K, block, bits=bits, asym=asym)
    if bits == 8:
        s = s / 16
    dA, ds = dev(A, tdt), dev(s, tdt)
    if edit is not None:
        edit(dA)
    got = host(ortmi.matmul_nbits(dA, dev(B), ds, dev(zp) if zp is not None else None, K=K, N=N,
                                  bits=bits, block_size=block)).astype(np.float64)
    A, s = dA.float().cpu().numpy(), ds.float().cpu().numpy()
    W = oracle.mnb_dequant(B, s, zp, N, K, bits, block).astype(np.float64)
    if bits == 4 and dt != "f32":
        W = torch.from_numpy(W.astype(np.float32)).to(tdt).double().numpy()
    return got, A.astype(np.float64), W


@pytest.mark.parametrize("dt", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,K,N,bits,block,asym", [
    (2, 256, 16, 4, 32, True),      # fewer steps than waves, one column tile
    (8, 4096, 1000, 4, 32, False),  # ragged N
    (16, 1176, 515, 4, 32, True),   # K ends inside a step and a block
    (17, 1536, 300, 4, 64, True),   # one row past a tile
    (33, 2048, 4100, 4, 128, True),
    (64, 896, 17000, 4, 32, True),  # four column tiles per workgroup
    (1, 3072, 1003, 8, 32, True),
    (1, 11072, 64, 8, 128, False),
    (5, 360, 130, 8, 64, True),
    (130, 712, 4200, 8, 32, True),
    (65, 1536, 130, 4, 32, True),   # past 64 rows, too few outputs for the prefill GEMM
    (200, 896, 515, 4, 64, False),
    (512, 360, 1030, 4, 32, True),
    (512, 360, 1000, 4, 32, True),  # 256 tiles of 32 x 64: a CU to each
    (33, 896, 8192, 4, 128, False),
    (33, 896, 8193, 4, 128, False), # and one column more, on the prefill GEMM
])
def test_mnb_blk(ortmi, oracle, dt, M, K, N, bits, block, asym):
    got, A, W = _run(ortmi, oracle, dt, M, K, N, bits, block, asym)
    exact = A @ W.T
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 2.0 ** -24}[dt]
    adds = 3 * 32 + (K + 31) // 32 + 8
    bound = ulp * np.abs(exact) + 2.0 ** -24 * adds * (np.abs(A) @ np.abs(W).T) + 1e-7
    excess = np.abs(got - exact) - bound
    assert excess.max() <= 0, f"max excess {excess.max():.3e}"


def test_mnb_blk_fp32_carries_24_bits(ortmi, oracle):
    """fp32 activations keep all mantissa bits: the error stays at fp32 level, far under
    what two bf16 pieces (2^-16 relative) would leave."""
    got, A, W = _run(ortmi, oracle, "f32", 40, 1024, 256, 4, 32, True)
    exact = A @ W.T
    assert np.linalg.norm(got - exact) / np.linalg.norm(exact) < 1e-6


def test_mnb_blk_fp32_extremes(ortmi, oracle):
    """Infinities and NaN stay in their rows, and activations near the largest fp32
    give what the scaled weights allow (no overflow of the unscaled sums)."""
    def edit(a):
        a[1, 3] = float("inf")
        a[2, 5] = float("nan")
        a[4] *= 1e37

    got, A, W = _run(ortmi, oracle, "f32", 20, 512, 96, 4, 32, True, edit)
    A[1:3] = np.where(np.isfinite(A[1:3]), A[1:3], 0)
    exact = A @ W.T
    rows = [i for i in range(20) if i not in (1, 2)]
    top = np.abs(exact[rows]).max(axis=1, keepdims=True)
    assert (np.abs(got[rows] - exact[rows]) <= 1e-5 * top).all()
    assert np.isnan(got[2]).all()
    w = W[:, 3]
    assert (got[1][w > 0] == np.inf).all() and (got[1][w < 0] == -np.inf).all()


@pytest.mark.parametrize("dt,K,N,block,asym", [
    ("bf16", 11008, 515, 32, True),
    ("bf16", 14336, 4096, 32, False),
    ("bf16", 10248, 9003, 128, True),   # more column tiles per workgroup, K inside a block
    ("f16", 16416, 1030, 32, True),
    ("f16", 20488, 9003, 64, False),
])
def test_mnb_blk_one_row_keeps_weights(ortmi, oracle, dt, K, N, block, asym):
    """One row of 4-bit weights past the K of the GEMV rounds no weight: nearly every output
    is the exact sum rounded once. An fp32 sum is off by about 2^-20 of the outputs' rms, so
    that less than one in a hundred lies near enough to a tie of the fp16 rounding (one in a
    thousand, bf16) to fall on its other side; weights rounded to the type would move one
    output in three. None is further off than one rounding and the bound of the sums."""
    import torch

    tdt = {"f16": torch.float16, "bf16": torch.bfloat16}[dt]
    rng = np.random.default_rng(K + N)
    A, B, s, zp = _mnb_inputs(rng, 1, N, K, block, asym=asym)
    dA, ds = dev(A, tdt), dev(s, tdt)
    got = host(ortmi.matmul_nbits(dA, dev(B), ds, dev(zp) if zp is not None else None, K=K, N=N,
                                  block_size=block))[0].astype(np.float64)
    A, s = dA.double().cpu().numpy()[0], ds.float().cpu().numpy()
    nb = -(-K // block)
    pick = np.arange(N) if N < 2000 else np.r_[np.arange(0, N, 17), N - 1]
    W = oracle.mnb_dequant(B[pick], s.reshape(N, nb)[pick].ravel(),
                           None if zp is None else zp.reshape(N, -1)[pick].ravel(), pick.size, K, 4,
                           block).astype(np.float64)
    exact, got = W @ A, got[pick]
    rounded = torch.from_numpy(exact).to(tdt).double().numpy()
    assert (got != rounded).mean() < 0.03, f"{(got != rounded).mean():.3f} rounded otherwise"
    ulp = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt]
    adds = 32 + (K + 31) // 32 + 8
    bound = ulp * np.abs(exact) + 2.0 ** -24 * adds * (np.abs(W) @ np.abs(A)) + 1e-7
    assert (np.abs(got - exact) <= bound).all()


@pytest.mark.parametrize("dt,M,N,bits", [
    ("bf16", 40, 96, 4), ("bf16", 600, 2048, 4), ("bf16", 3, 96, 8), ("f32", 20, 96, 4),
    ("f32", 20, 96, 8)])
def test_mnb_large_scales(ortmi, oracle, dt, M, N, bits):
    """Scales near the largest the type holds, activations that keep the sums finite: each
    form's weights (q - zp) * s are finite, and so are its products."""
    import torch

    K, tdt = 256, {"bf16": torch.bfloat16, "f32": torch.float32}[dt]
    rng = np.random.default_rng(M + bits)
    A, B, s, zp = _mnb_inputs(rng, M, N, K, 32, bits=bits)
    top = 2.0 ** (123 if bits == 4 else 119)  # * 15 or 255 < 2^127
    s = s / s.max() * top
    dA, ds = dev(A * 2.0 ** -20, tdt), dev(s, tdt)
    got = host(ortmi.matmul_nbits(dA, dev(B), ds, dev(zp), K=K, N=N, bits=bits, block_size=32))
    A, s = dA.double().cpu().numpy(), ds.float().cpu().numpy()
    W = oracle.mnb_dequant(B, s, zp, N, K, bits, 32).astype(np.float64)
    want, mag = A @ W.T, np.abs(A) @ np.abs(W).T
    assert np.isfinite(want).all() and np.isfinite(got).all()
    # Weights rounded to bf16 at 4 bits: one rounding of each product.
    u = 2.0 ** -8 if dt == "bf16" and bits == 4 else 2.0 ** -16
    assert (np.abs(got - want) <= u * mag + (2.0 ** -8 if dt == "bf16" else 0) * np.abs(want)).all()


@pytest.mark.parametrize("bits", [4, 8])
def test_mnb_blk_fp32_signalling_nan(ortmi, oracle, bits):
    """A NaN whose payload lies in the low 16 bits alone gives NaN rows, not infinities."""
    import torch

    def edit(a):
        words = a.view(torch.int32)
        words[3, 7] = 0x7F800001
        words[11, 200] = 0xFF80FFFF - (1 << 32)
        a[5, 9] = float("inf")

    with np.errstate(invalid="ignore"):
        got, A, W = _run(ortmi, oracle, "f32", 20, 512, 96, bits, 32, True, edit)
    assert np.isnan(A[3, 7]) and np.isnan(A[11, 200])
    rows = [i for i in range(20) if i not in (3, 5, 11)]
    assert np.isnan(got[[3, 11]]).all() and np.isfinite(got[rows]).all()
    assert np.isinf(got[5][W[:, 9] != 0]).all()
