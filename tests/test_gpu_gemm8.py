"""The dequant GEMM on 8-bit weights (sqx_int8_gemm and sqx_fp8_linear from 65 rows) and the split and ring edges of its
pipeline, at shapes that mostly take its 128 x 128 tile, on the MI355X (test_gpu_gemm_tiles.py has every tile).

int8 and E4M3 codes are exact in the activation dtype, so int8 differs from the float64 product only by the
fp32 accumulation, ``(k/32 + 8) * 2**-24 * sum|x w|`` (one rounded 32-term MFMA partial per step, two
roundings allowed per step), three fp32 roundings of the scaled sum and bias (2**-22 |y|), and the
output rounding; FP8 is held to the reference's own derived bound for fp8_linear.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import fp8_ref as F8
from tests.conftest import print_case

pytestmark = pytest.mark.gpu
DEV = "cuda"

# m, n, k: one row past a tile, partial column tiles, odd n, k of one stage, of fewer stages than the ring
# and with a partial last stage, enough splits for an uneven last one
SHAPES = [(65, 40, 64), (128, 129, 72), (129, 257, 200), (200, 1024, 1096), (257, 515, 328), (300, 4096, 520),
          (513, 4100, 384), (1000, 1024, 4096)]


def _check(y, ref, mag, k, dtype, what):
    yv = y.double().cpu().numpy()
    assert np.isfinite(yv).all(), f"{what}: non-finite output"
    ulp = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[dtype] * np.abs(ref) + 2.0**-25
    bound = (k / 32 + 8) * 2.0**-24 * mag + 2.0**-22 * np.abs(ref) + ulp
    worst = float((np.abs(yv - ref) / bound).max())
    assert worst <= 1.0, f"{what}: off by {worst:.2f}x the bound"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_int8_gemm(m, n, k, dtype):
    from scratch_llm_amd.quant import int8

    print_case("int8 gemm", f"m={m}", f"n={n}", f"k={k}", f"dtype={dtype}")
    g = torch.Generator().manual_seed(m + n + k)
    q = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    s = torch.rand(n, 1, generator=g) * 1e-3 + 1e-4
    x = torch.randn(m, k, generator=g).to(dtype)
    bias = torch.randn(n, generator=g).to(dtype) if m % 2 else None
    tw = int8.tile_int8(q.to(DEV), s.to(DEV))
    y = int8.int8_linear_tiled(x.to(DEV), tw, None if bias is None else bias.to(DEV))
    assert y.shape == (m, n) and y.dtype == dtype
    xd, wd = x.double().numpy(), q.double().numpy() * s.double().numpy()
    ref, mag = xd @ wd.T, np.abs(xd) @ np.abs(wd).T
    if bias is not None:
        b = bias.double().numpy()
        ref, mag = ref + b, mag + np.abs(b)
    _check(y, ref, mag, k, dtype, f"int8 {m}x{n}x{k}")
    # a second call gives the same bits
    assert torch.equal(y, int8.int8_linear_tiled(x.to(DEV), tw, None if bias is None else bias.to(DEV)))


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", SHAPES + [(70, 1024, 1024), (71, 1024, 1024)])  # the GEMV's last rows, the GEMM's first
def test_fp8_gemm(m, n, k, out_dtype):
    from scratch_llm_amd.quant import fp8_weights as f8

    print_case("fp8 gemm", f"m={m}", f"n={n}", f"k={k}", f"out={out_dtype}")
    g = torch.Generator().manual_seed(m + 3 * n + k)
    codes, scale = F8.quantize_rows(torch.randn(n, k, generator=g).numpy() * 0.02)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    bias = torch.randn(n, generator=g).to(torch.bfloat16) if m % 2 and out_dtype == torch.bfloat16 else None
    tw = f8.tile_fp8(torch.from_numpy(codes).to(DEV).view(torch.float8_e4m3fn), torch.from_numpy(scale).to(DEV))
    y = f8.fp8_linear_tiled(x.to(DEV), tw, None if bias is None else bias.to(DEV), out_dtype=out_dtype)
    assert y.shape == (m, n) and y.dtype == out_dtype
    b = None if bias is None else bias.float().numpy()
    ref = F8.fp8_linear_reference(x.float().numpy(), codes, scale, b)
    xc, xs = F8.quantize_rows(x.float().numpy())
    mag = np.abs(F8.dequantize(xc, xs).astype(np.float64)) @ np.abs(F8.dequantize(codes, scale).astype(np.float64)).T
    eps = 2.0**-7 if out_dtype == torch.bfloat16 else 2.0**-23
    bound = np.abs(ref) * eps / 2 + (mag + (0 if b is None else np.abs(b))) * math.sqrt(k) * 2.0**-23 + 2.0**-22 * np.abs(ref)
    worst = float((np.abs(y.double().cpu().numpy() - ref) / bound).max())
    assert worst <= 1.0, f"{worst:.3f}x the bound"


@pytest.mark.parametrize("k", [128, 256, 384, 640, 1024])
@pytest.mark.parametrize("m,n", [(65, 130), (129, 300), (300, 4096), (520, 8200)])
def test_gemm_ring_edges_4bit(m, n, k):
    """4-bit weights at few stages, mostly on 128-row output tiles: each output equals the same weights' product
    in float64 within the accumulation and output rounding (int4: of the bf16-rounded weights)."""
    from scratch_llm_amd.quant import int4_group as i4
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    print_case("gemm ring edges", f"m={m}", f"n={n}", f"k={k}")
    g = torch.Generator().manual_seed(m * k + n)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    xd = x.double().numpy()
    q = torch.randint(-8, 8, (n, k), generator=g, dtype=torch.int8)
    s = torch.rand(n, k // 128, generator=g) * 0.01 + 1e-3
    w = (q.view(n, -1, 128).float() * s[:, :, None]).view(n, k).to(torch.bfloat16).double().numpy()
    y = i4.int4_linear_tiled(x.to(DEV), i4.tile_int4(q.to(DEV), s.to(DEV)))
    _check(y, xd @ w.T, np.abs(xd) @ np.abs(w).T, k, torch.bfloat16, "int4")
    packed = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8)
    e8 = torch.randint(118, 123, (n, k // 32), generator=g, dtype=torch.uint8)
    w = f4.dequantize_mxfp4(packed.to(DEV), e8.to(DEV)).double().cpu().numpy()
    y = f4.fp4_linear_tiled(x.to(DEV), f4.tile_mxfp4_packed(packed.to(DEV), e8.to(DEV)))
    _check(y, xd @ w.T, np.abs(xd) @ np.abs(w).T, k, torch.bfloat16, "mxfp4")


# k % 128 of 32, 64, 96: the padded last 128 columns leave one or two of the k-stages past k
@pytest.mark.parametrize("k", [1312, 1344, 1376])
@pytest.mark.parametrize("m,n", [(300, 8200), (1000, 8200)])  # 128 x 128 and 256 x 256 output tiles
@pytest.mark.parametrize("fmt", ["int4", "mxfp4"])
def test_gemm_rows_stay_apart(m, n, k, fmt):
    """Inf and NaN in the first columns of some rows leave every other row's bits as they were."""
    from scratch_llm_amd.quant import int4_group as i4
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    print_case("gemm rows apart", fmt, f"m={m}", f"n={n}", f"k={k}")
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    if fmt == "int4":
        q = torch.randint(-8, 8, (n, k), generator=g, dtype=torch.int8).to(DEV)
        tw = i4.tile_int4(q, torch.rand(n, k // 32, generator=g).to(DEV) + 0.5, None, 32)
        run = i4.int4_linear_tiled
    else:
        packed = torch.randint(0, 256, (n, k // 2), generator=g, dtype=torch.uint8).to(DEV)
        e8 = torch.randint(118, 123, (n, k // 32), generator=g, dtype=torch.uint8).to(DEV)
        tw, run = f4.tile_mxfp4_packed(packed, e8), f4.fp4_linear_tiled
    y = run(x, tw)
    assert bool(torch.isfinite(y).all())
    bad = torch.tensor([1, 77, m - 1])
    x[bad, :64:7] = float("inf")
    x[bad, 3:64:9] = float("nan")
    z = run(x, tw)
    keep = torch.ones(m, dtype=torch.bool)
    keep[bad] = False
    assert torch.equal(z[keep.to(DEV)], y[keep.to(DEV)])
    assert bool(torch.isnan(z[bad.to(DEV)]).all())
