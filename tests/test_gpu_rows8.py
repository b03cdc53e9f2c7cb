"""The row-tiled decode kernels on FP4 and int8 weights (sqx_fp4_skinny, sqx_int8_skinny) at 2..64 rows.

The decoded weights are the values themselves (FP4: e2m1 times its block scale; int8: the code, with the row
scale on the fp32 sum), so a result differs from the float64 product by the fp32 accumulation,
``(k/32 + 8 + S) * 2**-24 * sum|x w|`` (one rounded 32-term MFMA partial per step, S ordered split sums), at most
three fp32 roundings of the scaled sum and bias, and the output rounding.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.conftest import print_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(y, ref, mag, k, what):
    ulp = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[y.dtype]
    yv = y.double().cpu().numpy()
    assert np.isfinite(yv).all(), f"{what}: non-finite output"
    bound = (k / 32 + 24) * 2.0**-24 * mag + (ulp + 2.0**-22) * np.abs(ref) + 2.0**-25
    worst = float((np.abs(yv - ref) / bound).max())
    assert worst <= 1.0, f"{what}: off by {worst:.2f}x the bound"


# partial row tiles, a partial last k-block, fewer k-blocks than waves, every dispatch range of rows
LINEAR = [(2, 16, 32), (3, 1000, 96), (8, 40, 224), (9, 6150, 512), (16, 4096, 1056), (17, 10240, 160), (32, 16400, 320),
          (33, 520, 4096), (63, 1024, 8224), (24, 6400, 8192),
          # the row-tiled kernels' side of the choice, for either format
          (6, 28700, 1568), (9, 6150, 2592), (12, 4096, 9248), (4, 10250, 12320), (18, 14400, 544), (40, 28700, 1056),
          (13, 18000, 2080), (2, 30000, 2592), (36, 5200, 1568), (5, 65552, 96),
          # 257..1023 tiles in one piece and in splits
          (12, 8200, 8224), (10, 4120, 6176), (7, 10250, 8224), (31, 6200, 8224), (33, 9000, 8096), (36, 5120, 4960),
          (14, 6160, 16416), (5, 7000, 16288), (16, 4120, 16288)]


@pytest.mark.parametrize("fmt", ["mx", "nv"])
@pytest.mark.parametrize("m,n,k", LINEAR)
def test_fp4_rows(m, n, k, fmt):
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    print_case("fp4 rows", f"m={m}", f"n={n}", f"k={k}", fmt)
    g = torch.Generator().manual_seed(m * n + k)
    dtype = torch.float16 if m % 3 == 0 else torch.bfloat16
    x = torch.randn(m, k, generator=g).to(dtype)
    bias = torch.randn(n, generator=g).to(dtype) if m % 2 else None
    w = torch.randn(n, k, generator=g).to(DEV) * 0.02
    q = f4.mxfp4_quantize(w) if fmt == "mx" else f4.nvfp4_quantize(w)
    wd = (f4.mxfp4_dequantize(q) if fmt == "mx" else f4.nvfp4_dequantize(q)).double().cpu().numpy()
    y = f4.fp4_linear_tiled(x.to(DEV), f4.tile_fp4(q), None if bias is None else bias.to(DEV))
    xd = x.double().numpy()
    ref, mag = xd @ wd.T, np.abs(xd) @ np.abs(wd).T
    if bias is not None:
        b = bias.double().numpy()
        ref, mag = ref + b, mag + np.abs(b)
    _check(y, ref, mag, k, f"{fmt} {m}x{n}x{k}")


@pytest.mark.parametrize("variant,tiles,waves,splits", [(0, 2, 8, 1), (0, 4, 4, 2), (0, 4, 8, 3), (1, 1, 8, 2), (1, 2, 8, 4),
                                                        (1, 4, 4, 1), (1, 2, 4, 8)])
@pytest.mark.parametrize("m", [7, 16, 40])
def test_fp4_launch_shapes(m, variant, tiles, waves, splits):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    n, k = 1030, 1440
    print_case("fp4 launch shape", f"m={m}", f"variant={variant}", f"tiles={tiles}", f"waves={waves}", f"splits={splits}")
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    q = f4.nvfp4_quantize(torch.randn(n, k, generator=g).to(DEV) * 0.02)
    tw, wd = f4.tile_fp4(q), f4.nvfp4_dequantize(q).double().cpu().numpy()
    lib, xg = _lib.load(), x.to(DEV)
    y = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(max(int(lib.sqx_fp4_skinny_workspace_bytes(m, n, k, splits)) // 4, 1), device=DEV)
    _lib.check(lib.sqx_fp4_skinny(tw.wt.data_ptr(), tw.st.data_ptr(), tw.fmt, tw.s_global.data_ptr(), xg.data_ptr(),
                                  _lib.DTYPE_BF16, y.data_ptr(), None, m, n, k, variant, tiles, waves, splits, ws.data_ptr(),
                                  ws.numel() * 4, _lib.stream_ptr(xg.device)), "sqx_fp4_skinny")
    xd = x.double().numpy()
    _check(y, xd @ wd.T, np.abs(xd) @ np.abs(wd).T, k, "fp4 shape")


# the GEMV's side of the choice, then the row-tiled kernel's (every range of weight rows that it takes)
@pytest.mark.parametrize("m,n,k", [(2, 16, 8), (5, 1000, 72), (16, 4096, 4096), (17, 40, 200), (33, 6160, 520), (64, 16400, 136),
                                   (20, 1024, 8200), (64, 4096, 1032),
                                   (16, 1030, 10248), (5, 5200, 8200), (64, 4096, 3080), (36, 3000, 8200), (12, 6160, 2056),
                                   (8, 10248, 2056), (48, 14330, 1032), (20, 18440, 2568), (4, 28680, 2568), (64, 32776, 72),
                                   # 257..383 tiles in one piece, and past them
                                   (16, 5120, 4104), (33, 4120, 2568), (64, 6120, 12280), (12, 6130, 12296),
                                   # small weights past 64 rows: the last rows of the GEMV, the GEMM's first
                                   (65, 512, 512), (80, 3070, 1536), (104, 1024, 1024), (105, 1024, 1024)])
def test_int8_rows(m, n, k):
    from scratch_llm_amd.quant import int8

    print_case("int8 rows", f"m={m}", f"n={n}", f"k={k}")
    g = torch.Generator().manual_seed(m + n + k)
    dtype = torch.float16 if m % 2 else torch.bfloat16
    q = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    s = torch.rand(n, 1, generator=g) * 1e-3 + 1e-4
    x = torch.randn(m, k, generator=g).to(dtype)
    bias = torch.randn(n, generator=g).to(dtype)
    y = int8.int8_linear_tiled(x.to(DEV), int8.tile_int8(q.to(DEV), s.to(DEV)), bias.to(DEV))
    xd, wd, b = x.double().numpy(), q.double().numpy() * s.double().numpy(), bias.double().numpy()
    # the GEMV (short shapes) sums codes offset by 128 and takes 128 * sum(x) off again
    off = 128.0 * s.double().numpy().T * np.abs(xd).sum(1, keepdims=True)
    _check(y, xd @ wd.T + b, np.abs(xd) @ np.abs(wd).T + np.abs(b) + 2 * off, k, f"int8 {m}x{n}x{k}")


@pytest.mark.parametrize("m,n,k", [(2, 40, 16), (8, 10240, 176), (20, 6160, 528), (33, 520, 4112), (63, 16400, 48)])
def test_nvfp4_rows_of_16_columns(m, n, k):
    """NVFP4 rows that end in half a 32-column chunk, on the kernels of 2..63 rows."""
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    print_case("nvfp4 k % 32 == 16", f"m={m}", f"n={n}", f"k={k}")
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    q = f4.nvfp4_quantize(torch.randn(n, k, generator=g).to(DEV) * 0.02)
    wd = f4.nvfp4_dequantize(q).double().cpu().numpy()
    y = f4.fp4_linear_tiled(x.to(DEV), f4.tile_fp4(q))
    xd = x.double().numpy()
    _check(y, xd @ wd.T, np.abs(xd) @ np.abs(wd).T, k, f"nvfp4 {m}x{n}x{k}")


@pytest.mark.parametrize("tiles,waves,splits", [(2, 8, 1), (4, 4, 2), (2, 1, 3), (4, 8, 4), (2, 4, 16)])
@pytest.mark.parametrize("m", [1, 8, 33, 64])
def test_int8_launch_shapes(m, tiles, waves, splits):
    """The row-tiled kernel with an explicit launch shape, partial row tiles and a partial last k-block among them."""
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import int8

    n, k = 1030, 1432
    print_case("int8 launch shape", f"m={m}", f"tiles={tiles}", f"waves={waves}", f"splits={splits}")
    g = torch.Generator().manual_seed(m)
    q = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int8)
    s = torch.rand(n, 1, generator=g) * 1e-3 + 1e-4
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    tw, lib, xg = int8.tile_int8(q.to(DEV), s.to(DEV)), _lib.load(), x.to(DEV)
    y = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    ws = torch.empty(max(int(lib.sqx_int8_skinny_workspace_bytes(m, n, k, splits)) // 4, 1), device=DEV)
    _lib.check(lib.sqx_int8_skinny(tw.wt.data_ptr(), tw.scale.data_ptr(), xg.data_ptr(), _lib.DTYPE_BF16, y.data_ptr(), None,
                                   m, n, k, tiles, waves, splits, ws.data_ptr(), ws.numel() * 4, _lib.stream_ptr(xg.device)),
               "sqx_int8_skinny")
    xd, wd = x.double().numpy(), q.double().numpy() * s.double().numpy()
    _check(y, xd @ wd.T, np.abs(xd) @ np.abs(wd).T, k, "int8 shape")


def test_few_rows_ask_for_no_workspace():
    """The GEMV's sizes need none, and a size is asked for once."""
    from scratch_llm_amd.quant import int8

    q = torch.randint(-128, 128, (512, 512), dtype=torch.int8, device=DEV)
    tw, x = int8.tile_int8(q, torch.ones(512, 1, device=DEV)), torch.randn(2, 512, device=DEV, dtype=torch.bfloat16)
    int8.int8_linear_tiled(x, tw)
    before = int8._rows_workspace.cache_info()
    int8.int8_linear_tiled(x, tw)
    after = int8._rows_workspace.cache_info()
    assert (after.hits, after.misses) == (before.hits + 1, before.misses) and int8._rows_workspace(2, 512, 512) == -1
