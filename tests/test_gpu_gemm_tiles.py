"""Every weight format of the dequant GEMM on each of its output tiles, with and without K splits, on the MI355X.

The tile and the splits that a shape takes are asked of the library and asserted, so a case cannot drift to another
kernel instance unnoticed. Shapes leave partial row tiles, partial column tiles, odd widths and a partial last k-stage.
The decoded weights are known exactly (int4: the fp32 ``(q - z) * s`` rounded to the activation type; int8, E4M3, E2M1
times the block scale: exact), so a result differs from the float64 product by the fp32 accumulation,
``(k/32 + 24) * 2**-24 * sum|x w|`` (one rounded 32-term MFMA partial per step, two roundings allowed per step, at most
16 ordered split sums), at most four fp32 roundings of the scaled sum and bias, and the output rounding.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from tests.conftest import print_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 0.0}

# m, n, k (brought to the format's multiple) and the tile and splits that it has to take
TILES = [
    (1000, 8201, 1312, (256, 256, 1)),
    (520, 8195, 1312, (128, 256, 1)),
    (300, 8197, 1312, (128, 128, 1)),
    (260, 4102, 8224, (128, 256, 5)),
    (130, 301, 1312, (128, 128, 5)),
    (1000, 8201, 128, (256, 256, 1)),  # fewer stages than the ring holds
    (400, 8201, 256, (128, 256, 1)),
]
INT4 = {  # asymmetric, parameter type, group
    "sym g128": (False, torch.float32, 128), "sym g64": (False, torch.float32, 64), "sym g32": (False, torch.float32, 32),
    "asym bf16 g128": (True, torch.bfloat16, 128), "asym bf16 g32": (True, torch.bfloat16, 32),
    "asym fp32 g128": (True, torch.float32, 128), "asym fp32 g64": (True, torch.float32, 64),
    "asym fp32 g32": (True, torch.float32, 32),  # two parameter copies a wave on the 256-column tiles
}


def _plan(weight, m, n, k):
    from scratch_llm_amd import _lib

    out = [ctypes.c_int() for _ in range(3)]
    _lib.check(_lib.load().sqx_gemm_plan(_lib.GEMM_WEIGHTS.index(weight), m, n, k, *map(ctypes.byref, out)), "plan")
    return tuple(v.value for v in out)


def _check(y, ref, mag, k, what):
    assert bool(torch.isfinite(y).all()), f"{what}: non-finite output"
    bound = (k / 32 + 24) * 2.0**-24 * mag + (2.0**-21 + ULP[y.dtype]) * ref.abs() + 2.0**-25
    worst = float(((y.double() - ref).abs() / bound).max())
    assert worst <= 1.0, f"{what}: off by {worst:.2f}x the bound"


def _workspaces(run, m, n, tile):
    """The result with a workspace for the splits' partials, without one, and with one that is too small."""
    nb = tile[2] * m * n * 4 if tile[2] > 1 else 0
    ws = torch.empty(max(nb // 4, 4), dtype=torch.float32, device=DEV)
    return [run(ws.data_ptr(), nb), run(None, 0), run(ws.data_ptr(), max(nb - 4, 0))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("kind", list(INT4))
@pytest.mark.parametrize("m,n,k,tile", TILES)
def test_int4_tiles(m, n, k, tile, kind, dtype):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import int4_group as i4

    asym, pdt, group = INT4[kind]
    k = -(-k // group) * group
    print_case("int4 tiles", kind, f"m={m}", f"n={n}", f"k={k}", f"dtype={dtype}")
    assert _plan("int4", m, n, k) == tile
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    bias = torch.randn(n, device=DEV, generator=g).to(dtype)
    q = torch.randint(0 if asym else -8, 16 if asym else 8, (n, k), device=DEV, generator=g).to(torch.uint8 if asym else torch.int8)
    s = (torch.rand(n, k // group, device=DEV, generator=g) * 0.01 + 1e-3).to(pdt)
    z = (torch.rand(n, k // group, device=DEV, generator=g) * 15).round().to(pdt) if asym else None
    tw = i4.tile_int4(q, s, z, group)
    w = q.float().view(n, -1, group)
    w = ((w if z is None else w - z.float()[:, :, None]) * s.float()[:, :, None]).view(n, k).to(dtype).double()
    ref = x.double() @ w.t() + bias.double()
    mag = x.double().abs() @ w.abs().t() + bias.double().abs()
    lib = _lib.load()

    def run(ws, nb):
        y = torch.empty(m, n, dtype=dtype, device=DEV)
        _lib.check(lib.sqx_int4_gemm(tw.wt.data_ptr(), tw.st.data_ptr(), _lib.ptr(tw.zt), _lib.sqx_dtype(tw.st.dtype),
                                     x.data_ptr(), _lib.sqx_dtype(dtype), y.data_ptr(), bias.data_ptr(), m, n, k, group, ws,
                                     nb, _lib.stream_ptr(x.device)), "int4 tiles")
        return y

    for y in _workspaces(run, m, n, tile):
        _check(y, ref, mag, k, f"int4 {kind}")


@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.bfloat16, torch.float32)],
                         ids=["bf16", "fp16", "bf16 to fp32"])
@pytest.mark.parametrize("fmt", ["mxfp4", "nvfp4"])
@pytest.mark.parametrize("m,n,k,tile", TILES)
def test_fp4_tiles(m, n, k, tile, fmt, dtype, out):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import nvfp4_mxfp4 as f4

    print_case("fp4 tiles", fmt, f"m={m}", f"n={n}", f"k={k}", f"dtype={dtype}", f"out={out}")
    assert _plan(fmt, m, n, k) == tile
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    bias = torch.randn(n, device=DEV, generator=g).to(dtype) if out == dtype else None
    wf = torch.randn(n, k, device=DEV, generator=g) * 0.02
    q = f4.mxfp4_quantize(wf) if fmt == "mxfp4" else f4.nvfp4_quantize(wf)
    tw = f4.tile_fp4(q)
    w = (f4.mxfp4_dequantize(q) if fmt == "mxfp4" else f4.nvfp4_dequantize(q)).double()
    ref, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
    if bias is not None:
        ref, mag = ref + bias.double(), mag + bias.double().abs()
    lib = _lib.load()

    def run(ws, nb):
        y = torch.empty(m, n, dtype=out, device=DEV)
        _lib.check(lib.sqx_fp4_gemm(tw.wt.data_ptr(), tw.st.data_ptr(), tw.fmt, _lib.ptr(tw.s_global), x.data_ptr(),
                                    _lib.sqx_dtype(dtype), y.data_ptr(), _lib.sqx_dtype(out), _lib.ptr(bias), m, n, k, ws, nb,
                                    _lib.stream_ptr(x.device)), "fp4 tiles")
        return y

    for y in _workspaces(run, m, n, tile):
        _check(y, ref, mag, k, fmt)  # (NVFP4's reference weights carry two fp32 roundings: 2**-23 of mag, in its bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m,n,k,tile", TILES)
def test_int8_tiles(m, n, k, tile, dtype):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import int8

    k -= 8  # rows of 8-column multiples
    print_case("int8 tiles", f"m={m}", f"n={n}", f"k={k}", f"dtype={dtype}")
    assert _plan("int8", m, n, k) == tile
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    bias = torch.randn(n, device=DEV, generator=g).to(dtype)
    q = torch.randint(-128, 128, (n, k), device=DEV, generator=g).to(torch.int8)
    s = torch.rand(n, 1, device=DEV, generator=g) * 1e-3 + 1e-4
    tw, w = int8.tile_int8(q, s), q.double() * s.double()
    ref = x.double() @ w.t() + bias.double()
    mag = x.double().abs() @ w.abs().t() + bias.double().abs()
    lib = _lib.load()

    def run(ws, nb):
        y = torch.empty(m, n, dtype=dtype, device=DEV)
        _lib.check(lib.sqx_int8_gemm(tw.wt.data_ptr(), tw.scale.data_ptr(), x.data_ptr(), _lib.sqx_dtype(dtype), y.data_ptr(),
                                     bias.data_ptr(), m, n, k, ws, nb, _lib.stream_ptr(x.device)), "int8 tiles")
        return y

    for y in _workspaces(run, m, n, tile):
        _check(y, ref, mag, k, "int8")


@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("m,n,k,tile", TILES)
def test_fp8_tiles(m, n, k, tile, out):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import fp8_weights as f8

    k -= 8
    print_case("fp8 tiles", f"m={m}", f"n={n}", f"k={k}", f"out={out}")
    assert _plan("fp8", m, n, k) == tile
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    bias = torch.randn(n, device=DEV, generator=g).to(torch.bfloat16) if out == torch.bfloat16 else None
    q, s = f8.quantize_per_channel(torch.randn(n, k, device=DEV, generator=g) * 0.02)
    xq, xs = f8.quantize_per_channel(x)  # the linear's own quantization of its rows
    tw = f8.tile_fp8(q, s)
    xd, wd = xq.double() * xs.double().reshape(-1, 1), q.double() * s.double().reshape(-1, 1)
    ref, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    if bias is not None:
        ref, mag = ref + bias.double(), mag + bias.double().abs()
    lib = _lib.load()
    nb_all = int(lib.sqx_fp8_linear_workspace_bytes(m, n, k))
    nb_rows = nb_all - tile[2] * m * n * 4 if tile[2] > 1 else nb_all  # without the partials: one pass per tile

    for nb in (nb_all, nb_rows, max(nb_all - 4, nb_rows)):
        ws = torch.empty(nb_all, dtype=torch.uint8, device=DEV)
        y = torch.empty(m, n, dtype=out, device=DEV)
        _lib.check(lib.sqx_fp8_linear(tw.wt.data_ptr(), tw.scale.data_ptr(), x.data_ptr(), _lib.DTYPE_BF16, y.data_ptr(),
                                      _lib.sqx_dtype(out), _lib.ptr(bias), m, n, k, 0, ws.data_ptr(), nb,
                                      _lib.stream_ptr(x.device)), "fp8 tiles")
        _check(y, ref, mag, k, "fp8")


# the tile with K splits where only some formats take it
@pytest.mark.parametrize("weight,m,n,k,tile", [("int4", 300, 12300, 4128, (256, 256, 2)), ("nvfp4", 500, 4100, 8224, (256, 256, 7))])
def test_large_tile_splits(weight, m, n, k, tile):
    if weight == "int4":
        test_int4_tiles(m, n, k, tile, "asym fp32 g32", torch.bfloat16)
    else:
        test_fp4_tiles(m, n, k, tile, weight, torch.bfloat16, torch.bfloat16)
