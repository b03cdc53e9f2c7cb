"""The vectorised quantizers and tilers against the general ones, and the W8A8 product at its tile edges.

A tensor that starts one element past an aligned address takes the element-wise kernels, the same values at an
aligned address take the vectorised ones where the sizes allow: codes and scales have to agree bit for bit. The
int8 product is exact in int32, so its fp32 result is within three roundings (the conversion, the two scales'
product, the scaled sum) of the integer product in float64.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.conftest import print_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _shifted(t):
    """The same values, contiguous, one element past a 16-byte aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


def _hostile(rows, cols, dtype, seed):
    """Rows of normal values, then rows of zeros, signed zeros, denormals, huge and mixed magnitudes, code ties."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g)
    x[0] = 0.0
    x[1 % rows] = -0.0
    if rows > 8:
        x[2] *= 1e-40
        x[3] *= 3e38 if dtype != torch.float16 else 6e4
        x[4, ::3] *= 1e6
        x[5] = (torch.arange(cols) % 29 - 14) * 0.5  # halves: every rounding tie
        x[6, cols // 2] = float("inf")
        x[7, 0] = -3e38
        x[8] = 448.0 * (torch.arange(cols) % 2 * 2 - 1)
    return x.to(dtype).to(DEV)


def _same(a, b, what):
    for i, (u, v) in enumerate(zip(a, b)):
        u, v = u.detach().contiguous(), v.detach().contiguous()
        assert u.shape == v.shape and u.dtype == v.dtype, f"{what}[{i}]"
        if u.dtype == torch.float32:
            both_nan = torch.isnan(u) & torch.isnan(v)
            ok = (u.view(torch.int32) == v.view(torch.int32)) | both_nan
        else:
            ok = u.view(torch.uint8) == v.view(torch.uint8)
        assert bool(ok.all()), f"{what}[{i}]: {int((~ok).sum())} of {ok.numel()} differ"


def _kv(x):
    from scratch_llm_amd.quant import fp8_kv_per_head as kv

    r, c = x.shape
    h = 3 if r % 3 == 0 else 1
    x4 = x.view(1, h, r // h, c)
    s = kv.per_head_scale(x4)
    t = torch.full_like(s, 0.01)  # a static scale: most values saturate
    return s, kv.per_head_amax(x4), kv.quantize_per_head(x4, s), kv.quantize_per_head(x4, t)


def _ops():
    from scratch_llm_amd.quant import fp8_weights as f8, int4_group as i4, int8 as i8, nvfp4_mxfp4 as f4

    def fp4(q):
        return [q.codes, q.s_block] + ([q.s_global.reshape(1)] if hasattr(q, "s_global") else [])

    return {
        "int4": lambda x: i4.quantize_groupwise_int4(x, 128 if x.shape[1] % 128 == 0 else 8),
        "int8": lambda x: i8.quantize_symmetric(x, axis=0),
        "int8_affine": lambda x: i8.quantize_affine(x, axis=0),
        "fp8": lambda x: f8.quantize_per_channel(x),
        "mxfp4": lambda x: fp4(f4.mxfp4_quantize(x)),
        "mxfp4_64": lambda x: fp4(f4.mxfp4_quantize(x, 64)),
        "nvfp4": lambda x: fp4(f4.nvfp4_quantize(x)),
        "kv": _kv,
    }


# one chunk, a partial last chunk per wave, several chunks a thread, the register kernels' largest row and one above it
SHAPES = [(1, 8), (2, 128), (9, 136), (33, 2048), (12, 4104), (10, 14336), (9, 32768), (9, 32776)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("op", ["int4", "int8", "int8_affine", "fp8", "mxfp4", "mxfp4_64", "nvfp4", "kv"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_quantizer_same_on_both_paths(rows, cols, op, dtype):
    print_case("quantizer paths", op, f"{rows}x{cols}", str(dtype))
    x = _hostile(rows, cols, dtype, rows + cols)
    f = _ops()[op]
    assert x.data_ptr() % 16 == 0
    _same(f(x), f(_shifted(x)), f"{op} {rows}x{cols}")


def _ordinary(rows, cols, dtype, seed):
    """Finite rows without a huge value, so that one scale for the whole tensor (NVFP4's global one) keeps ordinary
    quotients: blocks of mixed magnitudes, quotients that underflow, code ties and signed zeros."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * torch.exp2(torch.randint(-12, 1, (rows, max(cols // 8, 1)), generator=g).float()
                                                          ).repeat_interleave(8, dim=1)[:, :cols]
    x[:, 1::11] *= 1e-30 if dtype != torch.float16 else 1e-4
    x[:, 2::13] = -0.0
    x[-1] = (torch.arange(cols) % 25 - 12) * 0.25  # with 6 as the maximum of each block: every E2M1 tie
    x[-1, ::8] = 6.0
    return x.to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("op", ["int4", "int8", "int8_affine", "fp8", "mxfp4", "mxfp4_64", "nvfp4", "kv"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_quantizer_same_on_both_paths_finite(rows, cols, op, dtype):
    print_case("quantizer paths, finite", op, f"{rows}x{cols}", str(dtype))
    x = _ordinary(rows, cols, dtype, rows + cols)
    f = _ops()[op]
    out = f(x)
    _same(out, f(_shifted(x)), f"{op} {rows}x{cols}")
    if op == "nvfp4":
        assert bool(torch.isfinite(out[2]).all()) and out[0].unique().numel() >= (4 if cols < 128 else 12)


@pytest.mark.parametrize("rows,cols", [(1, 128), (16, 128), (17, 256), (40, 384), (1030, 1152), (33, 4096)])
def test_tilers_same_on_both_paths(rows, cols):
    from scratch_llm_amd.quant import fp8_weights as f8, int4_group as i4, int8 as i8, nvfp4_mxfp4 as f4

    print_case("tiler paths", f"{rows}x{cols}")
    g = torch.Generator().manual_seed(rows + cols)
    q4 = torch.randint(-8, 8, (rows, cols), generator=g, dtype=torch.int8).to(DEV)
    s4 = torch.rand(rows, cols // 128, generator=g).to(DEV)
    p4 = i4.pack_int4(q4.reshape(-1))
    q8 = torch.randint(-128, 128, (rows, cols), generator=g, dtype=torch.int8).to(DEV)
    s8 = torch.rand(rows, 1, generator=g).to(DEV)
    mx = f4.mxfp4_quantize(torch.randn(rows, cols, generator=g).to(DEV))
    mp, ms = f4.mxfp4_pack_weight(mx)
    mx2 = type(mx)(_shifted(mx.codes), mx.s_block, mx.shape, mx.n, mx.block)
    c8, sc8 = f8.quantize_per_channel(torch.randn(rows, cols, generator=g).to(DEV))
    pairs = {
        "int4": (i4.tile_int4(q4, s4).wt, i4.tile_int4(_shifted(q4), s4).wt),
        "int4 packed": (i4.tile_int4(q4, s4).wt, i4.tile_int4_packed(p4, s4, (rows, cols)).wt),
        "int8": (i8.tile_int8(q8, s8).wt, i8.tile_int8(_shifted(q8), s8).wt),
        "fp8": (f8.tile_fp8(c8, sc8).wt, f8.tile_fp8(_shifted(c8.view(torch.uint8)).view(c8.dtype), sc8).wt),
        "fp4": (f4.tile_fp4(mx).wt, f4.tile_fp4(mx2).wt),
        "fp4 packed": (f4.tile_mxfp4_packed(mp, ms).wt, f4.tile_mxfp4_packed(_shifted(mp), ms).wt),
    }
    for name, (a, b) in pairs.items():
        _same([a], [b], name)
    assert torch.equal(i8.untile_int8(i8.tile_int8(q8, s8)), q8)
    assert torch.equal(i4.untile_int4(i4.tile_int4(q4, s4))[0], q4)


# one row, partial tiles of both sizes, the larger tile (256 tiles of 128 and more), k below, at and past the ring's
# stages, a k that is no multiple of 16 (the ragged kernel), and n that is no multiple of 4 (scalar stores)
@pytest.mark.parametrize("m,n,k", [(1, 1, 16), (3, 70, 64), (64, 64, 128), (65, 129, 1040), (17, 200, 4096), (2049, 2050, 272),
                                   (2048, 2048, 512), (130, 66, 100), (5, 7, 1), (66, 130, 4095), (300, 4096, 48)])
def test_w8a8_edges(m, n, k):
    from scratch_llm_amd.quant import int8 as i8

    print_case("w8a8", f"m={m}", f"n={n}", f"k={k}")
    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g).to(DEV)
    w = torch.randn(n, k, generator=g).to(DEV)
    y = i8.w8a8_linear(x, w).double().cpu().numpy()
    (qx, sx), (qw, sw) = i8.quantize_symmetric(x, axis=0), i8.quantize_symmetric(w, axis=0)
    acc = qx.double().cpu().numpy() @ qw.double().cpu().numpy().T  # whole numbers below 2**53: exact
    ref = acc * sx.double().cpu().numpy().reshape(-1, 1) * sw.double().cpu().numpy().reshape(1, -1)
    assert np.all(np.abs(y - ref) <= 3.01 * 2.0**-24 * np.abs(ref))


# the call that quantizes both operands in one launch against the quantizer and the product called one by one, at the
# edges of its row chunks (2048, 4096, .. columns), and the forms that it does not take (k % 16, unaligned, two dtypes)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 1, 16), (1, 33, 2048), (5, 3, 2064), (33, 70, 4112), (2, 9, 16400), (3, 2, 32768),
                                   (3, 2, 32784), (4, 6, 100), (130, 515, 256)])
def test_w8a8_one_launch(m, n, k, dtype):
    from scratch_llm_amd import _lib
    from scratch_llm_amd.quant import int8 as i8

    print_case("w8a8 one launch", f"m={m}", f"n={n}", f"k={k}", f"dtype={dtype}")
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(dtype), torch.randn(n, k, generator=g).to(dtype)
    w[0] = 0.0  # the scale is eps
    if m > 2:
        x[1, 3], x[2, 5] = float("nan"), float("inf")
    x, w = x.to(DEV), w.to(DEV)

    def parts(x, w):
        (qx, sx), (qw, sw) = i8.quantize_symmetric(x, axis=0), i8.quantize_symmetric(w, axis=0)
        y = torch.empty(m, n, device=DEV)
        _lib.check(_lib.load().sqx_w8a8_gemm(qx.data_ptr(), sx.data_ptr(), _lib.sqx_dtype(sx.dtype), qw.data_ptr(),
                                             sw.data_ptr(), _lib.sqx_dtype(sw.dtype), y.data_ptr(), m, n, k,
                                             _lib.stream_ptr(y.device)), "w8a8")
        return y

    ref = parts(x, w)
    _same([i8.w8a8_linear(x, w)], [ref], "one launch")
    _same([i8.w8a8_linear(_shifted(x), w)], [ref], "unaligned x")
    _same([i8.w8a8_linear(x.t().contiguous().t(), w.t().contiguous().t())], [ref], "strided")
    _same([i8.w8a8_linear(x[None], w)], [ref[None]], "batch")
    other = torch.bfloat16 if dtype != torch.bfloat16 else torch.float32
    _same([i8.w8a8_linear(x, w.to(other))], [parts(x, w.to(other))], "two dtypes")


# more rows than a launch holds workgroups of 256 threads: rows too short for a workgroup each
@pytest.mark.parametrize("cols", [8, 16])
def test_int8_many_short_rows(cols):
    from scratch_llm_amd.quant import int8 as i8

    rows = 1 << 24
    print_case("int8 many short rows", f"{rows}x{cols}")
    g = torch.Generator(device=DEV).manual_seed(cols)
    x = torch.randn(rows, cols, device=DEV, generator=g, dtype=torch.bfloat16)
    parts = [slice(0, 100), slice(rows // 2 - 50, rows // 2 + 50), slice(rows - 100, rows)]
    for quantize in (i8.quantize_symmetric, i8.quantize_affine):
        whole = quantize(x, axis=0)
        for p in parts:
            _same([t[p] for t in whole], quantize(x[p].contiguous(), axis=0), f"{quantize.__name__} rows {p.start}")
        del whole
    if cols % 16 == 0:
        w = torch.randn(3, cols, device=DEV, generator=g, dtype=torch.bfloat16)
        y = i8.w8a8_linear(x, w)
        for p in parts:
            _same([y[p]], [i8.w8a8_linear(x[p].contiguous(), w)], f"w8a8 rows {p.start}")


def test_mxfp4_as_many_elements_as_a_launch_has_no_threads_for():
    """2^35 elements: eight a thread would be 2^32 threads, which no launch holds; a block of 128 a thread fits."""
    from scratch_llm_amd import _lib

    n, block = 1 << 35, 128
    free, _ = torch.cuda.mem_get_info()
    if free < 120 << 30:
        pytest.skip("needs 120 GiB of device memory")
    print_case("mxfp4 quantize", f"n={n}")
    lib = _lib.load()
    x = torch.zeros(n, device=DEV, dtype=torch.bfloat16)
    codes = torch.full((n,), 7, device=DEV, dtype=torch.uint8)
    s_block = torch.full((n // block,), 7.0, device=DEV)
    tail = torch.randn(block, device=DEV, generator=torch.Generator(device=DEV).manual_seed(5)).to(torch.bfloat16)
    x[-block:] = tail
    stream = _lib.stream_ptr(x.device)
    _lib.check(lib.sqx_mxfp4_quantize(x.data_ptr(), _lib.DTYPE_BF16, n, block, codes.data_ptr(), s_block.data_ptr(), None,
                                      stream), "sqx_mxfp4_quantize")
    tc, ts = torch.empty(block, device=DEV, dtype=torch.uint8), torch.empty(1, device=DEV)
    _lib.check(lib.sqx_mxfp4_quantize(tail.data_ptr(), _lib.DTYPE_BF16, block, block, tc.data_ptr(), ts.data_ptr(), None,
                                      stream), "sqx_mxfp4_quantize")
    assert torch.equal(codes[-block:], tc) and torch.equal(s_block[-1:], ts)
    assert bool((s_block[:-1] == s_block[0]).all()) and float(s_block[0]) != 7.0
    for lo in range(0, n - block, 1 << 31):  # parts small enough for a mask of their own
        assert not bool(codes[lo:min(lo + (1 << 31), n - block)].any())
    del x, codes, s_block
    torch.cuda.empty_cache()


# the edge between one workgroup per head and the sliced form (16384 elements a head), rows that split it unevenly,
# and a head count past one block of the finishing kernel
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,t,d", [(1, 1, 1, 1), (1, 8, 1, 128), (64, 8, 2, 128), (3, 5, 41, 131), (16383, 1, 1, 1), (1, 70, 129, 128),
                                     (129, 3, 1, 128), (0, 4, 3, 8)])
def test_per_head_amax(b, h, t, d, dtype):
    from scratch_llm_amd.quant import fp8_kv_per_head as kv

    print_case("per-head amax", f"{b}x{h}x{t}x{d}", str(dtype))
    g = torch.Generator().manual_seed(b + h + t + d)
    x = torch.randn(b, h, t, d, generator=g).to(dtype)
    if b:
        x[-1, -1, -1, -1] = -30.0  # the last element of the last slice
    ref = x.float().abs().permute(1, 0, 2, 3).reshape(h, -1).max(dim=1).values if b else torch.zeros(h)
    assert torch.equal(kv.per_head_amax(x.to(DEV)).float().cpu().reshape(-1), ref)
    want = (ref / 448.0).clamp_min(1.0 / (448.0 * 512.0))
    assert torch.equal(kv.per_head_scale(x.to(DEV)).float().cpu().reshape(-1), want)
    if b and h > 1:
        x[0, 0, 0, 0], x[b // 2, 1, 0, d // 2] = float("nan"), float("inf")
        a = kv.per_head_amax(x.to(DEV)).float().cpu().reshape(-1)
        assert bool(torch.isnan(a[0])) and float(a[1]) == float("inf") and torch.equal(a[2:], ref[2:])
