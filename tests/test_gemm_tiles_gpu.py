"""The 9-32 token GEMM at grids that take two, three and four row tiles per wave, short last
blocks among them, against the same tokens one by one (the one-token kernel's results are
checked against the oracle in test_gemm_gpu.py; a token's output does not depend on the
batch)."""
from __future__ import annotations

import pytest

from gpu_util import say

# format, row tiles, columns, splits, tokens, the shape the launcher takes (100 x row tiles per wave + groups per chunk):
# last blocks of every length, 2 to 14 ranges on up to eight waves (17408 columns: some waves take two ranges)
CASES = [
    (2, 1024, 1408, 1, 9, 205), (3, 1601, 1408, 1, 17, 202), (1, 1601, 1536, 1, 32, 202), (2, 1100, 2560, 1, 16, 205),
    (3, 1538, 1408, 1, 32, 202), (2, 1026, 2816, 2, 24, 302), (3, 1280, 2304, 1, 11, 205), (2, 9217, 1408, 1, 20, 402),
    (3, 1283, 1408, 1, 30, 205), (2, 2401, 1408, 1, 12, 202), (3, 2399, 1408, 1, 32, 202), (2, 1100, 5120, 1, 32, 302),
    (3, 1027, 4352, 2, 13, 303), (2, 1028, 4352, 2, 19, 303), (3, 2049, 3072, 1, 10, 302), (2, 1726, 5120, 1, 16, 402),
    (3, 1725, 5120, 1, 21, 402), (2, 1024, 17408, 1, 32, 402), (3, 1023, 17408, 1, 31, 202), (2, 1027, 17408, 1, 15, 302),
    (3, 1100, 17408, 1, 32, 302), (1, 3070, 4096, 1, 9, 402)]

# the same with 8-bit activations: format, row tiles, columns, tokens, shape
CASES_A8 = [
    (3, 1025, 2304, 16, 205), (2, 1727, 1408, 9, 202), (3, 1283, 3072, 13, 302), (2, 2175, 2176, 10, 303),
    (3, 2047, 3072, 16, 402), (2, 1027, 17408, 11, 302), (3, 1022, 17408, 15, 205), (2, 1024, 17408, 16, 402)]


@pytest.mark.parametrize("fmt,tiles,cols,tokens,shape", CASES_A8)
def test_shape_of_an_a8_case(gx, fmt, tiles, cols, tokens, shape):
    assert gx.lib().gfxinfer_debug_gemm_direct_shape(8, tiles * 16, cols, tokens, 1) == shape


@pytest.mark.parametrize("fmt,tiles,cols,splits,tokens,shape", CASES)
def test_shape_of_a_case(gx, fmt, tiles, cols, splits, tokens, shape):
    assert gx.lib().gfxinfer_debug_gemm_direct_shape(4, tiles * 16, cols, tokens, splits) == shape


def test_cases_take_every_shape(gx):
    for lo, hi in ((9, 16), (17, 32)):
        assert {c[5] for c in CASES if lo <= c[4] <= hi} == {202, 205, 302, 303, 402}
    assert gx.lib().gfxinfer_debug_gemm_direct_shape(4, 5120, 1280, 32, 1) == 104   # one range
    assert {c[4] for c in CASES_A8} == {202, 205, 302, 303, 402}


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,tiles,cols,splits,tokens,shape", CASES)
def test_row_tiles_per_wave(gx, device, fmt, tiles, cols, splits, tokens, shape):
    import torch
    rows = tiles * 16
    g = torch.Generator(device=device).manual_seed(tiles + tokens)
    codes = torch.randint(0, 256, (gx.tile_bytes(fmt, rows, cols),), dtype=torch.uint8, device=device, generator=g)
    scales = (torch.rand(rows * cols // 128, device=device, generator=g) * 0.02 - 0.01).half()
    x = torch.randn(tokens, cols, device=device, generator=g).half()
    a = torch.empty(tokens, cols // 2, dtype=torch.uint8, device=device)
    as_ = torch.empty(tokens, cols // 128, dtype=torch.float16, device=device)
    gx.launch_quantize_activation_i4(x, a, as_, cols, tokens)
    got = torch.full((splits, tokens, rows), float("nan"), device=device)
    say("GEMM row tiles", fmt, tiles, cols, splits, tokens)
    gx.launch_i4_gemm_split(fmt, codes, scales, a, as_, got, rows, cols, tokens, splits)
    want = torch.empty(splits, 1, rows, device=device)
    for t in range(tokens):
        gx.launch_i4_gemm_split(fmt, codes, scales, a[t], as_[t].contiguous(), want, rows, cols, 1, splits)
        assert torch.equal(got[:, t], want[:, 0]), t


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,tiles,cols,tokens,shape", CASES_A8)
def test_row_tiles_per_wave_a8(gx, device, fmt, tiles, cols, tokens, shape):
    import torch
    rows = tiles * 16
    g = torch.Generator(device=device).manual_seed(tiles + tokens)
    codes = torch.randint(0, 256, (gx.tile_bytes(fmt, rows, cols),), dtype=torch.uint8, device=device, generator=g)
    scales = (torch.rand(rows * cols // 128, device=device, generator=g) * 0.02 - 0.01).half()
    x = torch.randn(tokens, cols, device=device, generator=g).half()
    a = torch.empty(tokens, cols, dtype=torch.int8, device=device)
    as_ = torch.empty(tokens, cols // 128, dtype=torch.float16, device=device)
    gx.launch_quantize_activation_i8(x, a, as_, cols, tokens)
    got = torch.full((tokens, rows), float("nan"), device=device)
    say("A8 GEMM row tiles", fmt, tiles, cols, tokens)
    gx.launch_i8_gemm(fmt, codes, scales, a, as_, got, rows, cols, tokens)
    want = torch.empty(1, rows, device=device)
    for t in range(tokens):
        gx.launch_i8_gemm(fmt, codes, scales, a[t], as_[t].contiguous(), want, rows, cols, 1)
        assert torch.equal(got[t], want[0]), t
