"""The 9-32 token GEMM at grids that take two, three and four row tiles per wave, short last
blocks among them, against the same tokens one by one (the one-token kernel's results are
checked against the oracle in test_gemm_gpu.py; a token's output does not depend on the
batch)."""
from __future__ import annotations

import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu


# row tiles: 1024 and 1601 take 4 (1601 with a last block of one tile), 1100 and 1538 take 3,
# 1026 x 2 splits takes 3 with 3-group chunks, 1280 takes 2 or 3, 9217 takes 4 by the tie rule
@pytest.mark.parametrize("fmt,tiles,cols,splits,tokens", [
    (2, 1024, 1408, 1, 9), (3, 1601, 1408, 1, 17), (1, 1601, 1536, 1, 32), (2, 1100, 2560, 1, 16),
    (3, 1538, 1408, 1, 32), (2, 1026, 2816, 2, 24), (3, 1280, 2304, 1, 11), (2, 9217, 1408, 1, 20)])
def test_row_tiles_per_wave(gx, device, fmt, tiles, cols, splits, tokens):
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
