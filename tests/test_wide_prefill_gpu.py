"""The wide prefill pass (65 to 512 prompt tokens in one go): its GEMM against the
oracle's canonical sum and the block launchers, and the session's prefill against blocks."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import dev, host, say

pytestmark = pytest.mark.gpu


def _problem(gx, orc, fmt, rows, cols, tokens, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    w[rng.random((rows, cols // 128)).repeat(128, axis=1) < 0.02] = 0.0   # whole zero groups
    _, codes, scales = orc.quantize_group128(w, fmt)
    tiled, tscales = gx.tile_group128(fmt, codes, scales, rows, cols)
    x = (rng.standard_normal((tokens, cols)) * np.exp(rng.normal(0, 2, (tokens, 1)))).astype(np.float16)
    x[tokens // 2, :128] = 0.0
    packed = np.empty((tokens, cols // 2), np.uint8)
    ascales = np.empty((tokens, cols // 128), np.uint16)
    for a in range(0, tokens, 32):
        packed[a:a + 32], ascales[a:a + 32] = orc.quantize_activation_i4(x[a:a + 32].view(np.uint16))
    return codes, scales, tiled, tscales, packed, ascales


# Edges of the 128 x 128 block and of a 16-token tile, one and several ranges and splits,
# fewer and more steps than LDS stages, a short last row block; the reference's longest K in its planes.
@pytest.mark.parametrize("fmt,rows,cols,tokens,splits", [
    (3, 16, 128, 1, 1), (2, 128, 256, 16, 1), (1, 144, 384, 33, 1), (3, 272, 1280, 128, 1), (2, 112, 1408, 129, 1),
    (3, 256, 2688, 65, 2), (2, 160, 5120, 100, 4), (1, 16, 2560, 257, 8), (2, 128, 640, 47, 5),
    (3, 272, 17408, 97, 4), (2, 144, 5120, 200, 1)])
def test_prefill_gemm_equals_canonical_sum(gx, orc, device, fmt, rows, cols, tokens, splits):
    import torch
    codes, scales, tiled, tscales, packed, ascales = _problem(gx, orc, fmt, rows, cols, tokens, rows + cols + tokens)
    w, ws, a, as_ = (dev(v, device) for v in (tiled, tscales, packed, ascales))
    size = int(gx.lib().gfxinfer_debug_gemm_prefill_workspace_bytes(cols, tokens))
    work = torch.empty(size, dtype=torch.uint8, device=device)
    out = torch.full((splits, tokens, rows), float("nan"), device=device)
    stream = torch.cuda.current_stream().cuda_stream
    say("prefill GEMM", fmt, rows, cols, tokens, splits)

    def launch(target, half):
        return gx.lib().gfxinfer_debug_gemm_prefill(fmt, w.data_ptr(), ws.data_ptr(), a.data_ptr(), as_.data_ptr(),
                                                    target.data_ptr(), half, rows, cols, tokens,
                                                    1 if half else splits, work.data_ptr(), size, stream)
    gx.check(launch(out, 0))
    torch.cuda.synchronize()
    partials = orc.gemm_partials(orc.unpack_weights(codes, rows, cols, fmt), orc.unpack_a4(packed, cols))
    want = orc.gemm_epilogue_ranges(partials, orc.f32_to_f16_bits(scales), ascales, splits)
    assert np.array_equal(host(out), want)
    if splits == 1:
        half = torch.zeros(tokens, rows, dtype=torch.int16, device=device)
        gx.check(launch(half, 1))
        torch.cuda.synchronize()
        assert np.array_equal(host(half, np.uint16), orc.f32_to_f16_bits(want[0]))


@pytest.fixture(scope="module", params=["27b", "reference"])
def model(device, request):
    from gfxinfer_amd.runtime import SyntheticModel, reference_tiny_spec, tiny_spec
    spec = tiny_spec(full_attention_interval=2, gdn_key_head_count=4) if request.param == "27b" else reference_tiny_spec()
    say("synthetic model", request.param)
    m = SyntheticModel(spec, 17)
    yield m
    m.close()


BUFFERS = (("conv_states", np.uint16), ("gdn_states", np.uint32), ("key_caches", np.uint16), ("value_caches", np.uint16),
           ("mtp_key_cache", np.uint16), ("mtp_value_cache", np.uint16), ("hidden", np.uint16))
CONTEXT = 640


def _blocks(session, prompt, mtp):
    """The same prompt in calls of at most 32 tokens, which take the block pass."""
    for a in range(0, len(prompt), 32):
        token = session.prefill(prompt[a:a + 32], sync_mtp=mtp)
    return token


def _same(a, b, rows, context=CONTEXT):
    assert (a.position(), a.mtp_position()) == (b.position(), b.mtp_position())
    spec = a.model.spec
    kv = spec.kv_head_count * spec.attention_head_size
    for name, dtype in BUFFERS:
        x, y = a.buffer(name, dtype), b.buffer(name, dtype)
        if "cache" in name:
            used = a.mtp_position() if name.startswith("mtp") else a.position()
            x, y = (v.reshape(-1, context, kv)[:, :used] for v in (x, y))
        assert np.array_equal(x, y), name
    x, y = (s.buffer("logits", np.uint32, rows * spec.vocabulary_size) for s in (a, b))
    assert np.array_equal(x, y)


@pytest.mark.parametrize("n,mtp", [(64, True), (65, False), (97, True), (512, True), (513, True), (577, True)])
def test_wide_prefill_equals_blocks(model, n, mtp):
    from gfxinfer_amd.runtime import QwenDecodeSession
    prompt = np.random.default_rng(n).integers(0, 1000, n).astype(np.uint32)
    a, b = (QwenDecodeSession(model, CONTEXT, 5, keep_logits=True) for _ in range(2))
    say("block prefill", n)
    want = _blocks(a, prompt, mtp)
    say("wide prefill", n)
    assert b.prefill(prompt, sync_mtp=mtp) == want
    _same(a, b, (n - 1) % 32 + 1)
    # a second segment on a session that is not fresh, then a round (its graph reads the state parity)
    more = prompt[:70 if n < 500 else 40]
    assert b.prefill(more, sync_mtp=mtp) == (want := _blocks(a, more, mtp))
    if mtp:
        ra, rb = a.speculative_step(want, 4), b.speculative_step(want, 4)
        assert (ra.tokens, ra.accepted_drafts) == (rb.tokens, rb.accepted_drafts)
        _same(a, b, 5)
    a.close()
    b.close()


def test_wide_prefill_refuses_what_blocks_refuse(model):
    """A token outside the vocabulary: the blocks before it stay, its block does not run."""
    from gfxinfer_amd import GfxinferError
    from gfxinfer_amd.runtime import QwenDecodeSession
    prompt = np.random.default_rng(3).integers(0, 1000, 150).astype(np.uint32)
    prompt[110] = model.spec.vocabulary_size
    a, b = (QwenDecodeSession(model, CONTEXT, 0, keep_logits=True) for _ in range(2))
    _blocks(a, prompt[:96], True)
    with pytest.raises(GfxinferError):
        b.prefill(prompt)
    _same(a, b, 32)
    with pytest.raises(GfxinferError):
        b.prefill(np.zeros(CONTEXT, np.uint32))
    _same(a, b, 32)
    a.close()
    b.close()


def _scratch(model, refuse=-1):
    from gfxinfer_amd import lib
    return int(lib().gfxinfer_debug_model_wide_scratch(model.handle, refuse))


def test_scratch_belongs_to_the_model(model):
    """Sessions hold no memory for wide passes, the first such pass allocates the model's scratch, later sessions
    use the same one, and a session creation that does not fit gets it back."""
    from gfxinfer_amd import GfxinferError
    from gfxinfer_amd.runtime import QwenDecodeSession
    prompt = np.random.default_rng(9).integers(0, 1000, 200).astype(np.uint32)
    _scratch(model, 1), _scratch(model, 0)
    small, large = QwenDecodeSession(model, 64), QwenDecodeSession(model, 65)
    assert large.summary().arena_bytes - small.summary().arena_bytes < 1 << 20
    small.close(), large.close()
    a, b, c = (QwenDecodeSession(model, CONTEXT, 0, keep_logits=True) for _ in range(3))
    say("prompts on one scratch")
    _blocks(a, prompt[:100], True)
    b.prefill(prompt[:64])
    assert _scratch(model) == 0                       # short prompts need none
    c.prefill(prompt[:100])
    held = _scratch(model)
    assert held > 0 and c.prefill(prompt[100:]) == _blocks(a, prompt[100:], True)
    b.prefill(prompt[64:])
    assert _scratch(model) == held
    _same(a, c, 4)
    with pytest.raises(GfxinferError):
        QwenDecodeSession(model, 1 << 40)             # exceeds any memory: refused before anything is launched
    assert _scratch(model) == 0
    say("prompts after the scratch was given back")
    assert c.prefill(prompt) == _blocks(a, prompt, True) and _scratch(model) == held
    _same(a, c, 8)
    for s in (a, b, c):
        s.close()


def test_prompt_without_scratch_runs_in_blocks(model):
    """The scratch's allocation fails: the same results, and nothing later sees the failure."""
    from gfxinfer_amd.runtime import QwenDecodeSession
    prompt = np.random.default_rng(10).integers(0, 1000, 600).astype(np.uint32)
    a, b = (QwenDecodeSession(model, CONTEXT, 5, keep_logits=True) for _ in range(2))
    want = _blocks(a, prompt, True)
    _scratch(model, 1)
    try:
        say("prompt without scratch")
        assert b.prefill(prompt) == want and _scratch(model) == 0
    finally:
        _scratch(model, 0)
    _same(a, b, 24)
    ra, rb = a.speculative_step(want, 4), b.speculative_step(want, 4)
    assert (ra.tokens, ra.accepted_drafts) == (rb.tokens, rb.accepted_drafts)
    _same(a, b, 5)
    a.close()
    b.close()


# Four layers (three GDN, one attention) at real widths.  The attention of a pass runs in several launches here: at
# 40/8 x 128 with its partial results in the scratch (context 4096) and in the block workspace (8192), and at 24/4 x 256.
@pytest.mark.parametrize("shape,n,context", [("27b", 2600, 4096), ("27b", 1100, 8192), ("reference", 1125, 2048)])
def test_full_width_wide_prefill_equals_blocks(device, shape, n, context):
    from gfxinfer_amd import runtime as rt
    spec = rt.qwen38_27b_spec() if shape == "27b" else rt.qwen38_reference_spec()
    spec.layer_count, spec.w3_mlp_layers = 4, 3
    say("full-width model", shape)
    model = rt.SyntheticModel(spec, 23)
    prompt = np.random.default_rng(n).integers(0, spec.tokenizer_vocabulary_size, n).astype(np.uint32)
    a, b = (rt.QwenDecodeSession(model, context, 0, keep_logits=True) for _ in range(2))
    say("blocks", shape, n)
    want = _blocks(a, prompt, True)
    say("wide passes", shape, n)
    assert b.prefill(prompt) == want
    _same(a, b, (n - 1) % 32 + 1, context)
    ra, rb = a.speculative_step(want, 4), b.speculative_step(want, 4)
    assert (ra.tokens, ra.accepted_drafts) == (rb.tokens, rb.accepted_drafts)
    _same(a, b, 5, context)
    a.close()
    b.close()
    model.close()
