"""The all-layer GDN restore on both sides of its streamed-store rule (64 MB of states)
against the one-layer restore of each layer."""
from __future__ import annotations

import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,value_heads,accepted", [(32, 32, 3), (33, 32, 1), (22, 48, 32)])
def test_all_layers_equal_one_layer_restores(gx, device, layers, value_heads, accepted):
    import torch
    g = torch.Generator(device=device).manual_seed(layers)
    channels, logged = (32 + value_heads) * 128, 32

    def rand(*shape):
        return torch.randn(*shape, device=device, generator=g)
    conv = rand(layers, channels, 4).half()
    states = rand(layers, value_heads, 128, 128)
    logs = [rand(layers, logged, channels).half(), rand(layers, logged, 16 * 128), rand(layers, logged, value_heads * 128),
            torch.rand(layers, logged, value_heads, device=device, generator=g)]
    want_conv, want_states = conv.clone(), states.clone()
    stream = torch.cuda.current_stream().cuda_stream
    say("restore", layers, value_heads, accepted)
    gx.check(gx.lib().gfxinfer_launch_gdn_restore_prefix_all(
        conv.data_ptr(), states.data_ptr(), *(x.data_ptr() for x in logs), channels, layers, logged, accepted, 16,
        value_heads, 128, stream))
    for i in range(layers):
        gx.check(gx.lib().gfxinfer_launch_gdn_restore_prefix(
            want_conv[i].data_ptr(), want_states[i].data_ptr(), *(x[i].data_ptr() for x in logs), channels, accepted, 16,
            value_heads, 128, stream))
    torch.cuda.synchronize()
    assert torch.equal(conv, want_conv) and torch.equal(states, want_states)
