"""Packed weights kept between layer calls, where a call comes inside a graph
capture or on another stream than the one that packed."""

import pytest
import torch

from smolvla.params import _Gen, decoder_layer_params, vit_layer_params

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _capture(fn):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def test_vision_block_capture_after_a_warm_up_of_another_size():
    """One small eager call, then a capture of a size on the slab-blocked
    GEMM: an eager call before the first replay, and every replay, give the
    bits of a call whose weights were packed in the open."""
    from smolvla.config import VitConfig
    from smolvla.vla.vision_block_bf16 import vision_block
    g = _Gen(9, device="cuda", norm_init="random")
    params = vit_layer_params(g, VitConfig())
    x = torch.randn(4, 1024, 768, device="cuda").to(BF16)
    want = vision_block(x, dict(params))
    vision_block(x[:1, :196], params)
    graph, out = _capture(lambda: vision_block(x, params))
    assert torch.equal(vision_block(x, params), want)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(vision_block(x, params), want)


def test_capture_with_no_call_before():
    """Weights never packed before the capture: the graph packs them itself on
    every replay, and an eager call, before and after, packs its own."""
    from smolvla.config import DecoderConfig
    from smolvla.vla.text_encoder_bf16 import text_encoder_forward
    g = _Gen(10, device="cuda", norm_init="random")
    params = decoder_layer_params(g, DecoderConfig())
    x = torch.randn(2, 37, 960, device="cuda").to(BF16)
    want = text_encoder_forward(x, dict(params))
    graph, out = _capture(lambda: text_encoder_forward(x, params))

    def same(got):
        assert all(torch.equal(a, b) for a, b in zip(got, want))

    same(text_encoder_forward(x, params))
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        same(out)
        same(text_encoder_forward(x, params))


def test_a_call_on_another_stream_waits_for_the_packing():
    """The first call packs behind other work of its stream; a call on a second
    stream, made at once, gives the same bits."""
    from smolvla.vla.action_expert_bf16 import DEFAULT_CFG, action_expert_self_forward
    g = _Gen(11, device="cuda", norm_init="random")
    params = decoder_layer_params(g, DEFAULT_CFG)
    x = torch.randn(2, 50, 720, device="cuda").to(BF16)
    want = action_expert_self_forward(x, dict(params))
    busy = torch.randn(8192, 8192, device="cuda")
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        for _ in range(4):
            busy = busy @ busy * 1e-4
        a = action_expert_self_forward(x, params)
    with torch.cuda.stream(second):
        b = action_expert_self_forward(x, params)
    torch.cuda.synchronize()
    assert torch.equal(a, want) and torch.equal(b, want)
