"""The layer functions read their input where it is and write a new tensor:
inputs that are views (strided, or starting off a 16-byte boundary) give the
bits of a fresh copy, and no input is changed."""

import pytest
import torch

from smolvla.params import _Gen, decoder_layer_params, expert_cross_layer_params, vit_layer_params

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _views(x):
    """The same values: contiguous, off a 16-byte boundary, column slice."""
    flat = torch.zeros(x.numel() + 1, dtype=BF16, device="cuda")
    flat[1:] = x.reshape(-1)
    wide = torch.zeros(*x.shape[:-1], x.shape[-1] + 8, dtype=BF16, device="cuda")
    wide[..., 8:] = x
    return x.clone(), flat[1:].view(x.shape), wide[..., 8:]


def _same(run, x):
    want = None
    for v in _views(x):
        out = run(v)
        out = out if isinstance(out, tuple) else (out,)
        want = want or [t.clone() for t in out]
        for a, b in zip(out, want):
            assert a.is_contiguous() and torch.equal(a, b)
        assert torch.equal(v, x)


def test_views_and_inputs_kept():
    from smolvla.config import DecoderConfig
    from smolvla.vla.action_expert_bf16 import (DEFAULT_CFG, action_expert_cross_forward,
                                                action_expert_self_forward)
    from smolvla.vla.text_encoder_bf16 import text_encoder_forward
    from smolvla.vla.vision_block_bf16 import vision_block
    x_of = lambda *s: torch.randn(*s, device="cuda").to(BF16)  # noqa: E731
    g = _Gen(5, device="cuda", norm_init="random")
    p = decoder_layer_params(g, DecoderConfig())
    _same(lambda x: text_encoder_forward(x, p), x_of(2, 37, 960))
    p = decoder_layer_params(g, DEFAULT_CFG)
    _same(lambda x: action_expert_self_forward(x, p), x_of(3, 50, 720))
    c = expert_cross_layer_params(g, DEFAULT_CFG, 320)
    k, v = x_of(3, 70, 320), x_of(3, 70, 320)
    _same(lambda x: action_expert_cross_forward(x, k, v, c), x_of(3, 50, 720))
    from smolvla.config import VitConfig
    pv = vit_layer_params(g, VitConfig())
    _same(lambda x: vision_block(x, pv), x_of(1, 196, 768))
    _same(lambda x: vision_block(x, pv), x_of(12, 1024, 768))   # every projection slab-blocked


@pytest.mark.parametrize("L", [64, 65, 100, 128, 129, 300])
def test_rows_on_lines(L):
    """Weights and norm outputs whose rows start on 128-byte lines give the
    bits of packed ones (below and from LINE_MIN_ROWS)."""
    from smolvla import layers
    from smolvla.vla.action_expert_bf16 import DEFAULT_CFG as cfg
    g = _Gen(6, device="cuda", norm_init="random")
    rope = layers.Rope.make(L, cfg.head_dim, cfg.rope_theta, "cuda")
    x = torch.randn(L, cfg.hidden, device="cuda").to(BF16)
    p = decoder_layer_params(g, cfg)
    c = expert_cross_layer_params(g, cfg, 320)
    ck, cv = (torch.randn(70, cfg.kv_dim, device="cuda").to(BF16) for _ in range(2))
    got = []
    for rows in (0, L):
        P, C = layers.prep_decoder(p, "cuda", rows=rows), layers.prep_cross(c, "cuda", rows=rows)
        padded = rows >= layers.LINE_MIN_ROWS
        assert all((w.stride(0) == 768) == padded for w in (P["wqkv"], P["wgu"], C["wq"], C["wgu"]))
        y = x.clone()
        kv = layers.decoder_layer(y, P, cfg, 1, L, rope)
        z = x.clone()
        layers.cross_layer(z, ck, cv, C, cfg, 1, L, 70, rope)
        got.append((y, kv, z))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("rows", [1, 37])
def test_exported_kv_are_tensors_of_their_own(rows):
    """K and V share no storage and no version: keeping one does not hold the
    other, an edit of one is none of the other."""
    from smolvla.config import DecoderConfig
    from smolvla.vla.text_encoder_bf16 import text_encoder_forward
    p = decoder_layer_params(_Gen(7, device="cuda", norm_init="random"), DecoderConfig())
    x = torch.randn(rows, 960, device="cuda").to(BF16)
    _, key, value = text_encoder_forward(x, p)
    for t in (key, value):
        assert t.is_contiguous() and t.untyped_storage().nbytes() == t.numel() * 2
    kept = value._version
    key.zero_()
    assert value._version == kept and value.any()
