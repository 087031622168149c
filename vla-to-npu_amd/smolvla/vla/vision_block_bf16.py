"""SigLIP-style ViT block, bf16, on gfx950.

Drop-in for ``vision_block(x, params) -> out`` (reference
vla/vision_block_bf16.py:308-420): pre-LayerNorm (with the ``b_norm_*``
shifts), multi-head attention (12 heads x 64, no mask), GELU MLP, residuals.
Optional SigLIP biases ``bq bk bv bo b_up b_down`` are honoured when present.
Defaults: LN eps 1e-6 and tanh-GELU (target configuration); the reference
module's choices are ``VitConfig(ln_eps=1e-5, gelu="erf")``.
"""

from __future__ import annotations

import torch

from .. import layers
from ..config import VitConfig
from ._common import as_batched, as_rows, prepared, to_device

SEQ = 1024
EMBD = 768
N_HEAD = 12
HEAD_DIM = 64
FFN_HID = 3072
DEFAULT_CFG = VitConfig()


def _prep_any_rows(p, device):
    """One set of packed weights for calls of every size: beside the row-major
    ones blocked copies of every projection that a large enough call moves to
    the slab-blocked 256x256 GEMM (each call's own plan picks among them).  The
    first call, whatever its size, then packs for all others: one of another
    size finds nothing left to pack, also where it must not (under capture, or
    beside calls on other streams)."""
    return layers.prep_vit(p, device, rows=layers.ANY_ROWS)


def vision_block(x_np, params, cfg: VitConfig = DEFAULT_CFG):
    x, back = to_device(x_np)
    x3, squeeze = as_batched(x)
    B, T, H = x3.shape
    x2 = as_rows(x3)
    P = prepared(params, _prep_any_rows)
    out = torch.empty_like(x2)
    layers.vit_layer(x2, P, cfg, B, T, out=out)
    return back(out.view(T, H) if squeeze else out.view(B, T, H))


def vision_encoder(num_layers, x, params, cfg: VitConfig = DEFAULT_CFG):
    """``vision_encoder`` (vla/vla.py:185-188): the same block applied
    ``num_layers`` times, or a list of per-layer params."""
    plist = params if isinstance(params, (list, tuple)) else [params] * num_layers
    for p in plist[:num_layers]:
        x = vision_block(x, p, cfg)
    return x
