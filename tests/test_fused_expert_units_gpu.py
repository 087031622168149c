"""The fused expert's GEMM units at the shapes that select each of their forms
(row tiles x column tiles of a unit: 4x1, 2x1, 1x1, 2x2, 1x2), ragged row tiles
included, against the layer-by-layer engine and the oracle on the same seeded
weights and inputs.  Tolerances as in test_fused_expert_gpu.py: 5e-2 absolute
against the oracle's actions, 2e-2 between the engines."""

import dataclasses

import pytest
import torch

import oracle.smolvla_ref as ref
from smolvla.config import small_config
from smolvla.params import smolvla_inputs, smolvla_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,chunk,batch", [
    (144, 192, 10, 1),      # one row tile: 4x1
    (1040, 192, 50, 1),     # 65 column tiles: O and down 2x1 (norm over more than 1024)
    (144, 2048, 64, 1),     # 256 column tiles, every row in use: norm + gate|up 2x2
    (144, 1600, 33, 1),     # three row tiles: 2x2 with an empty fourth
    (144, 1600, 17, 1),     # two row tiles, one row in the second: 1x2
    (144, 1600, 25, 2),     # two samples: QKV keeps one row group
    (1280, 192, 50, 1),     # 80 column tiles: O and down 1x2 with the plain epilogue
    (2048, 192, 64, 1),     # the same with 128 column tiles, every row in use
])
def test_unit_forms(hidden, inter, chunk, batch):
    from smolvla.pipeline import SmolVLAEngine
    cfg = small_config()
    cfg = cfg.replace(expert=dataclasses.replace(cfg.expert, hidden=hidden, inter=inter),
                      chunk=chunk)
    P = smolvla_params(cfg, seed=hidden + chunk, norm_init="random")
    inputs = smolvla_inputs(cfg, batch=batch, seed=inter + batch)
    dev = [t.cuda() for t in inputs]
    print(f"hidden {hidden} inter {inter} chunk {chunk} batch {batch}", flush=True)
    eng = SmolVLAEngine(cfg, P, batch, fused_expert=True)
    got = eng.run(*dev).cpu()
    assert eng.fx.status() == 0 and torch.isfinite(got).all()
    assert torch.equal(eng.run(*dev).cpu(), got)
    layered = SmolVLAEngine(cfg, P, batch, fused_expert=False).run(*dev).cpu()
    want = ref.smolvla_chunk(*inputs, P, cfg)
    assert (got - layered).abs().max() <= 2e-2
    assert (got - want).abs().max() <= 5e-2
