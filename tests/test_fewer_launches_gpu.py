"""Two launches folded into one give the bits of the two: the RMSNorm that also
writes the RoPE tables."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).cuda()


# rows: one block's remainder, whole blocks; positions: fewer and more table
# entries than one block of 256, a remainder; columns: smallest and largest
@pytest.mark.parametrize("rows,cols,pos,dim", [
    (1, 8, 1, 2), (3, 720, 7, 64), (4, 720, 8, 64), (50, 720, 50, 64), (241, 960, 241, 64),
    (1665, 960, 333, 80), (5, 2048, 1, 512)])
def test_norm_with_tables(rows, cols, pos, dim):
    from smolvla import ops
    x, w = _rand(rows, cols + 8, seed=1)[:, :cols], _rand(cols, seed=2)
    c, s = ops.rope_table(pos, dim, 10000.0, device=x.device)
    c1, s1 = torch.full_like(c, 7), torch.full_like(s, 7)
    y = ops.rmsnorm_rope_table(x, w, 1e-5, c1, s1, 10000.0)
    assert torch.equal(y, ops.rmsnorm(x, w, 1e-5))
    assert torch.equal(c1, c) and torch.equal(s1, s)
