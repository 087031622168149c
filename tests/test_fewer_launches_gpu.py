"""Two launches folded into one give the bits of the two: the RMSNorm that also
writes the RoPE tables, and the pair of equal-shaped products."""
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


# one launch: up to one 32x32 tile per CU (ragged and whole tiles, one K stage,
# a K tail); two: more tiles, K under a stage, rows past the small tiles
@pytest.mark.parametrize("m,n,k", [
    (1, 8, 64), (33, 36, 72), (241, 320, 320), (256, 1024, 64), (257, 1024, 64), (31, 320, 56),
    (513, 64, 320), (1205, 320, 320)])
@pytest.mark.parametrize("split", [True, False], ids=["slices", "buffers"])
def test_linear_pair(m, n, k, split):
    from smolvla import ops
    if split:       # column slices of one buffer, as the prefix K/V cache holds them
        ld = (k + 7) // 8 * 8
        ab = _rand(m, 2 * ld, seed=3)
        a0, a1 = ab[:, :k], ab[:, ld:ld + k]
    else:
        a0, a1 = _rand(m, k, seed=3), _rand(m, k, seed=4)
    w0, w1 = _rand(n, k, seed=5, scale=0.1), _rand(n, k, seed=6, scale=0.1)
    c0, c1 = ops.linear_pair(a0, w0, a1, w1)
    assert torch.equal(c0, ops.linear(a0, w0)) and torch.equal(c1, ops.linear(a1, w1))


def test_linear_pair_of_unequal_shapes():
    from smolvla import ops
    a0, a1, w0, w1 = _rand(50, 320), _rand(60, 320), _rand(320, 320, seed=1), _rand(64, 320, seed=2)
    c0, c1 = ops.linear_pair(a0, w0, a1, w1)
    assert torch.equal(c0, ops.linear(a0, w0)) and torch.equal(c1, ops.linear(a1, w1))
