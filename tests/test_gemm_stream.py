"""The K-split line-DMA GEMMs (csrc/gemm_stream.hip): which tile an automatic
call takes (host-only query) and every tile against an fp32 product, at ragged
rows, columns and K.

Bound: the kernels accumulate bf16 products in fp32 (K <= 3072 terms: relative
error below K * 2^-24 < 2e-4 of the sum of magnitudes, far under a bf16 ulp)
and round once per rounding point, so an output is at most one bf16 ulp
(2^-7 relative at a binade's edge) from the fp32 reference rounded the same
way, plus an absolute floor of the accumulation error at outputs near zero."""

import math

import pytest
import torch

BF16 = torch.bfloat16

# (m, n, k, paired) -> tile: every configuration, on shapes the engine and the
# layers run and on ragged ones
CHOICES = [
    (1600, 720, 960, 0, 64080),      # batch-32 expert O
    (1600, 1600, 720, 1, 64160),     # batch-32 expert QKV
    (1600, 4096, 720, 1, 256128),    # batch-32 expert gate|up
    (7712, 960, 2560, 0, 256128),    # batch-32 prefix down
    (1665, 960, 2560, 0, 128064),    # five prompts of 333: down
    (1024, 768, 768, 0, 64064),      # one image: O
    (1024, 3072, 768, 0, 128096),    # one image: up
    (5103, 768, 3072, 0, 128128),    # seven images of 729 tokens: down
    (5103, 2304, 768, 0, 128192),    # seven images of 729 tokens: QKV
    (2723, 1600, 720, 1, 192128),    # an odd batch: QKV
    (1999, 768, 3000, 0, 64096),
    (241, 960, 960, 0, 0),           # batch-1 prefix: the 32-row small tiles
    (50, 4096, 720, 1, 0),           # batch-1 expert layer: the skinny tile
    (98304, 3072, 768, 0, 0),        # batch-32 ViT: the 256x256 kernel
    (300, 64, 56, 0, 0),             # under one K stage
]


@pytest.mark.parametrize("m,n,k,paired,tile", CHOICES)
def test_choice(m, n, k, paired, tile):
    from smolvla import _lib
    assert _lib.load().svla_gemm_stream_choice(m, n, k, paired) == tile


def test_choice_refuses_what_the_gemm_refuses():
    from smolvla import _lib
    for bad in ((0, 64, 64, 0), (8, 60, 64, 0), (8, 64, 60, 0), (8, 96, 64, 1), (8, 64, 0, 0)):
        assert _lib.load().svla_gemm_stream_choice(*bad) == -22


def _close(got, want, *through):
    """``through``: the rounded intermediates; one that rounds the other way
    (its fp32 sum taken in another order) moves the output by its own ulp."""
    got, want = got.float().cpu(), want.float()
    tol = 2e-3 * want.abs().mean()
    for t in (want, *through):
        tol = tol + 2 ** -7 * t.abs()
    bad = (got - want).abs() > tol
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} off, " \
                          f"max {(got - want).abs().max().item():.3e}"


# one shape per tile (rows and columns off the tile, K off the 64-deep stage),
# and the smallest problem: one tile, one stage
RAGGED = [(1601, 728, 968), (1590, 1608, 712), (1601, 4104, 720), (1665, 968, 2552),
          (1021, 776, 776), (1021, 3064, 760), (5103, 776, 3064), (5100, 2312, 776),
          (2723, 1608, 712), (1999, 776, 3000), (520, 64, 64), (513, 24, 72)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", RAGGED)
def test_plain_epilogues(m, n, k):
    """bias, scale, GELU / SiLU and an in-place residual; A and W are strided
    views whose padding is NaN (nothing past K may be read into a product)."""
    from smolvla import _lib, ops
    assert _lib.load().svla_gemm_stream_choice(m, n, k, 0) > 0
    g = torch.Generator().manual_seed(m + n + k)
    ld = (k + 63) // 64 * 64 + 8
    a = torch.full((m, ld), float("nan"), dtype=BF16)
    w = torch.full((n, ld), float("nan"), dtype=BF16)
    a[:, :k] = torch.randn(m, k, generator=g).to(BF16)
    w[:, :k] = (torch.randn(n, k, generator=g) * 0.05).to(BF16)
    b = (torch.randn(n, generator=g) * 0.5).to(BF16)
    r = torch.randn(m, n, generator=g).to(BF16)
    A, W, B = a.cuda()[:, :k], w.cuda()[:, :k], b.cuda()
    y = (a[:, :k].float() @ w[:, :k].float().t())
    _close(ops.linear(A, W, bias=B, alpha=0.5), (0.5 * y + b.float()).to(BF16))
    h = (y + b.float()).to(BF16).float()
    _close(ops.linear(A, W, bias=B, act="gelu_tanh"),
           torch.nn.functional.gelu(h, approximate="tanh").to(BF16), h)
    _close(ops.linear(A, W, bias_f32=B.float(), act="silu"),
           torch.nn.functional.silu(h).to(BF16), h)
    x = r.cuda()
    ops.linear(A, W, bias=B, res=x, out=x)
    _close(x, (h + r.float()).to(BF16), h)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1590, 1600, 712), (1601, 960, 720), (1601, 4096, 720),
                                   (2723, 1600, 720), (1665, 1600, 968), (513, 1600, 72),
                                   (700, 5120, 960)])
def test_paired_epilogues(m, n, k):
    """RoPE (with remainders; V columns as projected, their remainders
    untouched) and SiLU(gate) * up, tiles that start inside a 64-column pair
    block included."""
    from smolvla import _lib, ops
    assert _lib.load().svla_gemm_stream_choice(m, n, k, 1) > 0
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(BF16)
    w = (torch.randn(k, n, generator=g) * 0.05).to(BF16)
    proj = (a.float() @ w.float()).to(BF16).float()
    L, rot = 37, n - 320
    cos_t, sin_t = ops.rope_table(L, 64, 1e5)
    lo = torch.full((m, n), 7.0, dtype=BF16, device="cuda")
    hi = ops.linear_rope(a.cuda(), ops.pack_weight(w.cuda()), rot, L, cos_t, sin_t, out_lo=lo)
    pos = torch.arange(m) % L
    c, s = cos_t.cpu()[pos][:, None], sin_t.cpu()[pos][:, None]
    x = proj.view(m, n // 64, 64)
    want = torch.cat([x[..., :32] * c - x[..., 32:] * s, x[..., 32:] * c + x[..., :32] * s],
                     -1).reshape(m, n)
    want[:, rot:] = proj[:, rot:]
    # a projection that rounds the other way is one ulp (<= 2^-7 of it) off and
    # moves both members of its rotated pair by up to that; hi itself rounds
    # by half an ulp: 1.5 * 2^-7 of the pair's larger member
    scale = x.abs().amax(-1, keepdim=True).expand(-1, -1, 64).reshape(m, n)
    got = hi.float().cpu()
    worst = ((got - want).abs() / (2 ** -7 * scale + 1e-6)).max().item()
    assert worst <= 1.5, worst
    got[:, :rot] += lo.float().cpu()[:, :rot]
    exact = ((got - want).abs() <= 2 ** -14 * scale + 1e-6).float().mean().item()
    assert exact > 0.99, exact                # all but the projections that round the other way
    assert (lo.cpu()[:, rot:] == 7.0).all()
    # SiLU(gate) * up from the same weight's halves
    wg, wu = w[:, :n // 2].contiguous(), w[:, n // 2:].contiguous()
    got = ops.linear_silu_mul(a.cuda(), ops.pack_gate_up(wg.cuda(), wu.cuda()))
    gate = torch.nn.functional.silu(proj[:, :n // 2]).to(BF16).float()
    up = proj[:, n // 2:]
    _close(got, (gate * up).to(BF16), proj[:, :n // 2] * up, up * gate)
    assert math.isfinite(got.float().abs().max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("n,grid,hidden,scale,n_out", [
    (1, 32, 768, 4, 960), (3, 32, 768, 4, 960), (5, 32, 768, 4, 960), (9, 32, 768, 4, 960),
    (17, 32, 768, 4, 960), (33, 32, 768, 4, 960), (2, 24, 200, 3, 72), (5, 8, 104, 2, 968)])
def test_connector(n, grid, hidden, scale, n_out):
    """Pixel-shuffle gather, unsplit and with K split over workgroups, into
    plain rows and into each sample's slot of a larger buffer (whose other
    rows stay as they were)."""
    from smolvla import ops
    g = torch.Generator().manual_seed(n * grid + hidden)
    x = torch.randn(n, grid * grid, hidden, generator=g).to(BF16)
    K, per = hidden * scale * scale, (grid // scale) ** 2
    w = (torch.randn(K, n_out, generator=g) * 0.05).to(BF16)
    t = x.view(n, grid // scale, scale, grid // scale, scale, hidden).permute(0, 1, 3, 2, 4, 5)
    want = (t.reshape(n * per, K).float() @ w.float()).to(BF16)
    wp = ops.pack_weight(w.cuda())
    _close(ops.connector(x.cuda(), wp, scale), want)
    buf = torch.full((n * (per + 9), n_out), 3.0, dtype=BF16, device="cuda")
    ops.connector(x.cuda(), wp, scale, out=buf, rows_per_sample=per, sample_stride=per + 9)
    got = buf.cpu().view(n, per + 9, n_out)
    _close(got[:, :per].reshape(n * per, n_out), want)
    assert (got[:, per:] == 3.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n,chans,image,patch,embed", [
    (1, 3, 512, 16, 768), (2, 3, 512, 16, 768), (7, 3, 512, 16, 768), (3, 1, 72, 8, 72),
    (2, 3, 120, 24, 200),
    # short K: every tile that such a gather chooses, ragged rows and columns
    (1, 3, 512, 8, 776), (5, 3, 520, 8, 776), (24, 1, 224, 8, 200), (52, 1, 224, 8, 392)])
@pytest.mark.parametrize("pos", [True, False])
def test_patch_embed(n, chans, image, patch, embed, pos):
    from smolvla import ops
    g = torch.Generator().manual_seed(n * image + embed)
    x = (torch.rand(n, chans, image, image, generator=g) * 2 - 1).to(BF16)
    w = (torch.randn(embed, chans, patch, patch, generator=g) * 0.05).to(BF16)
    b = torch.randn(embed, generator=g).to(BF16)
    G = image // patch
    table = torch.randn(G * G, embed, generator=g).to(BF16) if pos else None
    y = torch.nn.functional.conv2d(x.float(), w.float(), b.float(), stride=patch)
    y = y.flatten(2).transpose(1, 2).to(BF16).float()
    want = (y + table.float()).to(BF16) if pos else y.to(BF16)
    got = ops.patch_embed(x.cuda(), w.reshape(embed, -1).cuda(), b.cuda(),
                          table.cuda() if pos else None, patch)
    _close(got.view(n, G * G, embed), want, y)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5, 9, 17])
def test_connector_past_256_rows_runs_unsplit(n):
    """The K split's workspace is one per device: gathers of more than 256 rows
    leave it alone, so they may overlap on two streams (same bits as with the
    split turned off)."""
    from smolvla import _lib, ops
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, 1024, 768, generator=g).to(BF16).cuda()
    w = (torch.randn(960, 12288, generator=g) * 0.05).to(BF16).cuda()
    lib = _lib.load()
    got = ops.connector(x, w, 4)
    assert lib.svla_gemm_set_split(1) == 0
    try:
        want = ops.connector(x, w, 4)
    finally:
        lib.svla_gemm_set_split(-1)
    assert torch.equal(got, want)


@pytest.fixture
def force_split():
    from smolvla import _lib
    lib = _lib.load()

    def force(n):
        assert lib.svla_gemm_set_split(n) == 0
    yield force
    lib.svla_gemm_set_split(-1)


@pytest.mark.parametrize("m,n,k", [(64, 960, 12288), (192, 960, 12288), (256, 72, 2048)])
def test_gathers_obey_a_forced_split(force_split, m, n, k):
    from smolvla import _lib
    choice = _lib.load().svla_gemm_gather_choice
    assert choice(m, n, k) // 1000000 > 1                 # split by themselves
    for z in (1, 2, 3, 5, 12, 13, 22):
        force_split(z)
        assert choice(m, n, k) // 1000000 == z


def test_forced_gather_splits_end_at_k_and_at_the_workspace(force_split):
    from smolvla import _lib
    choice = _lib.load().svla_gemm_gather_choice
    force_split(64)
    assert choice(64, 72, 200) // 1000000 == 4            # a 64-deep stage each
    # 2^22 floats of partial tiles: 22 times 192 x 960
    assert choice(192, 960, 12288) // 1000000 == 22
    assert choice(320, 960, 12288) // 1000000 == 1        # more rows never split


@pytest.mark.parametrize("m,n,k,tile", [
    (2048, 960, 128, 64064),         # 480 64x64 tiles
    (4096, 768, 192, 128192),        # 768: one 512-pixel image in 8-pixel patches
    (49152, 768, 192, 128192), (196608, 768, 192, 256128), (196608, 768, 64, 256128),
    (18816, 200, 64, 192128), (9408, 384, 192, 128192), (4704, 200, 64, 64064),
    (4096, 768, 256, 64096),         # four stages: the cost model alone
])
def test_gathers_of_short_k(m, n, k, tile):
    """Under four K stages no more than two 64x64 tiles per CU: past that their
    fixed costs add up (12 images of 8-pixel patches 76 us, 52 on 128x192)."""
    from smolvla import _lib
    assert _lib.load().svla_gemm_gather_choice(m, n, k) == 1000000 + tile


def test_dense_skinny_problems_obey_a_forced_split(force_split):
    """A count over 1 keeps them on the skinny tile, which splits; 1 does not
    need it."""
    from smolvla import _lib
    choice = _lib.load().svla_gemm_stream_choice
    auto = choice(100, 1600, 960, 1)
    assert auto > 0
    for z, want in ((4, 0), (1, auto), (-1, auto)):
        force_split(z)
        assert choice(100, 1600, 960, 1) == want


@pytest.mark.gpu
def test_connector_at_forced_splits(force_split):
    """Every count gives the product, and the counts' sums are their own."""
    from smolvla import ops
    ops.init()
    g = torch.Generator().manual_seed(4)
    x = torch.randn(3, 1024, 768, generator=g).to(BF16)
    w = (torch.randn(12288, 960, generator=g) * 0.05).to(BF16)
    t = x.view(3, 8, 4, 8, 4, 768).permute(0, 1, 3, 2, 4, 5).reshape(192, 12288)
    want = (t.float() @ w.float()).to(BF16)
    X, W = x.cuda(), ops.pack_weight(w.cuda())
    got = []
    for z in (-1, 1, 2, 3, 5, 13, 22):
        force_split(z)
        got.append(ops.connector(X, W, 4))
        _close(got[-1], want)
    assert all(not torch.equal(a, b) for a, b in zip(got[1:], got[2:]))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(100, 1600, 960), (65, 960, 720), (128, 1600, 2048)])
def test_paired_at_forced_splits(force_split, m, n, k):
    from smolvla import ops
    ops.init()
    g = torch.Generator().manual_seed(m)
    a = torch.randn(m, k, generator=g).to(BF16)
    wg, wu = ((torch.randn(k, n // 2, generator=g) * 0.05).to(BF16) for _ in range(2))
    W = ops.pack_gate_up(wg.cuda(), wu.cuda())
    gate, up = ((a.float() @ w.float()).to(BF16).float() for w in (wg, wu))
    s = torch.nn.functional.silu(gate).to(BF16).float()
    for z in (-1, 1, 2, 4):
        force_split(z)
        _close(ops.linear_silu_mul(a.cuda(), W), (s * up).to(BF16), gate * up, up * s)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,skinny", [
    (65, 1600, 720, True), (128, 960, 720, True), (100, 2048, 264, True), (65, 960, 1480, True),
    (100, 2112, 720, False), (100, 960, 200, True), (128, 1536, 72, True),
    (128, 2048, 200, False), (100, 960, 1544, False)])
def test_paired_rows_off_lines_keep_the_skinny_tile(m, n, k, skinny):
    """Packed rows (65 to 128 of them) that do not all start on 128-byte lines
    give the bits of the 16-column skinny tile, past its range those of rows on
    lines, which run on the K-split tile."""
    from smolvla import _lib, ops
    lib = _lib.load()
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g).to(BF16).cuda()
    lined = torch.empty(m, (k + 63) // 64 * 64, dtype=BF16, device="cuda")[:, :k].copy_(a)
    w = ops.pack_weight((torch.randn(k, n, generator=g) * 0.05).to(BF16).cuda())
    cos_t, sin_t = ops.rope_table(m, 64, 1e5)

    def run(x):
        lo = torch.zeros(m, n, dtype=BF16, device="cuda")
        return torch.stack([ops.linear_rope(x, w, n, m, cos_t, sin_t, out_lo=lo), lo])

    got = run(a)
    assert lib.svla_gemm_set_tile(12 if skinny else -1) == 0
    try:
        want = run(a if skinny else lined)
    finally:
        lib.svla_gemm_set_tile(-1)
    assert torch.equal(got, want)
