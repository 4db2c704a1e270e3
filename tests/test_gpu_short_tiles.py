"""Streaming tiles of 64 and 128 rows (16-bit types): the same bits as tiles of 256 rows at the edges of tiles, slabs and rounds of items, and the
shapes that the schedule gives them."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import sparse_conv3d, sparse_submanifold_conv3d_relu
from test_gpu_wgrad_split import coords_of

TILES = [(64, 64), (64, 128), (128, 64), (128, 128), (64, 32), (128, 32)]


def _layer(monkeypatch, tile, n, side, ci, co, dtype):
    coords = coords_of(n, side, n)
    g = torch.Generator(device="cuda").manual_seed(n + ci)
    feats = torch.randn(n, ci, generator=g, device="cuda").to(dtype).requires_grad_()
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5).to(dtype).requires_grad_()
    bias = torch.randn(co, generator=g, device="cuda").to(dtype).requires_grad_()
    nat.host()                  # (takes note of the table before it is replaced)
    real = nat.table_lookup

    def lookup(kind, *a, **k):
        s = real(kind, *a, **k)
        if kind != nat.PASS_WGRAD:
            s.tile_rows, s.tile_cols, s.slab_bytes, s.splitk, s.stream = *tile, 128, 1, 1
        return s
    monkeypatch.setattr(nat, "table_lookup", lookup)
    out, cache = sparse_submanifold_conv3d_relu(feats, coords, torch.Size([1, ci, side, side, side]), weight, bias)
    out.backward(torch.randn(out.shape, generator=g, device="cuda").to(dtype))
    monkeypatch.setattr(nat, "table_lookup", real)
    return out.detach(), feats.grad, weight.grad, feats.detach(), weight.detach(), bias.detach(), cache


# one row, a band and a tile more or less one row; K and columns that end inside a slab, a piece and a tile; 1 300 tiles of 64 rows by two of columns, more than
# two workgroups a CU take in one round
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,side,ci,co", [(1, 4, 64, 64), (63, 8, 40, 72), (65, 8, 136, 40), (129, 8, 96, 200), (1000, 12, 72, 136), (83201, 96, 40, 72)])
def test_same_bits_as_the_long_tiles(monkeypatch, dtype, n, side, ci, co):
    want = _layer(monkeypatch, (256, 64), n, side, ci, co, dtype)
    for tile in TILES:
        got = _layer(monkeypatch, tile, n, side, ci, co, dtype)
        for a, b in zip(got[:3], want[:3]):
            assert torch.equal(a, b), tile
    out, _, _, feats, weight, bias, cache = want
    nmap = cache["neighbor_map"].view(torch.int32).long()
    w = weight.reshape(co, 27, ci).float()
    ref = bias.float().expand(n, co).clone()
    for v in range(27):
        have = (nmap[:, v] >= 0).nonzero()[:, 0]
        ref[have] += feats[nmap[have, v]].float() @ w[:, v].t()
    # one rounding to the type of sums of about one, added in 32 bits in another order
    unit = torch.finfo(dtype).eps
    assert bool(((out.float() - ref.relu()).abs() <= unit * ref.abs() + 27 * ci * 2.0 ** -23).all())


@pytest.mark.parametrize("n,ci,co,tile", [
    (5119, 192, 192, None), (5120, 192, 192, (64, 64)), (10239, 512, 64, None), (10240, 512, 64, (64, 64)), (24575, 64, 64, None), (24576, 64, 64, (64, 64)),
    (36864, 64, 64, (64, 64)), (36865, 64, 64, (128, 64)), (262144, 64, 64, (128, 64)), (262145, 64, 64, (256, 64)), (524288, 48, 40, (128, 64)), (20574, 128, 128, (64, 128)),
    (57345, 128, 128, (256, 128)), (12288, 256, 256, (64, 128)), (12289, 256, 256, (256, 64)), (28672, 384, 96, (128, 128)), (20000, 32, 64, None),
    (32767, 64, 32, None), (32768, 64, 32, (64, 32)), (36865, 64, 32, (128, 32)), (98305, 64, 32, (256, 32)), (131071, 72, 24, (256, 32)), (131072, 72, 24, (128, 32)),
    (20479, 256, 16, None), (20480, 256, 16, (64, 32)), (262144, 128, 32, (64, 32)), (131073, 96, 64, (256, 64))])
def test_rule(n, ci, co, tile):
    s = nat.table_lookup(nat.PASS_FWD, torch.float16, n, ci, co, 27)
    got = (s.tile_rows, s.tile_cols) if s.stream else None
    if tile is None:
        assert got is None
    else:
        assert got == tile and (s.tile_rows == 256 or (s.slab_bytes, s.splitk) == (128, 1))


# 5 to 8 offsets: both directions of a layer on the same tile, whichever of its channels are more
@pytest.mark.parametrize("n,ci,co,v,small", [
    (20400, 128, 128, 8, True), (36864, 128, 128, 5, True), (36865, 128, 128, 8, False), (20400, 128, 128, 4, False), (20400, 128, 96, 7, False), (20400, 127, 128, 8, False),
    (24576, 256, 256, 8, True), (24577, 256, 256, 6, False), (12288, 384, 512, 8, True), (12289, 384, 512, 8, False), (20000, 512, 256, 7, False)])
def test_rule_of_few_offsets(n, ci, co, v, small):
    for kind in (nat.PASS_FWD, nat.PASS_DGRAD):
        s = nat.table_lookup(kind, torch.float16, n, ci, co, v)
        assert s.stream and ((s.tile_rows, s.tile_cols) == (64, 128)) == small


@pytest.mark.parametrize("n,ci,co", [(5120, 192, 192), (20574, 128, 128), (36864, 64, 64), (12288, 256, 256)])
def test_not_under_few_offsets_or_in_fp32(n, ci, co):
    for dtype, v in ((torch.float16, 4), (torch.float32, 8), (torch.float32, 27)):
        s = nat.table_lookup(nat.PASS_FWD, dtype, n, ci, co, v)
        assert not s.stream or 256 in (s.tile_rows, s.tile_cols)


# 2 x 2 x 2 and 5 x 1 x 1 under a stride of 2: the short tile that the rule chooses and 256 x 64 ones, outputs and gradients
@pytest.mark.gpu
@pytest.mark.parametrize("ks,n,side,ci,co", [((2, 2, 2), 30001, 64, 128, 128), ((5, 1, 1), 23000, 48, 136, 200), ((1, 2, 3), 24000, 56, 256, 136)])
def test_few_offsets_same_bits(monkeypatch, ks, n, side, ci, co):
    g = torch.Generator(device="cuda").manual_seed(n)
    coords, shape = coords_of(n, side, n), torch.Size([1, ci, side, side, side])
    feats = torch.randn(n, ci, generator=g, device="cuda").half().requires_grad_()
    weight = (torch.randn(co, *ks, ci, generator=g, device="cuda") / (8 * ci) ** 0.5).half().requires_grad_()
    nat.host()
    real, got, up = nat.table_lookup, [], None
    for tile in (None, (256, 64)):
        chosen = []

        def lookup(kind, dtype, rows, *a):
            s = real(kind, dtype, rows, *a)
            if kind != nat.PASS_WGRAD:
                if tile:
                    s.tile_rows, s.tile_cols, s.slab_bytes, s.splitk, s.stream = *tile, 128, 1, 1
                chosen.append((s.tile_rows, s.tile_cols))
            return s
        monkeypatch.setattr(nat, "table_lookup", lookup)
        out, _, _ = sparse_conv3d(feats, coords, shape, weight, None, None, None, (2, 2, 2))
        up = torch.randn(out.shape, generator=g, device="cuda").half() if up is None else up
        got.append((out.detach(), *torch.autograd.grad(out, [feats, weight], up)))
        assert set(chosen) == {tile or (64, 128)}           # (both directions: the tiled kernel adds in another order)
    for a, b in zip(*got):
        assert torch.equal(a, b)


# rows past the streaming kernel's 32-bit byte offsets: the tiled kernel, on a tile that it has
@pytest.mark.gpu
def test_operands_past_32_bit_offsets():
    n, side, ci, co = 131072, 64, 16384, 40
    s = nat.table_lookup(nat.PASS_FWD, torch.float16, n, ci, co, 27)
    assert s.stream and s.tile_rows < 256 and n * ci * 2 > 0xFF000000
    coords = coords_of(n, side, 3)
    g = torch.Generator(device="cuda").manual_seed(3)
    feats = torch.empty(n, ci, dtype=torch.float16, device="cuda").uniform_(-1, 1, generator=g)
    weight = (torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5).half()
    with torch.no_grad():
        out, cache = sparse_submanifold_conv3d_relu(feats, coords, torch.Size([1, ci, side, side, side]), weight)
    nmap, w = cache["neighbor_map"].view(torch.int32).long(), weight.reshape(co, 27, ci).float()
    for row in (0, 63, 70000, n - 1):
        have = (nmap[row] >= 0).nonzero()[:, 0]
        ref = (feats[nmap[row, have]].float()[:, None] * w[:, have].transpose(0, 1)).sum((0, 2))
        # one rounding to 16 bits; sums of about one of 27 ci products in 32 bits, in another order
        assert bool(((out[row].float() - ref.relu()).abs() <= 2.0 ** -10 * ref.abs() + (27 * ci) ** 0.5 * 2.0 ** -22).all())
