"""fp32 products made of bf16 parts: the streaming kernel's tiles, the pairs kernel and the weight gradient against 64-bit sums, and the repeat on
the fp32 units where the parts cannot stand for a value or a sum (infinities, NaN, values from 2^104 on, sums past 2^80 or under 2^-127)."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import SubMConv3dFunction, sparse_submanifold_conv3d
from flexgemm_amd.workloads import reference_test_shell
from test_gpu_nonfinite import INF, NAN, _agree, _defined, _spoil
from test_gpu_wgrad_split import coords_of

pytestmark = pytest.mark.gpu


def _layer(monkeypatch, tile, res, ci, co, change=None, scale=1.0, weight_scale=1.0):
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    g = torch.Generator(device="cuda").manual_seed(ci + co)
    feats = torch.randn(len(coords), ci, generator=g, device="cuda") * scale
    weight = torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5 * weight_scale
    if change is not None:
        change(feats, weight)
    nat.host()                  # (takes note of the table before it is replaced)
    if tile is not None:
        real = nat.table_lookup

        def lookup(kind, *a, **k):
            s = real(kind, *a, **k)
            if kind != nat.PASS_WGRAD:
                s.tile_rows, s.tile_cols, s.slab_bytes = tile
                s.splitk, s.stream = 1, 1
            return s
        monkeypatch.setattr(nat, "table_lookup", lookup)
    with torch.no_grad():
        out, cache = sparse_submanifold_conv3d(feats, coords, torch.Size([1, ci, res, res, res]), weight)
    assert (tile is None) == ("_pair_plan" in cache.__dict__)
    return out, _defined(feats, weight.reshape(co, 27, ci), cache.neighbor_map.view(torch.int32), 0), feats


# every streaming tile that the fp32 rule answers with, the pairs kernel's two (None: 96 and 64 columns); channels that end inside a
# slab, inside 16 values of K and inside a tile; rows that end inside a tile
TILES = [((128, 256, 128), 40, 136), ((256, 128, 128), 68, 72), ((256, 64, 64), 20, 36), ((256, 64, 128), 32, 40), ((256, 32, 64), 36, 24), (None, 68, 84), (None, 64, 36)]


@pytest.mark.parametrize("tile,ci,co", TILES)
def test_as_near_as_fp32_sums(monkeypatch, tile, ci, co):
    got, want, _ = _layer(monkeypatch, tile, 16, ci, co)
    # 27 ci products with a rounding each of sums of about one, which do not all point the same way
    assert float((got.double() - want).norm() / want.norm()) <= (27 * ci) ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("tile,ci,co", TILES)
def test_what_three_parts_cannot_stand_for(monkeypatch, tile, ci, co):
    def change(feats, weight):
        _spoil(feats, [(7, 3, INF), (31, ci - 1, -INF), (60, 0, NAN), (61, 5, INF), (61, 6, -INF), (200, 2, 3.4e38)])
        if tile is None:            # (masked tiles multiply the zeros of missing neighbors by every weight)
            weight[1, 1, 1, 1, 2], weight[co - 1, 2, 0, 1, ci - 1] = INF, NAN

    got, want, feats = _layer(monkeypatch, tile, 16, ci, co, change)
    fine = want.isfinite() & (want.abs() < 1e30)
    assert fine.any() and (want.abs() > 1e30).any()
    _agree(torch.where(fine | ~want.isfinite(), got.double(), want), want, 2.0 ** -23, 27 * ci * 2.0 ** -24 * 64)
    # 3.4e38: the sum it is in, as fp32 has it
    huge = want.isfinite() & ~fine
    assert bool(((got.double() - want).abs()[huge] <= 1e-6 * want.abs()[huge]).all())


@pytest.mark.parametrize("tile,ci,co", [t for t in TILES if t[0] is not None])
def test_the_repeat_leaves_out_what_the_product_leaves_out(monkeypatch, tile, ci, co):
    """An infinite weight at one offset: 32 rows of the order none of which has it are not multiplied by it, the second time either."""
    plain, _, _ = _layer(monkeypatch, tile, 16, ci, co)
    coords = torch.from_numpy(reference_test_shell(16)).cuda()
    cache = SubMConv3dFunction._compute_neighbor_cache(coords, torch.Size([1, ci, 16, 16, 16]), (3, 3, 3), (1, 1, 1), False)
    order = cache.sorted_idx
    has = cache.neighbor_map.view(torch.int32)[order] >= 0
    has = torch.cat([has, has.new_zeros((-len(has)) % 64, 27)]).view(-1, 32, 27).any(1)                  # [bands of 32 rows, offsets]
    # an offset that one band of a wavefront's 64 rows has and the other has not
    v = int((has[::2] != has[1::2]).any(0).nonzero()[0])

    def change(feats, weight):
        weight.view(co, 27, ci)[:, v] = INF
    got, _, _ = _layer(monkeypatch, tile, 16, ci, co, change)
    without = torch.zeros(len(order), dtype=torch.bool, device="cuda")
    without[order] = ~has[:, v].repeat_interleave(32)[:len(order)]
    assert without.any() and not got[~without].isfinite().any() and got[without].isfinite().all()
    assert float((got[without] - plain[without]).norm() / plain[without].norm()) <= 2 * (27 * ci) ** 0.5 * 2.0 ** -24


# 64 columns: slabs of 128 bytes where a row is whole ones, of 64 where one would be part empty
@pytest.mark.parametrize("ci,slab", [(32, 128), (36, 64), (64, 128), (80, 64), (96, 128), (128, 128)])
def test_slabs_of_64_columns(monkeypatch, ci, slab):
    s = nat.table_lookup(nat.PASS_FWD, torch.float32, 166232, ci, 64, 27)
    assert (s.tile_rows, s.tile_cols, s.slab_bytes, s.stream) == (256, 64, slab, 1)
    got, want, _ = _layer(monkeypatch, (256, 64, slab), 16, ci, 64)
    # (as above)
    assert float((got.double() - want).norm() / want.norm()) <= (27 * ci) ** 0.5 * 2.0 ** -24


# Long sums: what the matrix unit drops of every addition points downwards, and must cancel.  Six additions for 16 values of K, off by 2^-24 of the running
# sum or less in the mean of their squares, whose own square is half of the last one's on average; and errors that point neither way have a mean
# within six standard deviations of that of as many independent ones.
@pytest.mark.parametrize("tile,ci,co", [((128, 256, 128), 512, 136), ((256, 128, 128), 1024, 128), ((256, 64, 64), 512, 64), ((256, 64, 128), 1024, 64),
                                        ((256, 32, 64), 512, 96), (None, 512, 96), (None, 1024, 64)])
@pytest.mark.parametrize("positive", [False, True])
def test_long_sums_point_neither_way(monkeypatch, tile, ci, co, positive):
    got, want, _ = _layer(monkeypatch, tile, 16, ci, co, (lambda feats, weight: feats.abs_()) if positive else None)
    error = got.double() - want
    assert float(error.norm() / want.norm()) <= (27 * ci * 6 / 16 / 2) ** 0.5 * 2.0 ** -24
    assert abs(float(error.mean())) <= 6 * float(error.norm()) / error.numel()


@pytest.mark.parametrize("tile,ci,co", TILES)
def test_small_values_keep_their_bits(monkeypatch, tile, ci, co):
    got, want, _ = _layer(monkeypatch, tile, 16, ci, co, scale=1e-34)
    assert float((got.double() - want).norm() / want.norm()) <= (27 * ci) ** 0.5 * 2.0 ** -24


# (log2) features and weights about: small ones whose products are small; small against large, whose sums a guard on sums alone lets through: parts that fall
# below bf16's normal numbers, then below all of them (subnormal values); sums past 2^80 and values past 2^104, which are multiplied again
MAGNITUDES = [(-113, 0), (-116, 30), (-120, 40), (-126, 60), (-136, 60), (-142, 100), (30, -110), (50, -120), (60, -130), (60, 30), (110, -60), (-120, 115)]


@pytest.mark.parametrize("tile,ci,co", TILES)
@pytest.mark.parametrize("of_feats,of_weight", MAGNITUDES)
def test_magnitudes_apart(monkeypatch, tile, ci, co, of_feats, of_weight):
    got, want, _ = _layer(monkeypatch, tile, 16, ci, co, scale=2.0 ** of_feats, weight_scale=2.0 ** of_weight)
    assert float(want.norm()) > 0
    # as of values about one: a power of two more or less changes no rounding (the operands are taken as they came out, subnormal ones included)
    assert float((got.double() - want).norm() / want.norm()) <= (27 * ci) ** 0.5 * 2.0 ** -24


def _weight_grad(n, ci, co, scale=1.0, change=None, grad_scale=1.0):
    """The weight gradient, the same in 64 bits, and each sum's magnitude, of n voxels in a cube two thirds full."""
    side = round((1.5 * n) ** (1 / 3)) + 1
    cache = SubMConv3dFunction._compute_neighbor_cache(coords_of(n, side, n), torch.Size([1, ci, side, side, side]), (3, 3, 3), (1, 1, 1), True)
    g = torch.Generator(device="cuda").manual_seed(n + ci)
    feats, grad = torch.randn(n, ci, generator=g, device="cuda") * scale, torch.randn(n, co, generator=g, device="cuda") * grad_scale
    if change is not None:
        change(feats, grad)
    got = nat.host().wgrad(grad, feats, cache, 27, False, -1)[0].view(co, 27, ci)
    nmap = cache["neighbor_map"].view(torch.int32).cpu().long()
    f, u = feats.cpu().double(), grad.cpu().double()
    want, size = torch.zeros(co, 27, ci, dtype=torch.double), torch.zeros(co, 27, ci, dtype=torch.double)
    for v in range(27):
        r = (nmap[:, v] >= 0).nonzero()[:, 0]
        want[:, v], size[:, v] = u[r].T @ f[nmap[r, v]], u[r].abs().T @ f[nmap[r, v]].abs()
    return got.cpu().double(), want, size


# both tiles, channels that end inside one, segments of several folds and of less than half a step, two tiles, more than sixteen; rows on both sides
# of where the fp32 units end
SPLIT_GRADS = [(9215, 96, 96), (9216, 96, 96), (12001, 96, 92), (14335, 64, 64), (14336, 64, 64), (20000, 52, 60), (8000, 112, 48), (3001, 192, 180),
               (1024, 320, 260), (9000, 32, 64)]


@pytest.mark.parametrize("n,ci,co", SPLIT_GRADS)
@pytest.mark.parametrize("scale", [1.0, 1e-34])
def test_weight_gradient(n, ci, co, scale):
    got, want, size = _weight_grad(n, ci, co, scale)
    # k products summed in any order: within k units of the sum of their magnitudes; sums of random signs, on the whole, within sqrt(k) of their own size
    assert bool(((got - want).abs() <= n * 2.0 ** -23 * size + 2.0 ** -149 * n).all())
    assert float((got - want).norm() / want.norm()) <= n ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("n,ci,co", [(9216, 96, 96), (14336, 64, 64), (3001, 192, 180)])
@pytest.mark.parametrize("of_feats,of_grad", MAGNITUDES)
def test_weight_gradient_of_magnitudes_apart(n, ci, co, of_feats, of_grad):
    got, want, size = _weight_grad(n, ci, co, scale=2.0 ** of_feats, grad_scale=2.0 ** of_grad)
    assert float(want.norm()) > 0 and bool(((got - want).abs() <= n * 2.0 ** -23 * size).all())
    assert float((got - want).norm() / want.norm()) <= n ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("n,ci,co", [(9216, 96, 96), (14336, 64, 64), (3001, 192, 180)])
def test_weight_gradient_of_what_three_parts_cannot_stand_for(n, ci, co):
    def change(feats, grad):
        _spoil(feats, [(7, 3, INF), (n - 31, ci - 1, -INF), (60, 0, NAN), (200, 2, 3.4e38)])
        _spoil(grad, [(8, 1, INF), (n - 5, co - 1, NAN), (300, 5, -INF)])
    got, want, size = _weight_grad(n, ci, co, change=change)
    fine = want.isfinite() & (size < 1e30)
    assert fine.any() and (~want.isfinite()).any() and (size[want.isfinite()] > 1e30).any()
    assert bool(((got - want).abs() <= n * 2.0 ** -23 * size)[fine].all())
    odd = ~want.isfinite()
    assert not got[odd].isfinite().any()
    odd[:, :, 2] = False            # (3.4e38 times more than one is an infinity of either sign in 32 bits)
    assert torch.equal(got[odd].isnan(), want[odd].isnan()) and torch.equal(got[odd].nan_to_num(0), want[odd].nan_to_num(0))
    huge = want.isfinite() & ~fine & (want.abs() < 3e38)
    assert bool(((got - want).abs() <= n * 2.0 ** -23 * size)[huge].all())
