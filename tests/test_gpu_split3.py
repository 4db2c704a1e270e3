"""fp32 products made of bf16 parts: the streaming kernel's tiles and the pairs kernel against 64-bit sums, and the repeat on the fp32 units where
the parts cannot stand for a value (infinities, NaN, values that round to an infinity, values under 2^-110)."""
import pytest
import torch

from flexgemm_amd import _native as nat
from flexgemm_amd.ops.spconv import sparse_submanifold_conv3d
from flexgemm_amd.workloads import reference_test_shell
from test_gpu_nonfinite import INF, NAN, _agree, _defined, _spoil

pytestmark = pytest.mark.gpu


def _layer(monkeypatch, tile, res, ci, co, change=None, scale=1.0):
    coords = torch.from_numpy(reference_test_shell(res)).cuda()
    g = torch.Generator(device="cuda").manual_seed(ci + co)
    feats = torch.randn(len(coords), ci, generator=g, device="cuda") * scale
    weight = torch.randn(co, 3, 3, 3, ci, generator=g, device="cuda") / (27 * ci) ** 0.5
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


@pytest.mark.parametrize("tile,ci,co", TILES)
def test_small_values_keep_their_bits(monkeypatch, tile, ci, co):
    got, want, _ = _layer(monkeypatch, tile, 16, ci, co, scale=1e-34)
    assert float((got.double() - want).norm() / want.norm()) <= (27 * ci) ** 0.5 * 2.0 ** -24
