"""Neighbor caches through the index over the grid's cells, and the sorts of the cache, against the CPU oracle (bit-exact)."""
import ctypes as C
import sys

import numpy as np
import pytest
import torch

import flex_gemm
from flex_gemm.ops.spconv import SparseConv3dFunction, SubMConv3dFunction, sparse_submanifold_conv3d
from flexgemm_amd import _native as nat
from flexgemm_amd.workloads import reference_test_shell
from oracle import explicit_gemm as eg
from oracle import neighbor as nb
from oracle import sparse_conv as sc

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def grid_builder():
    flex_gemm.ops.spconv.set_neighbor_map_builder("grid")
    yield
    flex_gemm.ops.spconv.set_neighbor_map_builder("auto")


def _say(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


def _np(t):
    return t.cpu().view(torch.int32).numpy().view(np.uint32) if t.dtype == torch.uint32 else t.cpu().numpy()


def _voxels(dims, n, seed, order):
    """n distinct voxels of a (B, W, H, D) grid, clustered so that most have neighbors, in scan or random order."""
    rng = np.random.default_rng(seed)
    cells = np.unique(rng.integers(0, max(int(np.prod(dims)) // 40, 1), 2 * n) + int(np.prod(dims)) // 2)[:n]
    coords = np.stack(np.unravel_index(cells % int(np.prod(dims)), dims), 1).astype(np.int32)
    coords = np.unique(coords, axis=0)
    return coords if order == "scan" else coords[rng.permutation(len(coords))]


# both forms of the index: a word per cell up to 2^23 cells, a bit per cell beyond (203^3 and 204^3 lie on either side);
# long rows, cells that are no multiple of 128, fewer rows than a workgroup takes and one more than it takes
@pytest.mark.parametrize("dims,n", [((1, 203, 203, 203), 5000), ((1, 204, 204, 204), 5000), ((3, 5, 7, 90001), 4097), ((2, 1, 3, 2000003), 65),
                                    ((1, 300, 300, 300), 1), ((4, 11, 9, 13), 64)])
@pytest.mark.parametrize("order", ["scan", "shuffled"])
@pytest.mark.parametrize("dil", [(1, 1, 1), (2, 1, 3)])
def test_subm_cache(gpu_device, dims, n, order, dil):
    _say(f"grid cache dims={dims} n={n} {order} dilation={dil}")
    coords = _voxels(dims, n, 7, order)
    shape = torch.Size([dims[0], 0, *dims[1:]])
    cache = SubMConv3dFunction._compute_neighbor_cache(torch.from_numpy(coords).to(gpu_device), shape, (3, 3, 3), dil, True)
    ref = nb.neighbor_cache(coords, tuple(shape), (3, 3, 3), dil, needs_grad=True, blocks=(64,))
    for field in ("neighbor_map", "gray_code", "sorted_idx", "valid_signal_seg", "valid_signal_i", "valid_signal_o"):
        assert np.array_equal(_np(getattr(cache, field)), ref[field]), field


@pytest.mark.parametrize("res", [32, 210])
def test_subm_repeated_voxels_are_found_under_their_smallest_row(gpu_device, res):
    _say(f"grid map with repeated voxels res={res}")
    rng = np.random.default_rng(res)
    base = reference_test_shell(32)
    coords = np.concatenate([base, base[rng.choice(len(base), 300, replace=False)], base[:7], base[:7]])[rng.permutation(len(base) + 314)]
    cache = SubMConv3dFunction._compute_neighbor_cache(torch.from_numpy(coords).to(gpu_device), torch.Size([1, 0, res, res, res]), (3, 3, 3),
                                                       (1, 1, 1), False)
    first = {}
    for i, c in enumerate(map(tuple, coords)):
        first.setdefault(c, i)
    want = np.full((len(coords), 27), 0xFFFFFFFF, np.uint32)
    for i, (b, x, y, z) in enumerate(coords):
        for v in range(27):
            want[i, v] = first.get((b, x + v // 9 - 1, y + v // 3 % 3 - 1, z + v % 3 - 1), 0xFFFFFFFF)
        want[i, 13] = i
    assert np.array_equal(_np(cache.neighbor_map), want)


@pytest.mark.parametrize("dims,n", [((2, 40, 41, 39), 3000), ((1, 260, 250, 261), 4001), ((3, 5, 7, 90001), 700)])
@pytest.mark.parametrize("geom", [((2, 2, 2), (2, 2, 2), (0, 0, 0), (1, 1, 1)), ((3, 3, 3), (2, 1, 3), (1, 0, 2), (1, 2, 1)),
                                  ((1, 1, 5), (1, 1, 2), (0, 0, 1), (1, 1, 1))])
def test_generic_convolution(gpu_device, dims, n, geom):
    _say(f"grid conv dims={dims} n={n} geom={geom}")
    coords = _voxels(dims, n, 3, "shuffled")
    shape = torch.Size([dims[0], 0, *dims[1:]])
    dev_coords = torch.from_numpy(coords).to(gpu_device)
    out = SparseConv3dFunction._get_output_coords(dev_coords, shape, *geom)
    want = sc.output_coords(coords, tuple(shape), *geom)
    assert np.array_equal(out.cpu().numpy(), want)
    if len(want) == 0:
        return
    cache = SparseConv3dFunction._compute_neighbor_cache(dev_coords, out, shape, *geom, True)
    fwd, bwd = sc.neighbor_maps(coords, want, tuple(shape), *geom)
    assert np.array_equal(_np(cache.neighbor_map), fwd)
    assert np.array_equal(_np(cache.neighbor_map_bwd), bwd)
    gray, binary = nb.gray_binary(fwd)
    assert np.array_equal(_np(cache.gray_code), gray)
    assert np.array_equal(_np(cache.sorted_idx), nb.sorted_idx_canonical(binary))
    if any(s != 1 for s in geom[1]):
        gray, binary = nb.gray_binary(bwd)
        assert np.array_equal(_np(cache.gray_code_bwd), gray)
        assert np.array_equal(_np(cache.sorted_idx_bwd), nb.sorted_idx_canonical(binary))


# the rank sort's last size and the radix sort's first, the switch to long tiles, partial tiles; all code bits in use and few
@pytest.mark.parametrize("n", [1, 63, 64, 65, 16384, 16385, 786431, 786432, 1000003])
@pytest.mark.parametrize("volume,distinct", [(27, 3000), (32, 1 << 32), (3, 8)])
def test_mask_sort(gpu_device, n, volume, distinct):
    _say(f"mask sort n={n} volume={volume} distinct={distinct}")
    gen = torch.Generator(device=gpu_device).manual_seed(n)
    lo, hi = (-(1 << 31), (1 << 31) - 1) if volume == 32 else (0, 1 << volume)
    keys = torch.randint(lo, hi, (min(distinct, n),), generator=gen, device=gpu_device, dtype=torch.int64).to(torch.int32)
    keys = keys[torch.randint(0, keys.shape[0], (n,), generator=gen, device=gpu_device)].contiguous()
    order = torch.empty((n,), dtype=torch.int64, device=gpu_device)
    L = nat.lib()
    ws = nat.workspace(L.fgx_sort_workspace_bytes(nat.sz(n)), gpu_device)
    nat.check(L.fgx_sort_by_code(nat.ptr(keys), nat.sz(n), C.c_int(volume), nat.ptr(order), nat.ptr(ws), nat.sz(ws.numel()), nat.stream()))
    assert np.array_equal(order.cpu().numpy(), np.argsort(keys.cpu().numpy(), kind="stable"))


# the index's row order as the narrow layers' plan: first product of a fresh cache, rows in scan and random order, with and without
# voxels given twice, a grid whose columns need no padding and one whose do, a last chunk that is not full
@pytest.mark.parametrize("res,order,twice", [(256, "scan", 0), (256, "shuffled", 0), (205, "shuffled", 90), (230, "scan", 1)])
def test_narrow_layer_on_a_fresh_grid_cache(gpu_device, res, order, twice):
    _say(f"narrow layer on a fresh grid cache res={res} {order} twice={twice}")
    rng = np.random.default_rng(res)
    coords = reference_test_shell(96) + np.array([0, 50, 3, 101], np.int32)
    coords = np.concatenate([coords, coords[:twice]])
    if order == "shuffled":
        coords = coords[rng.permutation(len(coords))]
    n, c = len(coords), 16
    gen = torch.Generator().manual_seed(res)
    feats, grad = torch.randn(n, c, generator=gen).half(), torch.randn(n, c, generator=gen).half()
    weight = (torch.randn(c, 3, 3, 3, c, generator=gen) / (27 * c) ** 0.5).half()
    dev = gpu_device
    f, w = feats.to(dev).requires_grad_(True), weight.to(dev).requires_grad_(True)
    out, cache = sparse_submanifold_conv3d(f, torch.from_numpy(coords).to(dev), torch.Size([1, c, res, res, res]), w)
    out.backward(grad.to(dev))
    assert np.array_equal(np.sort(_np(cache["_cell_walk"])), np.arange(n)) and hasattr(cache, "_narrow_plan_buf")
    nmap = cache.neighbor_map.cpu().view(torch.int32)
    ref_gi, ref_gw, _ = eg.backward(grad.double(), feats.double(), nmap, weight.double())
    for got, ref in ((out, eg.forward(feats.double(), nmap, weight.double())), (f.grad, ref_gi), (w.grad, ref_gw)):
        assert eg.max_rel_err(got.detach().cpu(), ref) < 1e-2


# voxels given several times and voxels outside the grid have no cell of their own: they follow the others in row order, so that
# every build of the same coordinates gives the same walk (and with it the same chunks and sums of the narrow layers)
@pytest.mark.parametrize("twice,outside", [(0, 0), (1, 0), (0, 3), (5000, 700), (34000, 0)])
def test_walk_is_a_function_of_the_coordinates(gpu_device, twice, outside):
    res = 230
    _say(f"walk order twice={twice} outside={outside}")
    rng = np.random.default_rng(twice + outside)
    base = reference_test_shell(96) + np.array([0, 50, 3, 101], np.int32)
    coords = np.concatenate([base, base[rng.integers(0, len(base), twice)], base[:outside]])
    coords[len(coords) - outside:, 1 + rng.integers(0, 3)] += rng.choice(np.array([-res, res], np.int32), outside)
    coords = np.ascontiguousarray(coords[rng.permutation(len(coords))])
    n = len(coords)
    dev = torch.from_numpy(coords).to(gpu_device)
    shape = torch.Size([1, 0, res, res, res])
    walks = [_np(SubMConv3dFunction._compute_neighbor_cache(dev, shape, (3, 3, 3), (1, 1, 1), False)["_cell_walk"]) for _ in range(4)]
    inside = ((coords >= 0) & (coords < np.array([1, res, res, res]))).all(1)
    first = {}
    for i in np.nonzero(inside)[0]:
        first.setdefault(tuple(coords[i]), i)
    losers = np.setdiff1d(np.arange(n), np.fromiter(first.values(), np.int64))
    assert np.array_equal(np.sort(walks[0]), np.arange(n))
    assert np.array_equal(walks[0][n - len(losers):], losers)
    for walk in walks[1:]:
        assert np.array_equal(walk, walks[0])


# the index's two forms: such a voxel is nobody's neighbor, finds the voxels that are its own neighbors, and is its own middle entry
@pytest.mark.parametrize("res", [40, 210])
def test_voxels_outside_the_grid(gpu_device, res):
    _say(f"voxels outside the grid res={res}")
    rng = np.random.default_rng(res)
    coords = np.concatenate([reference_test_shell(40), [[0, -1, 5, 5], [0, res, 6, 6], [0, 5, -7, 5], [0, 8, 8, res], [0, 8, res + 900, 8], [1, 5, 5, 5],
                                                        [-1, 5, 5, 5], [0, 20, 0, -1]]]).astype(np.int32)
    coords = np.ascontiguousarray(coords[rng.permutation(len(coords))])
    inside = ((coords >= 0) & (coords < np.array([1, res, res, res]))).all(1)
    at = {tuple(c): i for i, c in enumerate(coords) if inside[i]}
    want = np.full((len(coords), 27), 0xFFFFFFFF, np.uint32)
    for i, (b, x, y, z) in enumerate(coords):
        for v in range(27):
            want[i, v] = at.get((b, x + v // 9 - 1, y + v // 3 % 3 - 1, z + v % 3 - 1), 0xFFFFFFFF)
        want[i, 13] = i
    cache = SubMConv3dFunction._compute_neighbor_cache(torch.from_numpy(coords).to(gpu_device), torch.Size([1, 0, res, res, res]), (3, 3, 3),
                                                       (1, 1, 1), False)
    assert np.array_equal(_np(cache.neighbor_map), want)


# an infinity or NaN in the upstream gradient reaches the weight gradient through its own pairs alone, not as its product with the
# zeros that stand for a missing neighbor
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ci,co", [(16, 16), (24, 32)])
def test_narrow_weight_gradient_with_infinities(gpu_device, dtype, ci, co):
    _say(f"narrow weight gradient with infinities {ci}->{co} {dtype}")
    res = 210
    coords = torch.from_numpy(reference_test_shell(96) + np.array([0, 50, 3, 101], np.int32)).to(gpu_device)
    n, inf = len(coords), float("inf")
    gen = torch.Generator(device=gpu_device).manual_seed(ci)
    feats = torch.randn(n, ci, generator=gen, device=gpu_device).to(dtype)
    feats[500, 1], feats[501, 2], feats[502, 3] = inf, -inf, 0.0
    weight = torch.randn(co, 3, 3, 3, ci, generator=gen, device=gpu_device).to(dtype).requires_grad_()
    bias = torch.randn(co, generator=gen, device=gpu_device).to(dtype).requires_grad_()
    out, cache = sparse_submanifold_conv3d(feats, coords, torch.Size([1, ci, res, res, res]), weight, bias)
    up = torch.randn(n, co, generator=gen, device=gpu_device).to(dtype)
    up[500, 0], up[501, 1], up[502, 2], up[3000, 3], up[n - 1, 4], up[n - 2, 4] = inf, -inf, inf, float("nan"), inf, -inf
    up[7000:7300, 5] = -inf
    gw, gb = torch.autograd.grad(out, (weight, bias), up)
    assert cache["_narrow_overflows"] == 0
    m, f, g = cache.neighbor_map.cpu().to(torch.int64), feats.cpu().double(), up.cpu().double()
    want = []
    for v in range(27):
        rows = (m[:, v] != 0xFFFFFFFF).nonzero()[:, 0]
        want.append(g[rows].t() @ f[m[rows, v]])
    for got, ref in ((gw.detach().cpu().double().view(co, 27, ci), torch.stack(want, 1)), (gb.detach().cpu().double(), g.sum(0))):
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got == inf, ref == inf) and torch.equal(got == -inf, ref == -inf)
        ok = ref.isfinite()
        # one rounding to the type of fp32 sums over n rows (random signs: their error grows with the root)
        assert ok.any() and (got - ref)[ok].abs().max() <= 2.0 ** (-11 if dtype == torch.float16 else -8) * ref[ok].abs().max() + n ** 0.5 * 2.0 ** -21
