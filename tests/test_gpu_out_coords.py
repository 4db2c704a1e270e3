"""Output coordinates by bit map: kernels that mix one, two and three positions, longer ones, strides with and without a division, padding past the kernel."""
import numpy as np
import pytest
import torch

from flexgemm_amd.ops import spconv
from flexgemm_amd.ops.spconv.sparse_conv3d import SparseConv3dFunction
from oracle import sparse_conv as sc


@pytest.mark.gpu
@pytest.mark.parametrize("dims,n", [((1, 1, 1, 1), 1), ((2, 40, 41, 39), 3000), ((3, 9, 7, 70), 63), ((1, 130, 128, 129), 20000), ((2, 5, 3000, 33), 257),
                                     ((1, 128, 512, 512), 3000), ((1, 129, 512, 512), 3000)])
@pytest.mark.parametrize("geom", [((3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1)), ((3, 3, 3), (2, 2, 2), (1, 1, 1), (1, 1, 1)), ((2, 2, 2), (2, 2, 2), (0, 0, 0), (1, 1, 1)),
                                  ((1, 2, 3), (3, 2, 1), (0, 4, 2), (1, 2, 3)), ((3, 1, 2), (1, 3, 2), (5, 0, 1), (2, 1, 1)), ((3, 3, 4), (2, 1, 2), (1, 1, 2), (1, 2, 1)),
                                  ((3, 2, 3), (4, 5, 3), (2, 2, 2), (3, 1, 2))])
def test_output_coordinates(gpu_device, monkeypatch, dims, n, geom):
    print(f"[case] dims={dims} n={n} geom={geom}", flush=True)
    monkeypatch.setattr(spconv, "NEIGHBOR_MAP_BUILDER", "grid")
    shape = torch.Size([dims[0], 0, *dims[1:]])
    rng = np.random.default_rng(n)
    if min(sc.out_dims(tuple(shape), *geom)) < 1:
        return
    coords = np.unique(rng.integers(0, dims, (n, 4)).astype(np.int32), axis=0)
    coords = np.ascontiguousarray(coords[rng.permutation(len(coords))] if n % 2 else coords)
    got = SparseConv3dFunction._get_output_coords(torch.from_numpy(coords).to(gpu_device), shape, *geom)
    assert np.array_equal(got.cpu().numpy(), sc.output_coords(coords, tuple(shape), *geom))
