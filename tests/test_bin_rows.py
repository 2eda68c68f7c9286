"""Binning past the mask path (K > 8192): a preparation over the chip, then a workgroup per tile row."""

from __future__ import annotations

import pytest
import torch

from guass_amd.cuda_field import ext
from oracle import field_oracle as fo
from tests.parity import binning_equal
from tests.test_gpu_parity import say, tiny_problem


@pytest.mark.gpu
@pytest.mark.parametrize("k", [8193, 9216, 16385])  # one round of 8 x 1024 rectangles and its remainders
@pytest.mark.parametrize("shape,tile", [((5, 7), 16), ((333, 16), 16), ((16, 17000), 16), ((610, 1283), 32), ((96, 80), 8)])
def test_tile_rows_binning(device, k, shape, tile):
    """One tile, one tile column, one tile row of more columns than the workgroup has threads, ragged grids:
    tile_ptr and ids bit-exact against the oracle's binning."""
    M, Nf = shape
    p = tiny_problem(M, Nf, k, k, log_scale_px=0.5, spread=0.9)
    g = torch.Generator().manual_seed(k)
    p.chol_raw[torch.arange(0, k, 901)] = torch.tensor([3.0, 0.2, 3.0])  # boxes past the matrix
    edge = torch.arange(k)[3::11]
    p.mu[edge] = torch.tensor([0.99, -0.99]) + 0.02 * torch.rand(len(edge), 2, generator=g)  # some outside
    say(f"row binning {M}x{Nf} K={k} tile {tile}")
    q = p.to(device)
    _, tp, ids = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tile, tile, 3.0,
                                            False, 80.0)
    ti = fo.build_tile_index(fo.tile_bounds(p.mu, fo.activate_cholesky(p.chol_raw), M, Nf, tile, tile, 3.0))
    binning_equal(tp, ids, ti.tile_ptr, ti.gaussian_ids)
