"""Fields of wide Gaussians: every element under tens of them (an adapter as its layer initialises it)."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from guass_amd import _native as N
from guass_amd import workloads as wl
from tests.parity import binning_equal, field_close, grad_close


def init_problem(M: int, Nf: int, K: int, seed: int, sigma: float | None = None) -> wl.FieldProblem:
    """A uniform grid of K Gaussians of sigma 3 / sqrt(K) in the [-1, 1] coordinates (the layer's
    initialisation), jittered: about 60-80 Gaussians at an element, whatever K is."""
    g = torch.Generator().manual_seed(seed)
    side = math.ceil(math.sqrt(K))
    ax = torch.linspace(-1.0, 1.0, side)
    mu = torch.stack(torch.meshgrid(ax, ax, indexing="ij"), dim=-1).reshape(-1, 2)[:K].clone()
    s = 3.0 / math.sqrt(K) if sigma is None else sigma
    mu = (mu + 0.1 * s * torch.randn(K, 2, generator=g)).clamp(-0.99, 0.99).contiguous()
    raw = torch.stack((torch.log(torch.expm1(s * torch.exp(0.1 * torch.randn(K, generator=g)))),
                       0.2 * s * torch.randn(K, generator=g),
                       torch.log(torch.expm1(s * torch.exp(0.1 * torch.randn(K, generator=g))))), dim=-1)
    amp = 1e-3 * torch.randn(K, 1, generator=g)
    rc, cc = wl.axes(M, Nf)
    grad = torch.randn(M * Nf, generator=g)
    return wl.FieldProblem(f"init_{M}x{Nf}_k{K}", M, Nf, rc, cc, mu, raw.contiguous(), amp, grad)


@pytest.mark.parametrize("shape,tile", [((1280, 1280), 16), ((1280, 1280), 32), ((320, 320), 32), ((2560, 5120), 16)])
def test_backward_workspace_grows_with_k(shape, tile):
    """Fewer Gaussians take more accumulator stripes, yet a workspace sized for a K holds every smaller
    one (plans move between K within a capacity without allocating)."""
    lib, cfg = N.lib(), ctypes.byref(N.make_config(tile, tile, 3.0, False, 80.0))
    need = [lib.gf_backward_workspace_bytes(*shape, k, cfg) for k in range(0, 2200, 7)]
    assert all(a <= b for a, b in zip(need, need[1:]))


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,tile", [(96, 80, 3, 16), (320, 320, 16, 32), (320, 320, 32, 32), (640, 640, 256, 32)])
def test_striped_reduction_of_few_gaussians(M, Nf, K, tile, device):
    """Stripes for few Gaussians on many blocks (1 to 32): the training backward twice on one forward
    (the accumulators are zero again in between) against the oracle."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    p = init_problem(M, Nf, K, 5)
    r = fo.gaussian_field_fwd_bwd_batched(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, tile, tile,
                                          3.0, False, 80.0)
    q = p.to(device)
    args = (tile, tile, 3.0, False, 80.0)
    delta, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    binning_equal(tp, ids, r[1], r[2])
    field_close(delta, r[0])
    for fws in (ws, ws, None):
        got = ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                          forward_workspace=fws)
        for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), got, r[3:]):
            grad_close(a, b, name)


def _mixed(M: int, Nf: int, K: int, seed: int) -> wl.FieldProblem:
    """init_problem with every fifth Gaussian a few elements wide, listed between the others."""
    p = init_problem(M, Nf, K, seed)
    sub = p.chol_raw[::5]
    p.chol_raw[::5] = torch.stack((torch.full_like(sub[:, 0], math.log(math.expm1(8.0 / M))), torch.zeros_like(sub[:, 1]),
                                   torch.full_like(sub[:, 2], math.log(math.expm1(8.0 / Nf)))), dim=-1)
    return p


# Blocks cut by the matrix's edges, one row and one column of blocks, lists of 24 (the fewest taken), 64, 65 and
# several times 64, narrow Gaussians between the wide ones, normalised ones, and a clamp that keeps them all
# element by element.
WIDE_CASES = {
    "ragged": (250, 333, 200, 32, {}),
    "one_row": (9, 700, 60, 16, {}),
    "n24": (64, 64, 24, 16, {}),
    "n64": (64, 80, 64, 32, {}),
    "n65": (80, 64, 65, 32, {}),
    "mixed": (330, 200, 150, 32, {}),
    "normalize": (128, 200, 90, 16, {"normalize": True}),
    "clamp24": (128, 200, 90, 32, {"clamp": 24.0}),
    "noclamp": (200, 128, 256, 16, {"clamp": None}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(WIDE_CASES))
def test_wide_gaussians_render(case, device):
    """Blocks of wide Gaussians as polynomials against the oracle's exponentials, at the parity bar."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    M, Nf, K, tile, kw = WIDE_CASES[case]
    p = (_mixed if case == "mixed" else init_problem)(M, Nf, K, 7, **({} if case == "mixed" else {"sigma": max(3.0 / math.sqrt(K), 0.7)}))
    norm, clamp = kw.get("normalize", False), kw.get("clamp", 80.0)
    r = fo.gaussian_field_fwd_bwd_batched(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, tile, tile,
                                          3.0, norm, clamp)
    q = p.to(device)
    delta, tp, ids = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tile, tile, 3.0,
                                                norm, clamp)
    binning_equal(tp, ids, r[1], r[2])
    field_close(delta, r[0])


@pytest.mark.gpu
def test_wide_gaussians_infinite_amplitude(device):
    """An infinite amplitude among wide Gaussians stays out of the block's polynomial: every element it
    reaches is infinite, not NaN."""
    from guass_amd.cuda_field import ext

    p = init_problem(64, 64, 64, 3, sigma=1.5)
    p.amp[10] = float("inf")
    q = p.to(device)
    delta, _, _ = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, 32, 32, 3.0, False, 80.0)
    assert torch.isposinf(delta).all()
