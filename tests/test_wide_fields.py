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
    # 257 to 1024 Gaussians on 16x16 tiles: pairs of tiles from a row list, an odd last column, one column, one row
    "rows": (250, 333, 257, 16, {}),
    "rows_mixed": (200, 140, 1024, 16, {}),
    "rows_one_column": (100, 16, 300, 16, {}),
    "rows_one_row": (16, 340, 321, 16, {"normalize": True}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(WIDE_CASES))
def test_wide_gaussians_render(case, device):
    """Blocks of wide Gaussians as polynomials against the oracle's exponentials, at the parity bar."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    M, Nf, K, tile, kw = WIDE_CASES[case]
    p = (_mixed if "mixed" in case else init_problem)(M, Nf, K, 7, **({} if "mixed" in case else {"sigma": max(3.0 / math.sqrt(K), 0.7)}))
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


@pytest.mark.gpu
@pytest.mark.parametrize("where", [(0, float("inf")), (1, float("inf")), (1, float("-inf"))])
@pytest.mark.parametrize("M,Nf,K,tile", [(320, 320, 100, 32), (320, 320, 300, 16)])
def test_wide_gaussians_infinite_mean(M, Nf, K, tile, where, device):
    """A Gaussian with an infinite mean among wide ones: its exponent is -inf wherever it is listed, so the field
    is that of the others (single fields of both renders, and the batch)."""
    from guass_amd.cuda_field import ext
    from guass_amd.ops import FieldBatchPlan

    p = init_problem(M, Nf, K, 3, sigma=0.7)
    p.mu[10, where[0]] = where[1]
    rest = wl.FieldProblem(p.name, M, Nf, p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp.clone(), p.grad)
    rest.amp[10] = 0.0
    rest.mu = p.mu.clone()
    rest.mu[10] = 0.0
    args = (tile, tile, 3.0, False, 80.0)
    q, o = p.to(device), rest.to(device)
    want = ext.gaussian_field_forward(o.row_coords, o.col_coords, o.mu, o.chol_raw, o.amp, *args)[0].cpu()
    got, tp, _ = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    pairs = int(tp[-1])
    assert pairs * (4 if tile == 32 else 1) >= 64 * K  # the rule of the single fields' polynomial kernels
    field_close(got, want)
    batch = FieldBatchPlan([q], device, capacities=[pairs], tile_out=tile, tile_in=tile)
    batch.forward()
    field_close(batch.plans[0].delta, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,backward", [(17, 2000, 96, False), (2000, 17, 96, False), (17, 2000, 300, False),
                                             (2000, 17, 300, False), (17, 17600, 60, True), (17600, 17, 60, True)])
def test_wide_gaussians_on_blocks_of_one_row(M, Nf, K, backward, device):
    """Gaussians as thin as the activation allows (1e-5) across the last block's only row or column: nothing in
    that block depends on the coefficients of the missing direction, however large."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    p = init_problem(M, Nf, K, 4, sigma=0.9)
    thin = 0 if M == 17 else 1
    p.mu[:, thin] = 1.0 - 1e-5
    p.chol_raw[:, 1] = 0.0
    p.chol_raw[:, 2 * thin] = -25.0
    p.amp *= 1e5
    args = (16, 16, 3.0, False, 80.0)
    r = fo.gaussian_field_fwd_bwd_fp64(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, *args)
    pairs, T = int(r[1][-1]), r[1].numel() - 1
    assert pairs >= 64 * K  # the rules of the polynomial kernels
    q = p.to(device)
    delta, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    field_close(delta, r[0])
    if backward:
        assert pairs >= 480 * K and pairs >= 24 * T and T >= 2048
        got = ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                          forward_workspace=ws)
        for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), got, r[3:]):
            grad_close(a, b, name, rtol=1e-5)


# The wide-field backward takes fields of 2048 blocks or more (256 in a batch) whose Gaussians span 480 blocks
# or more on average (192 in a batch): 16x16 and 32x32 tiles, ragged edges, Gaussians left to the element-wise kernel (narrow ones,
# and those of a block with an infinite dL/d(delta-W)), several times 64 listed, K past a bit row of 1024.
@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,tile,kind", [
    (800, 810, 70, 16, "init"), (790, 820, 70, 32, "init"), (800, 810, 150, 16, "mixed"), (800, 810, 150, 32, "mixed"),
    (730, 800, 1100, 16, "init"), (800, 805, 200, 32, "normalize")])
def test_wide_field_backward(M, Nf, K, tile, kind, device):
    from guass_amd.cuda_field import ext
    from guass_amd.ops import FieldBatchPlan
    from oracle import field_oracle as fo

    p = _mixed(M, Nf, K, 11) if kind == "mixed" else init_problem(M, Nf, K, 11, sigma=0.35 if K > 1000 else None)
    norm = kind == "normalize"
    r = fo.gaussian_field_fwd_bwd_fp64(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, tile, tile, 3.0,
                                       norm, 80.0)
    pairs = int(r[1][-1]) * (4 if tile == 32 else 1)
    assert pairs >= 480 * K and int(r[1][-1]) >= 24 * (r[1].numel() - 1)  # the rule the kernels go by
    q = p.to(device)
    args = (tile, tile, 3.0, norm, 80.0)
    delta, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    field_close(delta, r[0])
    plain = ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args)
    for _ in range(2):  # the accumulators and the flag are clear again in between
        got = ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                          forward_workspace=ws)
        for name, a, b, c in zip(("d_mu", "d_chol_raw", "d_amp"), got, r[3:], plain):
            grad_close(a, b, name, rtol=1e-5)
            grad_close(c, b, name, rtol=1e-5)
    layers = [p.to(device), init_problem(320, 330, 40, 12).to(device)]
    layers[1].grad = torch.randn(320 * 330, generator=torch.Generator().manual_seed(1)).to(device)
    batch = FieldBatchPlan(layers, device, capacities=[int(r[1][-1]), 400 * 40], tile_out=tile, tile_in=tile, normalize=norm)
    assert batch.info.wide_blocks > 0
    for _ in range(2):
        batch.forward()
        batch.backward()
    torch.cuda.synchronize()
    assert batch.status() == [0, 0]
    for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), (batch.plans[0].d_mu, batch.plans[0].d_chol_raw, batch.plans[0].d_amp),
                          r[3:]):
        grad_close(a, b, f"batch {name}", rtol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [16, 32])
def test_wide_field_backward_infinite_gradient(tile, device):
    """One infinite dL/d(delta-W): the Gaussians over it get non-finite gradients as from the element-wise
    kernels, the others finite ones."""
    from guass_amd.cuda_field import ext

    p = init_problem(800, 810, 300, 13, sigma=0.2)
    p.grad[5 * 810 + 7] = float("inf")
    q = p.to(device)
    args = (tile, tile, 3.0, False, 80.0)
    _, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    a, b = (ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                        forward_workspace=w) for w in (ws, None))
    listed = ids[tp[0]:tp[1]]
    assert listed.numel() >= 24
    for x, y in zip(a, b):
        fin = torch.isfinite(y).all(dim=-1)
        assert torch.equal(torch.isfinite(x).all(dim=-1), fin)
        assert not fin[listed].any() and int((~fin).sum()) == listed.numel()


@pytest.mark.gpu
def test_wide_field_backward_checks_saved_state(device):
    from guass_amd.cuda_field import ext

    p = init_problem(800, 810, 70, 14)
    q = p.to(device)
    args = (16, 16, 3.0, False, 80.0)
    _, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    for edit, msg in ((lambda t, i: i.__setitem__(100, 70), "out-of-range"), (lambda t, i: i.__setitem__(100, -1), "non-negative"),
                      (lambda t, i: t.__setitem__(9, 0), "monotonic")):
        t, i = tp.clone(), ids.clone()
        edit(t, i)
        with pytest.raises(RuntimeError, match=msg):
            ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, t, i, *args,
                                        forward_workspace=ws)
