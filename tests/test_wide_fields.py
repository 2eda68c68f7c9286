"""Fields of wide Gaussians: every element under tens of them (an adapter as its layer initialises it)."""

from __future__ import annotations

import ctypes
import math
import re
from pathlib import Path

import numpy as np
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


@pytest.mark.parametrize("deg,reach", [("kPolyDeg", "kPolyReach"), ("kMomentDeg", "kMomentReach")])
def test_cut_series_keeps_its_bound(deg, reach):
    """The degrees and reaches of the kernels: the series of exp(-(l t + k t^2)) cut at the degree is within
    2^-24 (2 + 4 q) of its value at t = 1, over every l and k that the test for wide Gaussians lets pass."""
    src = (Path(N.__file__).parent / "csrc" / "gaussfield.hip").read_text()
    D = int(re.search(rf"\b{deg} = (\d+)", src).group(1))
    R = float(re.search(rf"\b{reach} = ([0-9.]+)f", src).group(1))
    max_q = float(re.search(r"\bkPolyMaxQ = ([0-9.]+)f", src).group(1)) * math.log(2.0)
    for q in (0.0, 0.1, 0.5, 1.0, 2.0, 4.5, 9.0, 13.0, max_q):
        most = R * (1.0 + 2.0 * q) ** (1.0 / (D + 2))
        l, k = np.meshgrid(np.linspace(-most, most, 301), np.linspace(0.0, most / 8.0, 81), indexing="ij")
        c = [np.ones_like(l)]
        for n in range(D):
            c.append(-(l * c[n] + (2.0 * k * c[n - 1] if n else 0.0)) / (n + 1))
        err = np.abs(sum(c) * np.exp(l + k) - 1.0) * (np.abs(l) + 8.0 * k <= most)
        assert err.max() <= 2.0**-24 * (2.0 + 4.0 * q), (q, err.max())


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


def _mixed(M: int, Nf: int, K: int, seed: int, sigma: float | None = None) -> wl.FieldProblem:
    """init_problem with every fifth Gaussian a few elements wide, listed between the others."""
    p = init_problem(M, Nf, K, seed, sigma)
    sub = p.chol_raw[::5]
    p.chol_raw[::5] = torch.stack((torch.full_like(sub[:, 0], math.log(math.expm1(8.0 / M))), torch.zeros_like(sub[:, 1]),
                                   torch.full_like(sub[:, 2], math.log(math.expm1(8.0 / Nf)))), dim=-1)
    return p


def _by_polynomials(tile_ptr, K: int, tile: int) -> bool:
    """The rule of the renders that look for wide Gaussians, for fields whose widest rectangle is no outlier: 256 blocks
    a Gaussian or more on average, and a list of 24."""
    tp = tile_ptr.cpu()
    return int(tp[-1]) * (4 if tile == 32 else 1) >= 256 * K and int((tp[1:] - tp[:-1]).max()) >= 24


# Fields of wide Gaussians, most of them small, whose mean rectangle is below the polynomials' rule ("ragged" and "rows"
# are above it): element by element, on the lists and grids that the polynomials have to handle too (below).
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

# Fields that go by polynomials: blocks cut by the matrix's edges, one row and one column of blocks, lists of 24
# (the fewest taken), 64, 65 and several times 64, narrow Gaussians between the wide ones, normalised ones, and
# from 257 Gaussians on the pairs of tiles from a row list.
POLY_CASES = {
    "ragged": (330, 345, 200, 32, {}),
    "n24": (320, 320, 24, 32, {}),
    "n64": (320, 320, 64, 16, {}),
    "n65": (320, 330, 65, 32, {}),
    "n65_16": (330, 320, 65, 16, {}),
    "mixed": (333, 350, 150, 32, {}),
    "mixed_16": (333, 350, 256, 16, {}),
    "normalize": (320, 327, 90, 16, {"normalize": True}),
    "noclamp": (320, 320, 256, 32, {"clamp": None}),
    "one_row": (16, 4300, 60, 16, {}),
    "one_column": (4300, 16, 60, 16, {}),
    "rows": (330, 345, 257, 16, {}),
    "rows_mixed": (330, 345, 1024, 16, {}),
    "rows_mixed_few": (320, 333, 290, 16, {"normalize": True}),
    "rows_one_column": (4300, 16, 300, 16, {}),
    "rows_one_row": (16, 4300, 321, 16, {"clamp": None}),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(WIDE_CASES) + [f"poly_{c}" for c in POLY_CASES])
def test_wide_gaussians_render(case, device):
    """Fields of wide Gaussians, element by element and as polynomials, against the oracle's exponentials, at the parity
    bar."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    poly = case.startswith("poly_")
    M, Nf, K, tile, kw = POLY_CASES[case[5:]] if poly else WIDE_CASES[case]
    if poly:
        p = (_mixed if "mixed" in case else init_problem)(M, Nf, K, 7, sigma=1.5)
    else:
        p = (_mixed if "mixed" in case else init_problem)(M, Nf, K, 7, **({} if "mixed" in case else {"sigma": max(3.0 / math.sqrt(K), 0.7)}))
    norm, clamp = kw.get("normalize", False), kw.get("clamp", 80.0)
    r = fo.gaussian_field_fwd_bwd_batched(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, tile, tile,
                                          3.0, norm, clamp)
    assert _by_polynomials(r[1], K, tile) == (poly or case in ("ragged", "rows"))
    q = p.to(device)
    delta, tp, ids = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tile, tile, 3.0,
                                                norm, clamp)
    binning_equal(tp, ids, r[1], r[2])
    field_close(delta, r[0])


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,tile,poly", [(64, 64, 64, 32, False), (320, 320, 64, 32, True), (320, 320, 64, 16, True),
                                              (320, 320, 300, 16, True)])
def test_wide_gaussians_infinite_amplitude(M, Nf, K, tile, poly, device):
    """An infinite amplitude among wide Gaussians stays out of the block's polynomial: every element it
    reaches is infinite, not NaN."""
    from guass_amd.cuda_field import ext

    p = init_problem(M, Nf, K, 3, sigma=1.5)
    p.amp[10] = float("inf")
    q = p.to(device)
    delta, tp, _ = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tile, tile, 3.0, False, 80.0)
    assert _by_polynomials(tp, K, tile) == poly
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
    assert pairs * (4 if tile == 32 else 1) >= 256 * K  # the rule of the single fields' polynomial kernels
    field_close(got, want)
    batch = FieldBatchPlan([q], device, capacities=[pairs], tile_out=tile, tile_in=tile)
    batch.forward()
    field_close(batch.plans[0].delta, want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,backward", [(17, 6000, 96, False), (6000, 17, 96, False), (17, 6000, 300, False),
                                             (6000, 17, 300, False), (17, 17600, 60, True), (17600, 17, 60, True)])
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
    assert pairs >= 256 * K  # the rules of the polynomial kernels
    q = p.to(device)
    delta, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    field_close(delta, r[0])
    if backward:
        assert pairs >= 480 * K and pairs >= 24 * T and T >= 2048
        got = ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                          forward_workspace=ws)
        for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), got, r[3:]):
            grad_close(a, b, name, rtol=1e-5)


def _few_wide(M: int, Nf: int, K: int, wide: int, seed: int, around: float | None = None) -> wl.FieldProblem:
    """`wide` Gaussians of 0.7 of the square (0.3 around one place), the others a few elements wide."""
    p = init_problem(M, Nf, K, seed, sigma=0.7 if around is None else 0.3)
    if around is not None:
        p.mu = (around * torch.randn(K, 2, generator=torch.Generator().manual_seed(seed))).contiguous()
    sub = p.chol_raw[wide:]
    p.chol_raw[wide:] = torch.stack((torch.full_like(sub[:, 0], math.log(math.expm1(8.0 / M))), torch.zeros_like(sub[:, 1]),
                                     torch.full_like(sub[:, 2], math.log(math.expm1(8.0 / Nf)))), dim=-1)
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,wide,tile,around", [
    (320, 320, 256, 26, 32, None),  # lists of wide Gaussians, small means: element by element
    (320, 320, 256, 26, 16, None), (320, 320, 1000, 30, 16, None),
    (320, 320, 256, 60, 32, None),
    (1280, 1280, 40, 40, 32, 0.02), (1280, 1280, 256, 256, 32, None), (1280, 1280, 300, 300, 16, None)])  # polynomials
def test_render_bits_do_not_depend_on_the_id_capacity(M, Nf, K, wide, tile, around, device):
    """The id capacity is the size of a buffer: the same field has the same delta-W, bit for bit, with exactly the room
    it needs, with more, and with a Gaussian on every tile; in a plan, a plan of a live K and a batch."""
    from guass_amd.ops import FieldBatchPlan, FieldPlan, StaticFieldPlan

    p = _few_wide(M, Nf, K, wide, 5, around)
    q = p.to(device)
    args, kw = (q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp), dict(tile_out=tile, tile_in=tile)
    default = FieldPlan(M, Nf, K, device, **kw)
    want = default.forward(*args).clone()
    pairs = default.pairs()
    assert default.status() == 0
    for cap in (pairs, 2 * pairs, 40 * pairs):
        plan = FieldPlan(M, Nf, K, device, ids_capacity=cap, **kw)
        assert torch.equal(plan.forward(*args), want), cap
        assert torch.equal(plan.tile_ptr, default.tile_ptr) and torch.equal(plan.ids[:pairs], default.ids[:pairs])
    static = StaticFieldPlan(M, Nf, K + 3 if K + 3 <= 256 or K > 256 else K, device, ids_capacity=pairs, **kw)
    static.set_params(q.mu, q.chol_raw, q.amp)
    assert torch.equal(static.forward(q.row_coords, q.col_coords), want)
    out = []
    for cap in (pairs, 40 * pairs):
        batch = FieldBatchPlan([q], device, capacities=[cap], **kw)
        batch.forward()
        out.append(batch.plans[0].delta.clone())
    assert torch.equal(out[0], out[1])


def _exponents(p: wl.FieldProblem, x: torch.Tensor, y: torch.Tensor) -> torch.Tensor:
    """Each Gaussian's exponent q [K, len(x), len(y)] in float64."""
    raw, mu = p.chol_raw.double().to(x.device), p.mu.double().to(x.device)
    l11, l21, l22 = (torch.nn.functional.softplus(raw[:, 0]) + 1e-5, raw[:, 1],
                     torch.nn.functional.softplus(raw[:, 2]) + 1e-5)
    u = (x.double()[None] - mu[:, :1]) / l11[:, None]
    v = ((y.double()[None] - mu[:, 1:])[:, None] - (l21[:, None] * u)[:, :, None]) / l22[:, None, None]
    return 0.5 * (u.square()[:, :, None] + v.square())


def _spread(M: int, Nf: int, K: int, sigma: tuple[float, float], seed: int, around: float | None = None):
    """K Gaussians of about sigma elements, anywhere or within `around` elements' sigma of the middle."""
    g = torch.Generator().manual_seed(seed)
    p = init_problem(M, Nf, K, seed)
    unit = torch.tensor([2.0 / (M - 1), 2.0 / (Nf - 1)])
    p.mu = (1.98 * torch.rand(K, 2, generator=g) - 0.99 if around is None
            else (around * unit * torch.randn(K, 2, generator=g)).clamp(-0.99, 0.99)).contiguous()
    s = torch.tensor(sigma) * unit * torch.exp(0.1 * torch.randn(K, 2, generator=g))
    raw = torch.log(torch.expm1(s))
    p.chol_raw = torch.stack((raw[:, 0], 0.1 * s[:, 1] * torch.randn(K, generator=g), raw[:, 1]), dim=-1).contiguous()
    p.amp = 1e-3 * (0.5 + torch.rand(K, 1, generator=g))
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("sigma_mult", [3.0, 5.0])
@pytest.mark.parametrize("sigma", [(36.0, 36.0), (60.0, 60.0), (30.0, 120.0)])
@pytest.mark.parametrize("M,Nf,K,tile", [(640, 640, 100, 32), (640, 640, 400, 16)])
def test_wide_gaussians_far_elements(M, Nf, K, tile, sigma, sigma_mult, device):
    """Positive Gaussians about the middle: every element, also where all n that its tile lists are far away and
    small, is right to the rounding of its own terms: 2^-24 (8 + 8 q) of each (in first order the covariance's entries,
    their factor, the offsets, the products and the square are up to 16 roundings of half a unit, in a square; the cut may
    leave out 2 + 4 q) and 2^-24 2 sqrt(n) of their sum (n roundings of half a unit and of any sign, 7 times their
    standard deviation)."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    p = _spread(M, Nf, K, sigma, 1, around=15.0)
    args = (tile, tile, sigma_mult, False, 80.0)
    r = fo.gaussian_field_fwd_bwd_fp64(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, *args)[0]
    q = p.to(device)
    delta, tp, ids = ext.gaussian_field_forward(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    ref = r.double().view(M, Nf).to(device)
    err = (delta.double().view(M, Nf) - ref).abs()
    worst = 0.0
    for r0 in range(0, M, 64):  # the terms that an element's tile lists
        x = _exponents(p, q.row_coords[r0:r0 + 64], q.col_coords)
        # (past the clamp, x = 40, the render leaves exp(-x) where the reference has exp(-40))
        value = q.amp.double()[:, :, None] * torch.exp(-x)
        term = value * (8.0 + 8.0 * x) * 2.0**-24 + q.amp.double()[:, :, None] * math.exp(-40.0)
        for t0 in range(r0, r0 + 64, tile):
            for t in range(t0 // tile * (Nf // tile), (t0 // tile + 1) * (Nf // tile)):
                c0 = (t % (Nf // tile)) * tile
                listed = ids[int(tp[t]):int(tp[t + 1])]
                e = err[t0:t0 + tile, c0:c0 + tile]
                if listed.numel() == 0:
                    assert not bool(e.any())
                    continue
                at = (listed, slice(t0 - r0, t0 - r0 + tile), slice(c0, c0 + tile))
                bound = term[at].sum(0) + 2.0**-23 * math.sqrt(listed.numel()) * value[at].sum(0)
                worst = max(worst, float((e / bound).max()))
    assert worst <= 1.0, worst


@pytest.mark.gpu
@pytest.mark.parametrize("sigma_mult", [3.0, 5.0])
@pytest.mark.parametrize("sigma,tile", [((60.0, 60.0), 16), ((60.0, 60.0), 32), ((75.0, 75.0), 32), ((50.0, 200.0), 16)])
def test_wide_field_backward_of_one_block(sigma, tile, sigma_mult, device):
    """Positive dL/d(delta-W) in one 16x16 block, or one of its elements: no other block's terms hide an error there,
    and each Gaussian's gradient (in units of its amplitude and its axes, so that d_amp, a sum of positive terms, sets
    its scale) is right to the rounding of its exponent in the block, 2^-24 (16 + 32 q) with q the largest over the
    block: the cut's 2 + 4 q, times 8 for the chain rule's sums of moments."""
    from guass_amd.cuda_field import ext
    from oracle import field_oracle as fo

    M = Nf = 1280
    p = _spread(M, Nf, 256, sigma, 2)
    args = (tile, tile, sigma_mult, False, 80.0)
    q = p.to(device)
    _, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    pairs = int(tp[-1]) * (4 if tile == 32 else 1)
    assert pairs >= 480 * p.mu.shape[0]  # the rule the kernels go by
    axes, one = torch.nn.functional.softplus(p.chol_raw[:, ::2]).double(), torch.ones(p.mu.shape[0], dtype=torch.float64)
    for b0, b1 in ((40, 40), (0, 0), (25, 62)):
        rows, cols = slice(16 * b0, 16 * b0 + 16), slice(16 * b1, 16 * b1 + 16)
        t = (16 * b0 // tile) * (Nf // tile) + 16 * b1 // tile
        listed = ids[int(tp[t]):int(tp[t + 1])].cpu()
        x = _exponents(p, p.row_coords[rows], p.col_coords[cols]).flatten(1).amax(1)[listed]
        for only in (None, (15, 15), (0, 15)):
            block = 0.5 + torch.rand(16, 16, generator=torch.Generator().manual_seed(b0))
            if only is not None:
                block = torch.zeros(16, 16)
                block[only] = 1.0
            grad = torch.zeros(M, Nf)
            grad[rows, cols] = block
            # the block by itself, every Gaussian listed
            r = fo.gaussian_field_fwd_bwd_fp64(p.row_coords[rows], p.col_coords[cols], p.mu, p.chol_raw, p.amp,
                                               block.reshape(-1), 16, 16, 1e3, False, 80.0)
            got = ext.gaussian_field_backward(grad.reshape(-1).to(device), q.row_coords, q.col_coords, q.mu, q.chol_raw,
                                              q.amp, tp, ids, *args, forward_workspace=ws)
            a, b = (torch.cat((m.double() * axes, c.double() * torch.stack((one, axes[:, 1], one), -1), d.double() * p.amp), -1)[listed]
                    for m, c, d in ([v.cpu() for v in got], r[3:]))
            off = (a - b).norm(dim=-1) / b.norm(dim=-1)
            near = x <= 40.0  # (beyond, the values leave the numbers' range)
            worst = float((off / (2.0**-24 * (16.0 + 32.0 * x)))[near].max())
            assert worst <= 1.0, (b0, b1, only, worst)


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


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,tile,kind", [
    (320, 330, 300, 16, "narrow"), (320, 330, 300, 32, "narrow"),  # one launch, and the reduction element by element
    (800, 810, 70, 16, "init"), (800, 810, 70, 32, "init")])  # by moments
def test_live_k_backward_past_the_id_capacity(M, Nf, K, tile, kind, device):
    """A plan of a live K whose pairs do not fit: the backward reads the ids that have room, as a plan of the same
    capacity does, and says so in its status."""
    from guass_amd.ops import FieldPlan, StaticFieldPlan

    p = init_problem(M, Nf, K, 15) if kind == "init" else _few_wide(M, Nf, K, 0, 15)
    q = p.to(device)
    kw = dict(tile_out=tile, tile_in=tile)
    args = (q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp)
    whole = FieldPlan(M, Nf, K, device, **kw)
    whole.forward(*args)
    cap = whole.pairs() - 32
    if kind == "init":
        assert cap * (4 if tile == 32 else 1) >= 480 * K and cap >= 24 * whole.T  # the wide backward's rule
    plan = FieldPlan(M, Nf, K, device, ids_capacity=cap, **kw)
    plan.forward(*args)
    want = [v.clone() for v in plan.backward_direct(q.grad, *args)]
    static = StaticFieldPlan(M, Nf, K, device, ids_capacity=cap, **kw)
    static.set_params(q.mu, q.chol_raw, q.amp)
    static.forward(q.row_coords, q.col_coords)
    got = static.backward_direct(q.grad, q.row_coords, q.col_coords)
    assert static.status() == plan.status() and static.status() & N.GF_STATUS_CAPACITY
    assert static.status("backward") == plan.status("backward") != 0
    assert static.pairs() == cap + 32
    for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), got, want):
        grad_close(a, b.double().cpu(), name, rtol=1e-5)


def _flag(plan) -> int:
    """What a reduction by moments left in the backward workspace's header: whether some Gaussians were not wide."""
    return int(plan.bwd_ws[4:8].view(torch.int32)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("M,Nf,K,tile,kind", [
    (800, 810, 150, 16, "sparse"), (800, 810, 150, 32, "sparse"),  # a few elements wide everywhere
    (800, 810, 2100, 16, "clustered"),  # heavy tiles, their four-wave workgroups
    (800, 810, 150, 16, "mixed"), (800, 810, 150, 32, "mixed")])  # wide with some that are not
def test_bounded_pair_count_goes_by_tiles(M, Nf, K, tile, kind, device):
    """A pair count that may be a bound (the id capacity, by default a Gaussian on every tile) says nothing of the
    field: the backward reduces it tile by tile, without a pass by moments before, and also in a replayed graph."""
    from guass_amd.ops import FieldPlan, StaticFieldPlan
    from oracle import field_oracle as fo

    if kind == "mixed":
        p = _mixed(M, Nf, K, 21)
    else:
        p = _few_wide(M, Nf, K, 0, 21)
        if kind == "clustered":
            at = torch.randn(8, 2, generator=torch.Generator().manual_seed(22)).mul(0.4).clamp(-0.9, 0.9)
            p.mu = (at[torch.arange(K) % 8] + 0.05 * p.mu).contiguous()
    r = fo.gaussian_field_fwd_bwd_fp64(p.row_coords, p.col_coords, p.mu, p.chol_raw, p.amp, p.grad, tile, tile, 3.0,
                                       False, 80.0)
    T, P, quad = r[1].numel() - 1, int(r[1][-1]), 4 if tile == 32 else 1
    by_moments = quad * P >= 480 * K and P >= 24 * T and quad * T >= 2048
    assert by_moments == (kind == "mixed")
    q = p.to(device)
    args, kw = (q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp), dict(tile_out=tile, tile_in=tile)
    plan = FieldPlan(M, Nf, K, device, **kw)
    cap = plan.capacity
    assert quad * cap >= 480 * K and cap >= 24 * T and quad * T >= 2048  # the bound would make any field a wide one
    plan.forward(*args)
    pairs, span = plan.bin_info()
    assert pairs == P

    def close(got):
        for name, a, b in zip(("d_mu", "d_chol_raw", "d_amp"), got, r[3:]):
            grad_close(a, b, name, rtol=1e-5)

    plan.backward_reduce(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw)
    assert _flag(plan) == 0
    close(plan.backward_finish(q.chol_raw, q.amp))
    close(plan.backward(q.grad, *args))
    close(plan.backward(q.grad, *args, num_pairs=P))
    for num, sp in ((None, None), (None, span), (P, span)):
        plan.forward(*args)
        close(plan.backward_direct(q.grad, *args, num_pairs=num, max_span=sp))

    static = StaticFieldPlan(M, Nf, K + 40, device, ids_capacity=cap, **kw)
    static.set_params(q.mu, q.chol_raw, q.amp)

    def step():
        plan.forward(*args)
        a = plan.backward_direct(q.grad, *args, num_pairs=P, max_span=span)
        static.forward(q.row_coords, q.col_coords)
        return a, static.backward_direct(q.grad, q.row_coords, q.col_coords)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a, b = step()
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        close(a)
        close([v[:K] for v in b])
        q.amp.add_(0.0)  # the program's own work between the replays
    assert plan.status() == 0 and static.status() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind,tile", [("init", 16), ("mixed", 16), ("init", 32)])
def test_wide_field_backward_of_ids_listed_again(kind, tile, device):
    """A saved binning whose lists name a Gaussian more than once: each time counts, by moments as element by element
    (whose constants are recomputed from the parameters)."""
    from guass_amd.cuda_field import ext

    M, Nf, K = 800, 810, 150
    p = _mixed(M, Nf, K, 23) if kind == "mixed" else init_problem(M, Nf, K, 23)
    q = p.to(device)
    args = (tile, tile, 3.0, False, 80.0)
    _, tp, ids, ws = ext.forward_with_workspace(q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, *args)
    T, pairs = tp.numel() - 1, int(tp[-1])
    assert pairs * (4 if tile == 32 else 1) >= 480 * K and pairs >= 24 * T  # the rule the kernels go by
    listed = tp.cpu()
    for t in (0, 1, T // 2, T - 1):
        s, e = int(listed[t]), int(listed[t + 1])
        assert e - s >= 8
        ids[s + 3:e - 1:4] = ids[s + 2].clone()
        ids[e - 1] = ids[e - 2].clone()
    a, b = (ext.gaussian_field_backward(q.grad, q.row_coords, q.col_coords, q.mu, q.chol_raw, q.amp, tp, ids, *args,
                                        forward_workspace=w) for w in (ws, None))
    for name, x, y in zip(("d_mu", "d_chol_raw", "d_amp"), a, b):
        grad_close(x, y.double().cpu(), name, rtol=1e-5)
