"""Performance cases of the Gaussian-field path: what its users run, over the range they run it in.

A case is one pass of a training step's or a sampler's work on the field kernels, through the
package's public entry points:

* ``train``   ``gaussian_field_train`` and autograd's backward: what an adapted layer does by itself;
* ``graph``   ``FieldPlan.forward`` + ``backward_direct`` replayed from a HIP graph;
* ``fused``   ``FieldPlan.fwd_bwd_fused`` (a target known beforehand) replayed from a HIP graph;
* ``step``    ``FieldPlan.forward`` + ``backward_direct`` launched eagerly;
* ``render``  ``FieldBatchPlan.forward`` of many layers: a sampler's render of a loaded adapter;
* ``batch``   ``FieldBatchPlan.forward`` + ``backward`` of many layers: a model's training step;
* ``model``   ``GaussianFieldBatch.render``, the merged layers' forward and autograd's backward.

Fields (``field``): ``init`` is an adapter as ``GaussianLinear`` initialises it (a uniform grid of
Gaussians of sigma 3 / sqrt(K) in the [-1, 1] coordinates) some steps into training: every element
lies under tens of Gaussians, whatever K is.  ``trained`` has sizes of a few elements around random
places, ``clustered`` the same around eight centres (densification), as the benchmark's workloads.
"""

import math

import torch

DEVICE = "cuda"
SIGMA = 3.0
EPS = 1e-5  # added to the softplus of the Cholesky factor's diagonal
BLOCK_WIDTHS = (320, 320, 640, 640, 1280, 1280, 1280)  # an SD1.5 UNet's down blocks and its middle


def listed():
    one = dict(normalize=False, clamp=80.0)
    return [
        # The smallest call: the shipped configurations' smallest K on a narrow attention layer.
        dict(name="train_320_k32", kind="train", M=320, N=320, K=32, tile=32, field="init", **one),
        # The shipped configurations' middle K, tiles of 32, on a wide attention layer by itself.
        dict(name="train_1280_k256", kind="train", M=1280, N=1280, K=256, tile=32, field="init", **one),
        # A loaded adapter rendered once for sampling: to_q and to_v of seven transformer blocks.
        dict(name="render_k256_t32", kind="render", first=0, layers=28, K=256, tile=32, field="init", **one),
        # The benchmark's layer, as a program that keeps its plan and graph steps it.
        dict(name="graph_1280_k1024", kind="graph", M=1280, N=1280, K=1024, tile=16, field="trained", px=8.0, **one),
        # A fit to a fixed target on a small cross-attention layer.
        dict(name="fused_320x768_k256", kind="fused", M=320, N=768, K=256, tile=16, field="trained", px=6.0, **one),
        # A ragged layer (rows that are not 16-byte aligned, partial tiles), normalised Gaussians, no clamp.
        dict(name="step_1000x1283_k777", kind="step", M=1000, N=1283, K=777, tile=16, field="trained", px=8.0,
             normalize=True, clamp=None),
        # A densified feed-forward layer: eight clusters, very uneven tiles.
        dict(name="step_clustered_k4096", kind="step", M=1280, N=5120, K=4096, tile=16, field="clustered", px=5.0, **one),
        # The same layer freshly initialised, tiles of 16: the most work a single layer has.
        dict(name="step_init_1280x5120", kind="step", M=1280, N=5120, K=1024, tile=16, field="init", **one),
        # More Gaussians than the coverage masks take.
        dict(name="step_2560x5120_k16384", kind="step", M=2560, N=5120, K=16384, tile=16, field="trained", px=6.0, **one),
        # A model's step over to_q and to_v of seven transformer blocks, trained fields.
        dict(name="batch_k1024_t16", kind="batch", first=0, layers=28, K=1024, tile=16, field="trained", px=8.0, **one),
        # The same step at the start of training with the shipped tile size.
        dict(name="batch_init_k256_t32", kind="batch", first=0, layers=28, K=256, tile=32, field="init", **one),
        # Whole layers: one transformer block's eight attention linears, merged weights, GEMMs and autograd.
        dict(name="model_640_k256", kind="model", width=640, tokens=1024, K=256, tile=32, field="init", **one),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("train", "train", "graph", "fused", "step", "step", "step", "render", "batch", "batch", "model"))
    c = dict(kind=kind, tile=rng.choice((16, 32)), normalize=rng.random() < 0.2, clamp=rng.choice((80.0, 80.0, 80.0, None)),
             field=rng.choice(("init", "trained", "clustered")))
    if kind in ("render", "batch"):
        c["first"], c["layers"], c["K"] = rng.randrange(28), rng.randint(2, 28), spread(32, 1024)
    elif kind == "model":
        c["width"], c["K"] = rng.choice((320, 640, 1280)), spread(32, 1024)
        c["tokens"] = spread(64, 1310720 // c["width"])
    else:
        c["M"], c["N"] = spread(48, 1280), spread(48, 5120)
        # a field of more Gaussians than one per 64 elements is no longer a small adapter
        c["K"] = max(1, min(spread(8, 8192), c["M"] * c["N"] // 64))
        if kind == "fused":
            c["tile"], c["K"] = 16, min(c["K"], 2048)
        if kind == "step" and rng.random() < 0.25:  # past the masks' 8192 Gaussians
            c["M"], c["N"], c["K"] = spread(1024, 2560), spread(1024, 5120), spread(8193, 16384)
            c["field"] = rng.choice(("trained", "clustered"))
    if c["field"] != "init":
        c["px"] = round(math.exp(rng.uniform(math.log(3.0), math.log(10.0))), 2)
    return c


# ------------------------------------------------------------------------------------- inputs


def _shapes(case):
    """[(out, in)] of the case's fields."""
    if case["kind"] in ("render", "batch"):
        every = [(c, n) for c in BLOCK_WIDTHS for n in (c, c, c, 768)]  # attn1 to_q, to_v, attn2 to_q, to_v
        return [every[(case["first"] + i) % len(every)] for i in range(case["layers"])]
    if case["kind"] == "model":
        c = case["width"]
        return [(c, c)] * 6 + [(c, 768)] * 2  # attn1 q, k, v, out and attn2 q, out; attn2 k, v
    return [(case["M"], case["N"])]


def _unsoftplus(y):
    return torch.log(torch.expm1((y - EPS).clamp(min=1e-7)))


def _field(case, M, N, K, g):
    """(mu [K,2], chol_raw [K,3], amp [K,1]) in float32 on the CPU, from the generator."""
    f64 = torch.float64
    if case["field"] == "init":
        side = math.ceil(math.sqrt(K))
        ax = torch.linspace(-1.0, 1.0, side, dtype=f64)
        mu = torch.stack(torch.meshgrid(ax, ax, indexing="ij"), dim=-1).reshape(-1, 2)[:K].clone()
        sigma = 3.0 / math.sqrt(K)
        mu = (mu + 0.1 * sigma * torch.randn(K, 2, generator=g, dtype=f64)).clamp(-0.999999, 0.999999)
        raw = torch.zeros(K, 3, dtype=f64)
        raw[:, 0] = _unsoftplus(sigma * torch.exp(0.1 * torch.randn(K, generator=g, dtype=f64)))
        raw[:, 1] = 0.1 * sigma * torch.randn(K, generator=g, dtype=f64)
        raw[:, 2] = _unsoftplus(sigma * torch.exp(0.1 * torch.randn(K, generator=g, dtype=f64)))
        amp = 1e-4 * torch.randn(K, 1, generator=g, dtype=f64)
        return mu.float(), raw.float(), amp.float()
    size = torch.tensor([M, N], dtype=f64)
    at = torch.rand(K, 2, generator=g, dtype=f64) * size
    if case["field"] == "clustered":
        centres = torch.rand(8, 2, generator=g, dtype=f64) * size
        at = centres[torch.randint(0, 8, (K,), generator=g)] + 40.0 * torch.randn(K, 2, generator=g, dtype=f64)
        at = torch.minimum(at.clamp(min=0.0), size - 1.0)
    # axes of log-normal length in elements, at a random angle
    ln = math.log(case["px"]) + (0.6 * torch.randn(K, 2, generator=g, dtype=f64)).clamp(-1.5, 1.5)
    a = math.pi * torch.rand(K, generator=g, dtype=f64)
    c, s, v = torch.cos(a), torch.sin(a), torch.exp(2.0 * ln)
    unit = 2.0 / torch.clamp(size - 1.0, min=1.0)
    s00 = (c * c * v[:, 0] + s * s * v[:, 1]) * unit[0] * unit[0]
    s01 = c * s * (v[:, 0] - v[:, 1]) * unit[0] * unit[1]
    s11 = (s * s * v[:, 0] + c * c * v[:, 1]) * unit[1] * unit[1]
    l11 = s00.sqrt()
    l21 = s01 / l11
    l22 = (s11 - l21 * l21).clamp(min=0.0).sqrt()
    raw = torch.stack((_unsoftplus(l11), l21, _unsoftplus(l22)), dim=-1)
    return (at * unit - 1.0).float(), raw.float(), (1e-3 * torch.randn(K, 1, generator=g, dtype=f64)).float()


class _Inputs:
    """One field's tensors on the GPU."""


def _inputs(case, seed):
    """The fields of a case: parameters from a CPU generator, dL/d(delta-W) from a GPU one."""
    g = torch.Generator().manual_seed(seed)
    gd = torch.Generator(device=DEVICE).manual_seed(seed)
    fields = []
    for M, N in _shapes(case):
        f = _Inputs()
        f.M, f.N, f.K = M, N, case["K"]
        mu, raw, amp = _field(case, M, N, f.K, g)
        f.row_coords = torch.linspace(-1.0, 1.0, M).to(DEVICE)
        f.col_coords = torch.linspace(-1.0, 1.0, N).to(DEVICE)
        f.mu, f.chol_raw, f.amp = mu.to(DEVICE), raw.to(DEVICE), amp.to(DEVICE)
        f.grad = None
        if case["kind"] not in ("render", "model"):
            f.grad = torch.randn(M * N, generator=gd, device=DEVICE)
        fields.append(f)
    if case["kind"] != "model":
        return fields, None
    c, t = case["width"], case["tokens"]
    m = _Inputs()
    m.weights = [torch.randn(M, N, generator=gd, device=DEVICE) / math.sqrt(N) for M, N in _shapes(case)]
    x, ctx = torch.randn(t, c, generator=gd, device=DEVICE), torch.randn(77, 768, generator=gd, device=DEVICE)
    m.xs = [x] * 6 + [ctx] * 2
    m.gs = [torch.randn(xi.shape[0], c, generator=gd, device=DEVICE) for xi in m.xs]
    for f in fields:
        f.mu_raw = torch.atanh(f.mu.clamp(-0.999999, 0.999999))
    return fields, m


# ------------------------------------------------------------------------------------- prepare


def _config(case):
    return dict(tile_out=case["tile"], tile_in=case["tile"], sigma_multiplier=SIGMA, normalize=case["normalize"],
                clamp_quad=case["clamp"])


def _graph(fn):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _plan(case, f):
    """A FieldPlan with room for the field's pairs, and (pairs, widest rectangle) as its binning says."""
    from guass_amd.ops import FieldPlan

    kw = _config(case)
    cap = 16 * f.K + 4096
    while True:
        plan = FieldPlan(f.M, f.N, f.K, DEVICE, ids_capacity=cap, **kw)
        plan.forward(f.row_coords, f.col_coords, f.mu, f.chol_raw, f.amp)
        pairs, span = plan.bin_info()
        if pairs == cap:
            return plan, pairs, span
        cap = max(pairs, 1)


def prepare(case, seed):
    fields, m = _inputs(case, seed)
    s = _Inputs()
    s.kind = case["kind"]
    if s.kind == "train":
        f = s.f = fields[0]
        s.kw = _config(case)
        s.params = [t.requires_grad_(True) for t in (f.mu, f.chol_raw, f.amp)]
    elif s.kind in ("graph", "fused", "step"):
        f = s.f = fields[0]
        s.plan, s.pairs, s.span = _plan(case, f)
        if s.kind != "step":
            s.graph, s.out = _graph(lambda: _plan_pass(s))
    elif s.kind in ("render", "batch"):
        from guass_amd.ops import FieldBatchPlan

        s.fields = fields
        s.plan = FieldBatchPlan(fields, DEVICE, capacities=[32 * f.K for f in fields], **_config(case))
        for _ in range(4):
            s.plan.forward()
            status, pairs = s.plan.read(clear=True)
            if not any(status):
                break
            s.plan.update(capacities=[int(1.25 * p) + 1 for p in pairs])
    else:
        from guass_amd.layers import GaussianAdapterConfig, GaussianFieldBatch, GaussianLinear

        s.m, s.layers = m, []
        for f, w in zip(fields, m.weights):
            cfg = GaussianAdapterConfig(init_num_gaussians=f.K, tile_out=case["tile"], tile_in=case["tile"],
                                        normalize_gaussian=case["normalize"], delta_apply="merged")
            ly = GaussianLinear(f.N, f.M, bias=False, adapter_config=cfg, device=DEVICE)
            with torch.no_grad():
                ly.weight.copy_(w)
            ly.load_adapter_state(dict(mu_raw=f.mu_raw, chol_raw=f.chol_raw, amp=f.amp))
            s.layers.append(ly)
        s.batch = GaussianFieldBatch(s.layers)
        s.params = [p for ly in s.layers for p in (ly.mu_raw, ly.chol_raw, ly.amp)]
    return s


# ------------------------------------------------------------------------------------- run


def _plan_pass(s):
    f, plan = s.f, s.plan
    if s.kind == "fused":
        delta, (d_mu, d_chol, d_amp) = plan.fwd_bwd_fused(f.row_coords, f.col_coords, f.mu, f.chol_raw, f.amp, f.grad,
                                                          num_pairs=s.pairs, max_span=s.span)
    else:
        delta = plan.forward(f.row_coords, f.col_coords, f.mu, f.chol_raw, f.amp)
        d_mu, d_chol, d_amp = plan.backward_direct(f.grad, f.row_coords, f.col_coords, f.mu, f.chol_raw, f.amp,
                                                   num_pairs=s.pairs, max_span=s.span)
    return dict(delta=delta, tile_ptr=plan.tile_ptr, d_mu=d_mu, d_chol_raw=d_chol, d_amp=d_amp)


def run(s):
    if s.kind == "train":
        from guass_amd.cuda_field.runtime import gaussian_field_train

        f = s.f
        delta = gaussian_field_train(row_coords=f.row_coords, col_coords=f.col_coords, mu=f.mu, chol_raw=f.chol_raw,
                                     amp=f.amp, **s.kw)
        d_mu, d_chol, d_amp = torch.autograd.grad(delta, s.params, f.grad)
        return dict(delta=delta.detach(), d_mu=d_mu, d_chol_raw=d_chol, d_amp=d_amp)
    if s.kind == "step":
        return _plan_pass(s)
    if s.kind in ("graph", "fused"):
        s.graph.replay()
        return s.out
    if s.kind == "render":
        s.plan.forward()
        return dict(deltas=[p.delta for p in s.plan.plans])
    if s.kind == "batch":
        s.plan.forward()
        s.plan.backward()
        return dict(deltas=[p.delta for p in s.plan.plans], grads=s.plan.grad_flat[:s.plan.grad_numel])
    s.batch.render()
    ys = [ly(x) for ly, x in zip(s.layers, s.m.xs)]
    grads = torch.autograd.grad(ys, s.params, s.m.gs)
    return dict(ys=[y.detach() for y in ys], grads=list(grads))


# ------------------------------------------------------------------------------------- what a pass needs


def _mean_cover(case, M, N):
    """Gaussians whose tiles hold an element, on average over the field: an estimate from the sizes."""
    K, t = case["K"], case["tile"]
    if case["field"] == "init":
        side = 2 * SIGMA * 3.0 / math.sqrt(K)  # of the [-1, 1] axes
        # the box of a uniformly placed Gaussian cut at the matrix's edges, and half a tile on either side
        share = [min(1.0, (side - side * side / 8 if side < 4 else 2.0) / 2 + min(t, n) / n) for n in (M, N)]
        return K * share[0] * share[1]
    box = 2 * SIGMA * case["px"] * math.exp(0.18) + t
    return K * min(1.0, box / M) * min(1.0, box / N)


def work(case):
    """Bytes: every output element written and every dL/d(delta-W) element read once, parameters in
    and gradients out (24 B each a Gaussian).  Operations: 15 an evaluation of a Gaussian at an
    element in the forward, 41 in the backward, and a model's matrix products."""
    b = f = 0.0
    for M, N in _shapes(case):
        e = _mean_cover(case, M, N) * M * N
        b += 4.0 * M * N + 24.0 * case["K"]
        f += 15.0 * e
        if case["kind"] != "render":
            b += 4.0 * M * N + 24.0 * case["K"]
            f += 41.0 * e
    if case["kind"] == "model":
        c, t = case["width"], case["tokens"]
        for (M, N), rows in zip(_shapes(case), [t] * 6 + [77] * 2):
            b += 4.0 * (2 * M * N + rows * (N + 2 * M))
            f += 4.0 * rows * M * N
    return {"bytes": b, "flops": f}


def tolerance(case):
    # All sums are in 32 bits: gradients of some hundred thousand terms, atomics in any order.
    # tile_ptr holds whole numbers, which are the same.
    return {"rel": 1e-5, "max": 2e-4}


# ------------------------------------------------------------------------------------- in 64 bits


def _rectangles(case, f, mu):
    """First and last tile row and column of each Gaussian: the 3-sigma box, whose float32
    operations are part of the definition (it decides which tiles a Gaussian belongs to)."""
    raw, mu, t = f.chol_raw.detach().cpu(), mu.detach().cpu(), case["tile"]
    L = torch.zeros(f.K, 2, 2)
    L[:, 0, 0] = torch.nn.functional.softplus(raw[:, 0]) + EPS
    L[:, 1, 0] = raw[:, 1]
    L[:, 1, 1] = torch.nn.functional.softplus(raw[:, 2]) + EPS
    cov = L @ L.transpose(-1, -2)
    out = []
    for i, n in enumerate((f.M, f.N)):
        std = torch.sqrt(torch.clamp(cov[:, i, i], min=1e-8))
        centre, half = (mu[:, i] + 1.0) * 0.5 * (n - 1), SIGMA * std * 0.5 * max(n - 1, 1)
        lo = torch.floor(centre - half).to(torch.int64).clamp_(0, n - 1)
        hi = torch.ceil(centre + half).to(torch.int64).clamp_(0, n - 1)
        t_n = min(t, n)
        out += [lo // t_n, hi // t_n]
    return [v.to(DEVICE) for v in out]


def _exact_field(case, f, mu, grad):
    """(delta [M, N], moments [K, 6] or None) of one field in float64."""
    M, N, K = f.M, f.N, f.K
    tr, tc = min(case["tile"], M), min(case["tile"], N)
    r0, r1, c0, c1 = _rectangles(case, f, mu)
    R, C = -(-M // tr), -(-N // tc)
    mu, raw, amp = mu.detach().double(), f.chol_raw.detach().double(), f.amp.detach().double()[:, 0]
    l11, l21, l22 = (torch.nn.functional.softplus(raw[:, 0]) + EPS, raw[:, 1],
                     torch.nn.functional.softplus(raw[:, 2]) + EPS)
    scale = amp / (2 * math.pi * l11 * l22) if case["normalize"] else amp
    count = (r1 - r0 + 1) * (c1 - c0 + 1)
    gid = torch.repeat_interleave(torch.arange(K, device=DEVICE), count)
    local = torch.arange(gid.numel(), device=DEVICE) - torch.repeat_interleave(torch.cumsum(count, 0) - count, count)
    width = (c1 - c0 + 1)[gid]
    row, col = r0[gid] + local // width, c0[gid] + local % width
    # tiles as rows of elements, past the matrix's edges with zero gradient
    xs, ys = torch.zeros(R * tr, device=DEVICE).double(), torch.zeros(C * tc, device=DEVICE).double()
    xs[:M], ys[:N] = f.row_coords.double(), f.col_coords.double()
    xs, ys = xs.view(R, tr), ys.view(C, tc)
    delta = torch.zeros(R * C, tr * tc, device=DEVICE, dtype=torch.float64)
    tiles = moments = None
    if grad is not None:
        whole = torch.zeros(R * tr, C * tc, device=DEVICE, dtype=torch.float64)
        whole[:M, :N] = grad.view(M, N)
        tiles = whole.view(R, tr, C, tc).permute(0, 2, 1, 3).reshape(R * C, tr * tc)
        moments = torch.zeros(K, 6, device=DEVICE, dtype=torch.float64)
    step = max(1, (1 << 24) // (tr * tc))
    for a in range(0, gid.numel(), step):
        g, i, j = gid[a:a + step], row[a:a + step], col[a:a + step]
        n = g.numel()
        dx = xs[i] - mu[g, 0, None]
        dy = ys[j] - mu[g, 1, None]
        u = dx / l11[g, None]
        v = (dy[:, None, :] - (l21[g, None] * u)[:, :, None]) / l22[g, None, None]
        q = u.square()[:, :, None] + v.square()
        e = torch.exp(-0.5 * (q if case["clamp"] is None else q.clamp(max=case["clamp"])))
        delta.index_add_(0, i * C + j, (scale[g, None, None] * e).view(n, -1))
        if tiles is not None:
            e = e * tiles[i * C + j].view(n, tr, tc)
            m0, m1, m2 = e.sum(2), (e * dy[:, None, :]).sum(2), (e * dy.square()[:, None, :]).sum(2)
            moments.index_add_(0, g, torch.stack((m0.sum(1), (dx * m0).sum(1), m1.sum(1), (dx.square() * m0).sum(1),
                                                  (dx * m1).sum(1), m2.sum(1)), dim=-1))
    delta = delta.view(R, C, tr, tc).permute(0, 2, 1, 3).reshape(R * tr, C * tc)[:M, :N]
    return delta.contiguous(), moments


def _exact_grads(case, f, mu, moments):
    """(d_mu, d_chol_raw, d_amp) in float64: the chain rule from the moments sum(g e [1, dx, dy, dx^2, dx dy, dy^2])."""
    with torch.enable_grad():
        mu, raw, amp = (t.detach().double().requires_grad_(True) for t in (mu, f.chol_raw, f.amp))
        l11, l21, l22 = (torch.nn.functional.softplus(raw[:, 0]) + EPS, raw[:, 1],
                         torch.nn.functional.softplus(raw[:, 2]) + EPS)
        norm = 1.0 / (2 * math.pi * l11 * l22) if case["normalize"] else torch.ones_like(l11)
        # the inverse covariance [[a, b], [b, c]]
        c = 1.0 / l22.square()
        b = -l21 / (l11 * l22.square())
        a = 1.0 / l11.square() + (l21 / (l11 * l22)).square()
        s0, s1, s2, s3, s4, s5 = moments.unbind(1)
        w = (amp[:, 0] * norm).detach()
        loss = (amp[:, 0] * norm * s0).sum() - 0.5 * (w * (a * s3 + 2 * b * s4 + c * s5)).sum()
        a, b, c = a.detach(), b.detach(), c.detach()
        loss = loss + (w * (mu[:, 0] * (a * s1 + b * s2) + mu[:, 1] * (b * s1 + c * s2))).sum()
        return torch.autograd.grad(loss, (mu, raw, amp))


def exact(case, seed):
    fields, m = _inputs(case, seed)
    deltas, grads = [], []
    for k, f in enumerate(fields):
        mu = f.mu if m is None else torch.tanh(f.mu_raw)
        grad = f.grad
        if m is not None:
            grad = (m.gs[k].double().T @ m.xs[k].double()).reshape(-1)
        delta, moments = _exact_field(case, f, mu, grad)
        deltas.append(delta)
        if grad is not None:
            d = list(_exact_grads(case, f, mu, moments))
            if m is not None:
                d[0] = d[0] * (1.0 - torch.tanh(f.mu_raw.double()).square())
            grads.append(d)
    if case["kind"] == "render":
        return dict(deltas=[d.reshape(-1) for d in deltas])
    if case["kind"] == "batch":
        return dict(deltas=[d.reshape(-1) for d in deltas], grads=torch.cat([t.reshape(-1) for d in grads for t in d]))
    if case["kind"] == "model":
        ys = [x.double() @ (w.double() + d).T for x, w, d in zip(m.xs, m.weights, deltas)]
        return dict(ys=ys, grads=[t for d in grads for t in d])
    out = dict(delta=deltas[0].reshape(-1), d_mu=grads[0][0], d_chol_raw=grads[0][1], d_amp=grads[0][2])
    if case["kind"] != "train":
        out.update(tile_ptr=None)
    return out
