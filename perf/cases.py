"""The work that programs have this library do, as cases that can be timed and compared.

A case names its entry point (`call`), its inputs' distribution and sizes, the opening parameter
theta, and the expansion order and leaf capacity of the solve.  Calls:

  dropin            treecode_potential / treecode_force_mrag on host arrays: FP64 at the library's
                    fixed order / leaf (12 / 512 potential, 24 / 192 force); a solver that was linked
                    against the C library
  float             treecode_potential_float on host float arrays
  context           Context.potential / Context.force with everything in HBM: a solver that keeps its
                    particles on the GPU and solves each step
  host              Context.potential on host arrays at a chosen order / leaf (what a served request does)
  resident          Context.potential_resident: new targets against a tree that is kept
  targets           Context.force_targets: the gradient at arbitrary points

Sources are uniform, half uniform / half Plummer (clustered), 4 or 16 Gaussians, as in the
package's workloads.  Targets of a potential are the sources' own coordinates (m = n) or other
points of the same distribution; force targets are 32x32 blocks.
"""
import importlib
import math

import numpy as np
import torch

tc = importlib.import_module("2d-treecodes_amd")

EPS = 10.0 * np.finfo(np.float64).eps  # the direct sums' regularisation
EXACT_PAIRS = 2.5e11                   # direct sums up to this many pairs (a few seconds)


def listed():
    return [
        # the smallest solves: one thousand vortices / the smallest served force request, where a call
        # is launches, copies and round trips
        dict(name="potential drop-in tiny", kind="potential", call="dropin", src="uniform", n=1000, m=1000,
             theta=0.5, order=12, leaf=512, f32=False),
        dict(name="force drop-in tiny", kind="force", call="dropin", src="gauss4", n=10000, nb=16, theta=0.5,
             order=24, leaf=192, f32=False),
        # a served potential request of middling size, host arrays, odd sizes
        dict(name="potential host served", kind="potential", call="host", src="gauss4", n=31623, m=31623,
             theta=0.7, order=14, leaf=128, f32=True),
        # ordinary device-resident solve at the library's default parameters
        dict(name="potential 64k fp64", kind="potential", call="context", src="uniform", n=65536, m=65536,
             theta=0.5, order=12, leaf=512, f32=False),
        # the float build's users
        dict(name="potential float ragged", kind="potential", call="float", src="uniform", n=200003, m=150001,
             theta=0.5, order=12, leaf=512, f32=True),
        # a field sampled again and again against one set of sources
        dict(name="potential resident", kind="potential", call="resident", src="plummer", n=1 << 20, m=250007,
             theta=0.5, order=10, leaf=128, f32=True),
        # large clustered solves in either precision at the tuned order / leaf
        dict(name="potential 4M fp64", kind="potential", call="context", src="plummer", n=(1 << 22) + 3,
             m=(1 << 22) + 3, theta=0.3, order=9, leaf=64, f32=False),
        dict(name="potential 16M fp32", kind="potential", call="context", src="plummer", n=1 << 24, m=1 << 24,
             theta=0.5, order=9, leaf=128, f32=True),
        # the gradient at scattered points (particle velocities), default parameters
        dict(name="force targets", kind="force", call="targets", src="gauss4", n=200000, m=100003, theta=0.5,
             order=24, leaf=192, f32=False),
        # a flow solver linked against the C library: forces on its blocks, default parameters
        dict(name="force drop-in", kind="force", call="dropin", src="gauss4", n=240000, nb=1000, theta=0.5,
             order=24, leaf=192, f32=False),
        # device-resident force solves: one grid, and blocks of mixed spacing at full size
        dict(name="force 1M fp32", kind="force", call="context", src="gauss4", n=1 << 20, nb=4096, theta=0.5,
             order=8, leaf=64, f32=True),
        dict(name="force 8M fp32", kind="force", call="context", src="gauss16", n=1 << 23, nb=16384, theta=0.5,
             order=8, leaf=128, f32=True),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["dropin", "float", "context", "context", "host", "resident", "targets"])
    kind = {"float": "potential", "host": "potential", "resident": "potential", "targets": "force"}.get(call)
    kind = kind or rng.choice(["potential", "force"])
    theta = rng.choice([0.3, 0.5, 0.7])
    if kind == "potential":
        c = dict(kind=kind, call=call, src=rng.choice(["uniform", "plummer", "gauss4"]),
                 n=_log_size(rng, 1000, 1 << 20 if call in ("dropin", "float", "host") else 1 << 22), theta=theta)
        c["m"] = c["n"] if rng.random() < 0.5 else _log_size(rng, 500, c["n"])
        c["f32"] = call == "float" or (call != "dropin" and rng.random() < 0.6)
        if call in ("dropin", "float") or rng.random() < 0.2:
            c["order"], c["leaf"] = 12, 512
        else:
            c["order"] = {0.3: 8, 0.5: 9, 0.7: 14}[theta] if rng.random() < 0.7 else rng.choice([6, 10, 16, 20])
            c["leaf"] = rng.choice([64, 128, 192, 256])
        return c
    if call == "targets":
        return dict(kind=kind, call=call, src=rng.choice(["uniform", "gauss4"]), n=_log_size(rng, 10000, 1 << 20),
                    m=_log_size(rng, 1000, 200000), theta=theta, order=24, leaf=192, f32=rng.random() < 0.3)
    c = dict(kind=kind, call=call, src=rng.choice(["gauss4", "gauss16"]),
             n=_log_size(rng, 10000, 2000000 if call == "context" else 500000), nb=_log_size(rng, 16, 2048),
             theta=theta, order=24, leaf=192, f32=False)
    if call == "context":
        c["f32"] = rng.random() < 0.6
        c["order"] = {0.3: 8, 0.5: 8, 0.7: 12}[theta] if rng.random() < 0.7 else rng.choice([9, 16, 24])
        c["leaf"] = rng.choice([32, 64, 128, 192])
    return c


# ---------------------------------------------------------------- inputs
def _uniform(g, n):
    return torch.rand(n, generator=g, device=g.device, dtype=torch.float64)


def _points(src, g, n):
    """n points and strengths of the distribution `src`."""
    if src in ("gauss4", "gauss16"):
        if src == "gauss4":
            cen = torch.tensor([[0.3, 0.3], [0.7, 0.3], [0.3, 0.7], [0.7, 0.7]], dtype=torch.float64, device=g.device)
            sig = torch.full((4,), 0.05, dtype=torch.float64, device=g.device)
        else:
            cen = 0.1 + 0.8 * _uniform(g, 32).reshape(16, 2)
            sig = 0.005 * torch.exp(math.log(10.0) * _uniform(g, 16))
        k = torch.clamp((_uniform(g, n) * len(sig)).long(), max=len(sig) - 1)
        sign = torch.where(_uniform(g, len(sig)) < 0.5, -1.0, 1.0).double()
        d = torch.randn(2, n, generator=g, device=g.device, dtype=torch.float64) * sig[k]
        return cen[k, 0] + d[0], cen[k, 1] + d[1], sign[k] * torch.exp(-(d * d).sum(0) / (2.0 * sig[k] ** 2))
    v = 2.0 * _uniform(g, n) - 1.0
    x, y = _uniform(g, n), _uniform(g, n)
    if src == "plummer":
        nu = n // 2
        got, need = [], n - nu
        while need > 0:
            u, a = _uniform(g, need + need // 16 + 64), 2.0 * math.pi * _uniform(g, need + need // 16 + 64)
            r = 0.02 * torch.sqrt(u / (1.0 - u))
            p = torch.stack([0.5 + r * torch.cos(a), 0.5 + r * torch.sin(a)])
            p = p[:, ((p >= 0.0) & (p <= 1.0)).all(0)][:, :need]
            got.append(p)
            need -= p.shape[1]
        x[nu:], y[nu:] = torch.cat(got, 1)
    return x, y, v


def _blocks(c, g, x, y):
    """Origins and spacings of nb blocks of 32x32 points."""
    nb = c["nb"]
    if c["src"] == "gauss4":  # distinct cells of a 64x64 grid of blocks
        cell = torch.randperm(4096, generator=g, device=g.device)[:nb].sort().values
        s = 32.0 / 2048
        return (cell % 64) * s, (cell // 64) * s, torch.full((nb,), 1.0 / 2048, dtype=torch.float64, device=g.device)
    # the densest cells at three spacings: an eighth to a quarter coarse, half mid, the rest fine
    coarse, mid = min(nb // 4, 1024), min(nb // 2, 4096)
    out = []
    for h, cnt in ((1.0 / 4096, nb - coarse - mid), (1.0 / 2048, mid), (1.0 / 1024, coarse)):
        side, nc = 32 * h, int(round(1.0 / (32 * h)))
        ix, iy = (torch.clamp((p / side).long(), 0, nc - 1) for p in (x, y))
        top = torch.argsort(torch.bincount(iy * nc + ix, minlength=nc * nc), descending=True, stable=True)[:cnt]
        out.append(torch.stack([(top % nc) * side, (top // nc) * side, torch.full_like(top, h, dtype=torch.float64)]))
    return tuple(torch.cat(out, 1))


def _inputs(c, seed):
    """Sources (x, y, v), and targets (x, y) or blocks (x0, y0, h), as float64 tensors."""
    g = torch.Generator(device="cuda" if torch.cuda.is_available() else "cpu")
    g.manual_seed(int(seed))
    s = _points(c["src"], g, c["n"])
    if "nb" in c:
        return s, _blocks(c, g, s[0], s[1])
    if c["m"] == c["n"] and c["kind"] == "potential":
        return s, (s[0].clone(), s[1].clone())
    return s, _points(c["src"], g, c["m"])[:2]


class HbmArray:
    """A tensor as the library takes it: a device address and a length."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = self.t.data_ptr()

    def __len__(self):
        return self.t.numel()


_contexts = {}


def _context(c):
    """The context that a program keeps for its solves with these options."""
    key = (c["kind"], c["f32"], c["order"], c["leaf"])
    if key not in _contexts:
        _contexts[key] = _new_context(c)
    return _contexts[key]


def _new_context(c):
    p = "pot" if c["kind"] == "potential" else "force"
    return tc.Context(precision=tc.FP32 if c["f32"] else tc.FP64, **{p + "_order": c["order"], p + "_leaf": c["leaf"]})


def prepare(case, seed):
    s, t = _inputs(case, seed)
    st = {"case": case}
    if case["call"] in ("dropin", "float", "host"):
        dt = torch.float32 if case["call"] == "float" else torch.float64
        st["in"] = [a.to(dt).cpu().numpy() for a in (*s, *t)]
        if case["call"] == "host":
            st["ctx"] = _context(case)
        return st
    st["in"] = [HbmArray(a) for a in (*s, *t)]
    m = 1024 * case["nb"] if "nb" in case else case["m"]
    st["out"] = [HbmArray(torch.zeros(m, dtype=torch.float64, device="cuda")) for _ in range(1 if case["kind"] == "potential" else 2)]
    torch.cuda.synchronize()
    if case["call"] == "resident":  # the sources are solved once; their tree stays in this context
        st["ctx"] = _new_context(case)
        st["ctx"].potential(case["theta"], *st["in"], out=st["out"][0], device=True)
        st["ctx"].synchronize()
    else:
        st["ctx"] = _context(case)
    return st


def run(state):
    c, a = state["case"], state["in"]
    theta, call = c["theta"], c["call"]
    if call == "dropin":
        return (tc.treecode_potential if c["kind"] == "potential" else tc.treecode_force_mrag)(theta, *a)
    if call == "float":
        return tc.treecode_potential_float(theta, *a)
    ctx = state["ctx"]
    if call == "host":
        return ctx.potential(theta, *a)
    out = state["out"]
    if call == "resident":
        ctx.potential_resident(theta, a[3], a[4], out=out[0], device=True)
    elif call == "targets":
        ctx.force_targets(theta, *a, xr=out[0], yr=out[1], device=True)
    elif c["kind"] == "potential":
        ctx.potential(theta, *a, out=out[0], device=True)
    else:
        ctx.force(theta, *a, xr=out[0], yr=out[1], device=True)
    return [o.t for o in out] if len(out) > 1 else out[0].t


def work(case):
    """Inputs read once and outputs written once; the operations of the interactions that a tree
    with these parameters has for evenly spread points: per level about 22 (0.5 / theta)^2 multipole
    evaluations a target and (0.5 / theta)^2 of about three full leaves of direct pairs."""
    n, p, leaf = case["n"], case["order"], case["leaf"]
    m = 1024 * case["nb"] if "nb" in case else case["m"]
    size = 4 if case["call"] == "float" else 8
    force = case["kind"] == "force"
    src = 0 if case["call"] == "resident" else 3 * n
    tgt = 3 * case["nb"] if "nb" in case else 2 * m
    open_ = (0.5 / case["theta"]) ** 2
    levels = max(0.0, math.log(max(1.0, n / leaf), 4.0) - 1.0)
    pairs = min(float(n), 3.0 * open_ * leaf)
    if "nb" in case:  # far nodes are shared by a brick of 64 targets
        far = 22.0 * open_ * levels * ((4 * p * p + 21 * p) / 64.0)
    else:
        far = 22.0 * open_ * levels * ((16 if force else 10) * p)
    return {"bytes": size * (src + tgt + (2 if force else 1) * m), "flops": m * ((11 if force else 9) * pairs + far)}


# ---------------------------------------------------------------- 64-bit direct sums
def exact(case, seed):
    n = case["n"]
    m = 1024 * case["nb"] if "nb" in case else case["m"]
    if float(n) * m > EXACT_PAIRS:
        return None
    s, t = _inputs(case, seed)
    if case["call"] == "float":
        s, t = ([a.float().double() for a in u] for u in (s, t))
    sx, sy, sv = s
    if "nb" in case:
        i = torch.arange(1024, device=sx.device)
        tx = (t[0][:, None] + (i % 32) * t[2][:, None]).reshape(-1)
        ty = (t[1][:, None] + (i // 32) * t[2][:, None]).reshape(-1)
    else:
        tx, ty = t
    outs = [torch.empty(m, dtype=torch.float64, device=sx.device) for _ in range(2 if case["kind"] == "force" else 1)]
    step = max(1, (1 << 26) // n)
    for k in range(0, m, step):
        dx = tx[k:k + step, None] - sx[None, :]
        dy = ty[k:k + step, None] - sy[None, :]
        r2 = torch.addcmul(dx * dx, dy, dy).add_(EPS)
        if case["kind"] == "potential":
            outs[0][k:k + step] = (r2.log_().mul_(sv)).sum(1) * 0.5
        else:
            f = torch.div(sv, r2)
            outs[0][k:k + step] = dx.mul_(f).sum(1)
            outs[1][k:k + step] = dy.mul_(f).sum(1)
    return outs[0].cpu().numpy() if len(outs) == 1 else [o.cpu().numpy() for o in outs]
