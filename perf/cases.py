"""Workloads of the ScatCov engine: what its users run, through the public entry points.

A case is a dict of plain values: `kind` (which call sequence), `precision`, `nside`, `j`, `batch` and
the options of the kind.  `prepare` makes what a program holds before the call (the engine or ensemble,
maps on the device or the host, target statistics), `run` is one pass, `work` the bytes and operations
the pass cannot do without, and `exact` the same outputs in 64 bits from a plain torch model of the
statistics (tap gathers, autograd), independent of the library.

Maps follow the benchmark's lognormal recipe: a coarse N(0, 1) field copied to its NESTED children plus
N(0, 0.1^2) per pixel, exponentiated, mean removed.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "stl-dev-mpi_amd"))

L = 4          # orientations
KSZ = 5        # kernel size
SLOTS = 44.1   # distinct cells a convolution row reads, mean
DEC_ROW = 30.0  # fine pixels a decimation row reads, mean


# ---------------------------------------------------------------------------------------------
# The cases

def listed():
    return [
        # One small map in double precision, the reference's validation size: the call of a quick look
        # or a unit test, where launches and latency count.
        {"name": "map64_fp64", "kind": "eval", "precision": "fp64", "nside": 64, "j": 5, "batch": 1},
        # A medium map at the default precision: synthesis of one nside-256 target.
        {"name": "map256_fp64", "kind": "eval", "precision": "fp64", "nside": 256, "j": 7, "batch": 1},
        # A differentiable layer in a training step: an odd batch of float32 maps through the torch layer,
        # statistics as real pairs, the gradient back in float32.
        {"name": "layer128x5_mixed", "kind": "layer", "precision": "mixed", "nside": 128, "j": 6, "batch": 5},
        # The drop-in use of the reference binding: numpy maps in, numpy gradients out, four members.
        {"name": "host128x4_fp64", "kind": "host", "precision": "fp64", "nside": 128, "j": 6, "batch": 4},
        # Maps of uneven nside evaluated together (the benchmark's ensemble).
        {"name": "ensemble_mixed", "kind": "ensemble", "precision": "mixed", "groups": "128x8,256x4,512x2"},
        # Cut-sky statistics: averages over three overlapping latitude masks.
        {"name": "masks256x2_fp64", "kind": "masks", "precision": "fp64", "nside": 256, "j": 7, "batch": 2,
         "masks": 3},
        # Cross statistics of a pair of maps.
        {"name": "cross256_fp64", "kind": "cross", "precision": "fp64", "nside": 256, "j": 7, "batch": 1},
        # Target statistics with the variances that make the ergodic weights (stl-stats, the start of
        # stl-synth): a forward only, with second moments.
        {"name": "moments512_mixed", "kind": "moments", "precision": "mixed", "nside": 512, "j": 8, "batch": 1},
        # A short device L-BFGS synthesis of an ensemble of four members against one target.
        {"name": "synth128x4_fp64", "kind": "synth", "precision": "fp64", "nside": 128, "j": 6, "batch": 4,
         "iters": 4},
        # The benchmark's own workload: one map at nside 1024, mixed precision.
        {"name": "map1024_mixed", "kind": "eval", "precision": "mixed", "nside": 1024, "j": 9, "batch": 1},
        # The same map at the default precision.
        {"name": "map1024_fp64", "kind": "eval", "precision": "fp64", "nside": 1024, "j": 9, "batch": 1},
        # The largest map the benchmark runs.
        {"name": "map2048_mixed", "kind": "eval", "precision": "mixed", "nside": 2048, "j": 10, "batch": 1},
    ]


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval", "layer", "host", "ensemble", "masks", "cross", "moments", "synth"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "ensemble":
        orders = rng.sample([5, 6, 7, 8, 9], rng.randint(2, 3))
        return {"kind": kind, "precision": precision,
                "groups": ",".join("%dx%d" % (1 << o, rng.randint(1, max(1, min(9, 1 << (18 - 2 * o + 3)))))
                                   for o in sorted(orders))}
    top = {"eval": 10, "layer": 9, "host": 8, "masks": 9, "cross": 9, "moments": 10, "synth": 8}[kind]
    order = rng.randint(5, top)
    room = 4 << (2 * (top - order))  # maps that cost about what four do at the top of the range
    batch = min(int(math.exp(rng.uniform(0.0, math.log(room + 0.99)))), 11) if order < top else rng.randint(1, 2)
    j = rng.randint(max(2, order - 3), order - 1)
    if kind == "eval" and order == top:
        batch, j = 1, rng.randint(3, order - 2)  # with every scale it is a listed case
    case = {"kind": kind, "precision": precision, "nside": 1 << order, "j": j, "batch": batch}
    if kind == "masks":
        case["masks"] = rng.randint(1, 7)
    if kind == "synth":
        # At the default precision: the search's path is then the method's, not the rounding's.
        case.update(precision="fp64", iters=rng.randint(2, 4))
    return case


# ---------------------------------------------------------------------------------------------
# Inputs

def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def lognormal(nside, count, seed, base=32, sigma=0.1):
    """float64 [count, 12 nside^2] maps of the benchmark's recipe, made on the device from the seed."""
    gen = torch.Generator(device=device()).manual_seed(seed)
    base = min(base, nside // 2)
    g = torch.randn(count, 12 * base * base, dtype=torch.float64, device=device(), generator=gen)
    g = g.repeat_interleave((nside // base) ** 2, dim=1)
    g = g + sigma * torch.randn(g.shape, dtype=torch.float64, device=device(), generator=gen)
    x = torch.exp(0.5 * g)
    return x - x.mean(dim=1, keepdim=True)


def white(nside, count, seed):
    gen = torch.Generator(device=device()).manual_seed(seed)
    return torch.randn(count, 12 * nside * nside, dtype=torch.float64, device=device(), generator=gen)


def maps_of(case, seed):
    """The maps and the target maps of a case (pairs for the cross statistics)."""
    count = case["batch"] * (2 if case["kind"] == "cross" else 1)
    x = lognormal(case["nside"], count, 2 * seed)
    t = lognormal(case["nside"], count, 2 * seed + 1)
    if case["kind"] == "cross":
        shape = (case["batch"], 2, -1)
        # Correlated channels, as two observations of one sky.
        x, t = (torch.stack([m[:, 0], 0.6 * m[:, 0] + 0.8 * m[:, 1]], dim=1)
                for m in (x.reshape(shape), t.reshape(shape)))
    return x, t


def groups_of(case):
    return [tuple(int(v) for v in g.split("x")) for g in case["groups"].split(",")]


def default_j(nside):
    return nside.bit_length() - 2


def group_maps(case, seed):
    groups = groups_of(case)
    return ([lognormal(n, b, 100 * seed + g) for g, (n, b) in enumerate(groups)],
            [lognormal(n, b, 100 * seed + 50 + g) for g, (n, b) in enumerate(groups)])


def latitude_masks(nside, count):
    """`count` masks: the pixels further than a cut from the equator, and one hemisphere in every third."""
    z = centres(nside)[0].cos()
    out = []
    for k in range(count):
        keep = z.abs() > 0.15 + 0.6 * k / max(count, 2)
        if k % 3 == 2:
            keep = keep & (z > 0)
        out.append(torch.nonzero(keep).reshape(-1).cpu().numpy())
    return out


# ---------------------------------------------------------------------------------------------
# The entry points

def prepare(case, seed):
    from stl_port import NativeEngine, NativeEnsemble, ergodic_weights
    from stl_port.torch_fn import Stats

    kind = case["kind"]
    if kind == "ensemble":
        x, t = group_maps(case, seed)
        ens = NativeEnsemble(groups_of(case), precision=case["precision"])
        return {"kind": kind, "engine": ens, "x": x, "target": ens.forward_device(t),
                "grad": [torch.empty_like(v) for v in x]}
    options = {"cross": True} if kind == "cross" else {}
    if kind == "masks":
        options["masks"] = latitude_masks(case["nside"], case["masks"])
    eng = NativeEngine(case["nside"], case["j"], batch=case["batch"], precision=case["precision"], **options)
    state = {"kind": kind, "engine": eng, "generation": 0}
    x, t = maps_of(case, seed)
    if kind == "moments":
        state["x"] = x
    elif kind == "layer":
        state.update(x=x.float().requires_grad_(), stats=Stats(eng))
        state["target"] = state["stats"](t.float()).detach()
    elif kind == "host":
        state.update(x=x.cpu().numpy(), target=eng.forward(t.cpu().numpy())[0])
    elif kind == "synth":
        target, var = eng.forward_device(t, moments=True)
        state.update(x0=white(case["nside"], case["batch"], 3 * seed), target=target.mean(axis=0),
                     weights=ergodic_weights(eng.native_pixels(), var.mean(axis=0)), iters=case["iters"])
    else:
        state.update(x=x, target=eng.forward_device(t)[0], grad=torch.empty_like(x))
    return state


def run(state):
    kind, eng = state["kind"], state["engine"]
    if kind == "ensemble":
        values = eng.forward_device(state["x"])
        eng.vjp_device([2.0 * (v - t) for v, t in zip(values, state["target"])], state["grad"])
        return {"values": values, "grad": state["grad"]}
    if kind == "layer":
        x = state["x"]
        x.grad = None
        stats = state["stats"](x)
        (stats - state["target"]).square().sum().backward()
        return {"values": stats.detach(), "grad": x.grad}
    if kind == "synth":
        x = state["x0"].clone()
        losses = eng.synthesize(x, state["target"], weights=state["weights"], max_iter=state["iters"], ensemble=True)
        return {"losses": losses, "x": x}
    state["generation"] += 1
    gen = state["generation"]
    if kind == "moments":
        values, variance = eng.forward_device(state["x"], generation=gen, moments=True)
        return {"values": values, "variance": variance}
    if kind == "host":
        values, _ = eng.forward(state["x"], generation=gen)
        return {"values": values, "grad": eng.vjp(2.0 * (values - state["target"]), generation=gen)}
    values, _ = eng.forward_device(state["x"], generation=gen)
    eng.vjp_device(2.0 * (values - state["target"]), state["grad"], generation=gen)
    return {"values": values, "grad": state["grad"]}


def work(case):
    """Bytes: maps in, gradients out, and every stored operator once (the convolution's rows of two of the
    twelve faces, which the sphere's symmetries leave, 8 values a slot; a decimation's of three faces).
    Operations: the slots' products forward and (with a gradient) reverse, the Gram products and their reverse."""
    if case["kind"] == "ensemble":
        parts = [work({"kind": "eval", "precision": case["precision"], "nside": n, "j": default_j(n), "batch": b})
                 for n, b in groups_of(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    size = 8 if case["precision"] == "fp64" else 4
    backward = case["kind"] != "moments"
    pairs = 2 if case["kind"] == "cross" else 1
    rows = case["batch"] * pairs
    io = 4 if case["kind"] == "layer" else 8
    top = 12 * case["nside"] ** 2
    bytes_, flops = rows * top * io * (2 if backward else 1), 0.0
    for n in range(case["j"]):
        N, K = top >> (2 * n), 4 * n + 5
        bytes_ += N / 6 * SLOTS * 2 * L * size + (N / 16 * DEC_ROW * size if n + 1 < case["j"] else 0)
        conv = N * rows * SLOTS * 2 * L * 2 * (1 + L * (n + 1))
        gram = N * case["batch"] * L * K * K * (8 if pairs == 2 else 4)
        flops += conv * (2 if backward else 1) + gram + (N * rows * L * K * K * 8 if backward else 0)
        flops += gram / 2 if case["kind"] == "moments" else 0
    passes = case.get("iters", 1)  # at least one evaluation an iteration; the operators are read in each
    return {"bytes": float(bytes_ * passes), "flops": float(flops * passes)}


# ---------------------------------------------------------------------------------------------
# The same outputs in 64 bits: the statistics as plain torch, gradients by autograd

JRLL = (2, 2, 2, 2, 3, 3, 3, 3, 4, 4, 4, 4)
JPLL = (1, 3, 5, 7, 0, 2, 4, 6, 1, 3, 5, 7)


def longs(v):
    return torch.tensor(v, dtype=torch.int64, device=device())


def interleave(x, y):
    out = torch.zeros_like(x)
    for b in range(14):
        out |= (((x >> b) & 1) << (2 * b)) | (((y >> b) & 1) << (2 * b + 1))
    return out


def face_xy(pix, nside):
    """In-face coordinates and face of NESTED ids."""
    loc = pix % (nside * nside)
    x, y = torch.zeros_like(pix), torch.zeros_like(pix)
    for b in range(14):
        x |= ((loc >> (2 * b)) & 1) << b
        y |= ((loc >> (2 * b + 1)) & 1) << b
    return x, y, pix // (nside * nside)


def centres(nside, pix=None):
    """theta, phi of NESTED pixel centres, and whether they lie south of the equator."""
    pix = torch.arange(12 * nside * nside, device=device()) if pix is None else pix
    x, y, face = face_xy(pix, nside)
    jr = longs(JRLL)[face] * nside - x - y - 1
    north, south = jr < nside, jr > 3 * nside
    nr = torch.where(north, jr, torch.where(south, 4 * nside - jr, torch.full_like(jr, nside)))
    shift = torch.where(north | south, torch.zeros_like(jr), (jr - nside) & 1)
    t = nr.double() ** 2 / (3.0 * nside * nside)
    cap = torch.atan2((t * (2.0 - t)).sqrt(), 1.0 - t)
    belt = torch.acos(((2.0 * nside - jr.double()) * (2.0 / (3.0 * nside))).clamp(-1.0, 1.0))
    theta = torch.where(north, cap, torch.where(south, math.pi - cap, belt))
    jp = (longs(JPLL)[face] * nr + x - y + 1 + shift) // 2
    jp = torch.where(jp > 4 * nr, jp - 4 * nr, jp)
    jp = torch.where(jp < 1, jp + 4 * nr, jp)
    phi = (jp.double() - 0.5 * (shift.double() + 1.0)) * (0.5 * math.pi / nr.double())
    return theta, phi, jr > 2 * nside


def isqrt(v):
    r = v.double().sqrt().long()
    r = torch.where(r * r > v, r - 1, r)
    return torch.where((r + 1) * (r + 1) <= v, r + 1, r)


def ring_to_nest(pix, nside):
    npix, ncap, nl2 = 12 * nside * nside, 2 * nside * (nside - 1), 2 * nside
    zero = torch.zeros_like(pix)
    # north cap
    a = (1 + isqrt(1 + 2 * pix)) >> 1
    pa = pix + 1 - 2 * a * (a - 1)
    # belt
    ip = pix - ncap
    q = torch.div(ip, 4 * nside, rounding_mode="floor")
    b = q + nside
    pb = ip - q * 4 * nside + 1
    ire = b - nside + 1
    irm = nl2 + 2 - ire
    ifm = torch.div(pb - torch.div(ire, 2, rounding_mode="floor") + nside - 1, nside, rounding_mode="floor")
    ifp = torch.div(pb - torch.div(irm, 2, rounding_mode="floor") + nside - 1, nside, rounding_mode="floor")
    fb = torch.where(ifp == ifm, ifp | 4, torch.where(ifp < ifm, ifp, ifm + 8))
    # south cap
    ips = npix - pix
    c = (1 + isqrt((2 * ips - 1).clamp(min=0))) >> 1
    pc = 4 * c + 1 - (ips - 2 * c * (c - 1))
    north, south = pix < ncap, pix >= npix - ncap
    pick = lambda u, v, w: torch.where(north, u, torch.where(south, w, v))  # noqa: E731
    ring = pick(a, b, 2 * nl2 - c)
    phi = pick(pa, pb, pc)
    nr = pick(a, torch.full_like(pix, nside), c)
    face = pick((pa - 1) // a.clamp(min=1), fb, 8 + (pc - 1) // c.clamp(min=1))
    shift = pick(zero, (b + nside) & 1, zero)
    irt = ring - longs(JRLL)[face] * nside + 1
    ipt = 2 * phi - longs(JPLL)[face] * nr - shift - 1
    ipt = torch.where(ipt >= nl2, ipt - 8 * nside, ipt)
    return interleave((ipt - irt) >> 1, (-ipt - irt) >> 1) + face * nside * nside


def ring_pair(phi, ring, nside):
    """The two pixels of a ring around phi, their weights and the ring's colatitude."""
    mirrored = ring > 2 * nside
    r = torch.where(mirrored, 4 * nside - ring, ring)
    cap = r < nside
    t = r.double() ** 2 / (3.0 * nside * nside)
    theta = torch.where(cap, torch.atan2((t * (2.0 - t)).clamp(min=0).sqrt(), 1.0 - t),
                        torch.acos(((2 * nside - r).double() * (2.0 / (3.0 * nside))).clamp(-1.0, 1.0)))
    count = torch.where(cap, 4 * r, torch.full_like(r, 4 * nside))
    half = torch.where(cap | (((r - nside) & 1) == 0), 0.5, 0.0).double()
    start = torch.where(cap, 2 * r * (r - 1), 2 * nside * (nside - 1) + (r - nside) * 4 * nside)
    theta = torch.where(mirrored, math.pi - theta, theta)
    start = torch.where(mirrored, 12 * nside * nside - start - count, start)
    step = 2.0 * math.pi / count.double()
    i1 = torch.floor(phi / step - half)
    w = (phi - (i1 + half) * step) / step
    i1 = i1.long()
    i2 = i1 + 1
    i1 = torch.where(i1 < 0, i1 + count, i1)
    i2 = torch.where(i2 >= count, i2 - count, i2)
    return start + i1, start + i2, 1.0 - w, w, theta


def interpolate(theta, phi, nside):
    """Bilinear interpolation on the ring scheme: 4 NESTED pixels and weights a direction."""
    z = theta.cos()
    az = z.abs()
    polar = torch.trunc(nside * (3.0 * (1.0 - az)).clamp(min=0).sqrt()).long()
    ring = torch.where(az <= 2.0 / 3.0, torch.trunc(nside * (2.0 - 1.5 * z)).long(),
                       torch.where(z > 0, polar, 4 * nside - polar - 1))
    below = ring + 1
    p0, p1, w0, w1, t1 = ring_pair(phi, ring.clamp(min=1), nside)
    p2, p3, w2, w3, t2 = ring_pair(phi, below.clamp(max=4 * nside - 1), nside)
    north, south = ring == 0, below == 4 * nside
    f = (theta - t1) / torch.where(t2 == t1, torch.ones_like(t1), t2 - t1)
    fn, fs = theta / t2, (theta - t1) / (math.pi - t1)
    qn, qs = 0.25 * (1.0 - fn), 0.25 * fs
    pick = lambda a, b, c: torch.where(north, a, torch.where(south, c, b))  # noqa: E731
    top = 12 * nside * nside - 4
    pix = [pick((p2 + 2) & 3, p0, p0), pick((p3 + 2) & 3, p1, p1), pick(p2, p2, ((p0 + 2) & 3) + top),
           pick(p3, p3, ((p1 + 2) & 3) + top)]
    wgt = [pick(qn, w0 * (1 - f), w0 * (1 - fs) + qs), pick(qn, w1 * (1 - f), w1 * (1 - fs) + qs),
           pick(w2 * fn + qn, w2 * f, qs), pick(w3 * fn + qn, w3 * f, qs)]
    return [ring_to_nest(p, nside) for p in pix], wgt


def kernel():
    """Real and imaginary weights of the 25 taps (zero mean, unit l1 norm, rounded to 32 bits)."""
    taps = [(j - KSZ // 2, i - KSZ // 2) for i in range(KSZ) for j in range(KSZ)]
    k = np.array([complex(math.cos(0.5 * math.pi * x), math.sin(0.5 * math.pi * x)) * math.exp(-0.5 * (x * x + y * y))
                  for x, y in taps])
    k = k - k.mean()
    k = k / np.abs(k).sum()
    return taps, k.real.astype(np.float32).astype(float), k.imag.astype(np.float32).astype(float)


class Convolution:
    """The oriented wavelets of one level: 25 taps on each pixel's tangent plane, turned by the gauge."""

    def __init__(self, nside):
        self.N = 12 * nside * nside
        taps, self.re, self.im = kernel()
        size = (L, KSZ * KSZ, 4, self.N)
        self.pos = torch.empty(size, dtype=torch.int32, device=device())
        self.wgt = torch.empty(size, dtype=torch.float64, device=device())
        alpha = math.sqrt(4.0 * math.pi / self.N)
        for lo in range(0, self.N, 1 << 21):
            pix = torch.arange(lo, min(self.N, lo + (1 << 21)), device=device())
            theta, phi, south = centres(nside, pix)
            ct, st, cp, sp = theta.cos(), theta.sin(), phi.cos(), phi.sin()
            et, ep, n = (cp * ct, sp * ct, -st), (-sp, cp, torch.zeros_like(sp)), (cp * st, sp * st, ct)
            for g in range(L):
                turn = torch.where(south, phi - g * math.pi / L, -phi + g * math.pi / L)
                ca, sa = turn.cos(), turn.sin()
                for t, (x, y) in enumerate(taps):
                    d, a = alpha * math.hypot(x, y), math.atan2(y, x)
                    vx, vy, vz = math.sin(d) * math.cos(a), math.sin(d) * math.sin(a), math.cos(d)
                    u, v = vx * ca - vy * sa, vx * sa + vy * ca
                    w = [u * et[i] + v * ep[i] + vz * n[i] for i in range(3)]
                    # Twice: a tiny negative longitude first becomes 2 pi, then 0.
                    lon = torch.atan2(w[1], w[0]).remainder(2.0 * math.pi).remainder(2.0 * math.pi)
                    p, q = interpolate(torch.acos(w[2].clamp(-1.0, 1.0)), lon, nside)
                    total = q[0] + q[1] + q[2] + q[3]
                    for k in range(4):
                        self.pos[g, t, k, lo:lo + pix.numel()] = p[k].int()
                        self.wgt[g, t, k, lo:lo + pix.numel()] = q[k] / total

    def forward(self, x):
        y = torch.zeros(x.shape[0], L, self.N, 2, dtype=torch.float64, device=x.device)
        for g in range(L):
            for t in range(KSZ * KSZ):
                v = 0.0
                for k in range(4):
                    v = v + x.index_select(1, self.pos[g, t, k]) * self.wgt[g, t, k]
                y[:, g, :, 0] += self.re[t] * v
                y[:, g, :, 1] += self.im[t] * v
        return y

    def adjoint(self, gy):
        gx = torch.zeros(gy.shape[0], self.N, dtype=torch.float64, device=gy.device)
        for g in range(L):
            for t in range(KSZ * KSZ):
                v = self.re[t] * gy[:, g, :, 0] + self.im[t] * gy[:, g, :, 1]
                for k in range(4):
                    gx.index_add_(1, self.pos[g, t, k], v * self.wgt[g, t, k])
        return gx


# Neighbouring face of a face by direction 4 + dx + 3 dy, and how its coordinates turn.
NEXT_FACE = ((8, 9, 10, 11, -1, -1, -1, -1, 10, 11, 8, 9), (5, 6, 7, 4, 8, 9, 10, 11, 9, 10, 11, 8),
             (-1, -1, -1, -1, 5, 6, 7, 4, -1, -1, -1, -1), (4, 5, 6, 7, 11, 8, 9, 10, 11, 8, 9, 10),
             (0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11), (1, 2, 3, 0, 0, 1, 2, 3, 5, 6, 7, 4),
             (-1, -1, -1, -1, 7, 4, 5, 6, -1, -1, -1, -1), (3, 0, 1, 2, 3, 0, 1, 2, 4, 5, 6, 7),
             (2, 3, 0, 1, -1, -1, -1, -1, 0, 1, 2, 3))
NEXT_TURN = ((0, 0, 3), (0, 0, 6), (0, 0, 0), (0, 0, 5), (0, 0, 0), (5, 0, 0), (0, 0, 0), (6, 0, 0), (3, 0, 0))


def neighbour(x, y, face, nside):
    """NESTED id at (x, y) of a face's frame continued over its edges, -1 where three faces meet."""
    step = 4 + (x >= nside).long() - (x < 0).long() + 3 * ((y >= nside).long() - (y < 0).long())
    x, y = x % nside, y % nside
    f, turn = longs(NEXT_FACE)[step, face], longs(NEXT_TURN)[step, face // 4]
    x = torch.where((turn & 1) > 0, nside - 1 - x, x)
    y = torch.where((turn & 2) > 0, nside - 1 - y, y)
    x, y = torch.where((turn & 4) > 0, y, x), torch.where((turn & 4) > 0, x, y)
    return torch.where(f < 0, f, interleave(x, y) + f * nside * nside)


class Decimation:
    """Gaussian cones of the fine pixels around each coarse one, rows of unit sum."""

    def __init__(self, nside):
        self.N, coarse = 12 * nside * nside, nside // 2
        c = torch.arange(self.N // 4, device=device())
        x, y, face = face_xy(c, coarse)
        tc, pc, _ = centres(coarse)
        radius = 3.0 * math.sqrt(4.0 * math.pi / self.N)
        self.pos, self.wgt = [], []
        if coarse >= 4:
            for dy in range(-2, 3):
                for dx in range(-2, 3):
                    v = neighbour(x + dx, y + dy, face, coarse)
                    for child in range(4):
                        self.pos.append(torch.where(v < 0, v, 4 * v + child))
        else:
            self.pos = [torch.full_like(c, p) for p in range(self.N)]
        tf, pf, _ = centres(nside)
        for p in self.pos:
            q = p.clamp(min=0)
            a = (0.5 * (tf[q] - tc)).sin() ** 2 + tc.sin() * tf[q].sin() * (0.5 * (pf[q] - pc)).sin() ** 2
            gamma = 2.0 * torch.asin(a.clamp(0.0, 1.0).sqrt())
            w = torch.exp(-0.5 * (gamma / (0.5 * radius)) ** 2)
            self.wgt.append(torch.where((p < 0) | (gamma > radius), torch.zeros_like(w), w))
        total = sum(self.wgt)
        self.wgt = [w / total for w in self.wgt]
        self.pos = [p.clamp(min=0).int() for p in self.pos]

    def forward(self, x):
        return sum(x.index_select(1, p) * w for p, w in zip(self.pos, self.wgt))

    def adjoint(self, gy):
        gx = torch.zeros(gy.shape[0], self.N, dtype=torch.float64, device=gy.device)
        for p, w in zip(self.pos, self.wgt):
            gx.index_add_(1, p, gy * w)
        return gx


class Apply(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, op):
        ctx.op = op
        return op.forward(x)

    @staticmethod
    def backward(ctx, gy):
        return ctx.op.adjoint(gy.contiguous()), None


class Statistics:
    """S(x) of maps [B, C, N]: the plan's coefficients, and the spatial variance of their terms."""

    def __init__(self, nside, j, masks=None, cross=False):
        self.j, self.cross = j, cross
        self.conv = [Convolution(nside >> n) for n in range(j)]
        self.dec = [Decimation(nside >> n) for n in range(j - 1)]
        self.masks = [None]
        if masks is not None:
            m = torch.zeros(len(masks), 12 * nside * nside, dtype=torch.float64, device=device())
            for k, ids in enumerate(masks):
                m[k, torch.from_numpy(ids).to(device())] = 1.0
            self.masks = [m]
            for _ in range(1, j):
                self.masks.append(self.masks[-1].reshape(len(masks), -1, 4).amax(dim=2))

    def mean(self, terms, n):
        """Means of terms [..., N] over the sky, or over each mask: [..., K]."""
        if self.masks[0] is None:
            return terms.mean(dim=-1, keepdim=True)
        m = self.masks[n]
        return torch.stack([(terms * m[k]).sum(dim=-1) / m[k].sum() for k in range(m.shape[0])], dim=-1)

    def products(self, a, b, n):
        """Means of a_i conj(b_j), a and b [K', N]: [K', K', K]."""
        if self.masks[0] is None:
            return (a @ b.conj().T.contiguous() / a.shape[-1]).unsqueeze(-1)
        m = self.masks[n]
        return torch.stack([(a * m[k]) @ b.conj().T.contiguous() / m[k].sum() for k in range(m.shape[0])], dim=-1)

    def entries(self, n):
        """Rows (l3, i, j) of the level's S3 and S4 coefficients, in the plan's order."""
        rows, last = [], 4 * (n + 1)
        for j2 in range(n + 1):
            rows += [(l3, 4 * j2 + l2, last) for l2 in range(L) for l3 in range(L)]
            rows += [(l3, 4 * j1 + l1, 4 * j2 + l2) for j1 in range(j2 + 1) for l1 in range(L) for l2 in range(L)
                     for l3 in range(L)]
        return longs(rows).T

    def __call__(self, maps, moments=False):
        B, C = maps.shape[:2]
        x, moduli = maps.reshape(B * C, -1), []
        out, second = [], []

        def add(terms, sq, n):
            out.append(self.mean(terms, n).unsqueeze(1))
            if moments:
                second.append(self.mean(sq, n).unsqueeze(1))

        if not self.cross:
            add(torch.complex(x, torch.zeros_like(x)), x * x, 0)
            add(torch.complex(x * x, torch.zeros_like(x)), x ** 4, 0)
        for n in range(self.j):
            if n > 0:
                x = Apply.apply(x, self.dec[n - 1])
                moduli = [Apply.apply(m, self.dec[n - 1]) for m in moduli]
            z = torch.view_as_complex(Apply.apply(x, self.conv[n]))  # [BC, L, N]
            moduli.append(z.abs().reshape(B * C * L, -1))
            rows = [torch.view_as_complex(Apply.apply(m, self.conv[n])).reshape(B, C, L, L, -1).transpose(2, 3)
                    for m in moduli]
            zz = z.reshape(B, C, L, -1)
            V = torch.cat(rows + [zz.unsqueeze(3)], dim=3)  # [B, C, l3, K', N]
            if self.cross:
                rn = zz / (zz.abs() + 1e-8).sqrt()
                for terms in (rn[:, 0] * rn[:, 1].conj(), zz[:, 0] * zz[:, 1].conj()):
                    for l in range(L):
                        add(terms[:, l], terms[:, l].abs() ** 2, n)
            else:
                p = zz[:, 0].abs()
                for terms, sq in ((p, p ** 2), (p ** 2, p ** 4)):
                    for l in range(L):
                        add(torch.complex(terms[:, l], torch.zeros_like(terms[:, l])), sq[:, l], n)
            l3, i, k = self.entries(n)
            for a, b in (((0, 1), (1, 0)) if self.cross else ((0, 0),)):
                gram = torch.stack([torch.stack([self.products(V[m, a, l], V[m, b, l], n) for l in range(L)])
                                    for m in range(B)])
                out.append(gram[:, l3, i, k])
                if moments:
                    sq = torch.stack([torch.stack([self.products(V[m, a, l].abs() ** 2, V[m, b, l].abs() ** 2, n)
                                                   for l in range(L)]) for m in range(B)])
                    second.append(sq[:, l3, i, k])
        values = torch.cat(out, dim=1).transpose(1, 2)  # [B, K, coefficients]
        if not moments:
            return values
        return values, (torch.cat(second, dim=1).transpose(1, 2) - values.abs() ** 2).clamp(min=0.0)


def exact_eval(case, maps, target, masks=None):
    """Values and map gradient of sum |S(x) - S(t)|^2."""
    cross = case["kind"] == "cross"
    model = Statistics(case["nside"], case["j"], masks, cross)
    shape = (case["batch"], 2 if cross else 1, -1)
    with torch.no_grad():
        t = model(target.reshape(shape))
    x = maps.reshape(shape).clone().requires_grad_()
    values = model(x)
    (values - t).abs().square().sum().backward()
    return values.detach(), x.grad.reshape(maps.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        if sum(b * n * n for n, b in groups_of(case)) > 1 << 20:
            return None
        values, grads = [], []
        for (n, b), x, t in zip(groups_of(case), *group_maps(case, seed)):
            v, g = exact_eval({"kind": "eval", "nside": n, "j": default_j(n), "batch": b}, x, t)
            values.append(v[:, 0].cpu().numpy())
            grads.append(g)
        return {"values": values, "grad": grads}
    if case["batch"] * (2 if kind == "cross" else 1) * case["nside"] ** 2 > 1 << 19:
        return None
    x, t = maps_of(case, seed)
    if kind == "moments":
        with torch.no_grad():
            values, variance = Statistics(case["nside"], case["j"])(x.reshape(case["batch"], 1, -1), moments=True)
        return {"values": values[:, 0].cpu().numpy(), "variance": variance[:, 0].cpu().numpy()}
    if kind == "synth":
        return exact_synthesis(case, seed, t)
    if kind == "layer":
        values, grad = exact_eval(case, x.float().double(), t.float().double())
        return {"values": torch.view_as_real(values[:, 0].contiguous()), "grad": grad}
    masks = latitude_masks(case["nside"], case["masks"]) if kind == "masks" else None
    values, grad = exact_eval(case, x, t, masks)
    values = (values if kind == "masks" else values[:, 0]).cpu().numpy()
    return {"values": values, "grad": grad.cpu().numpy() if kind == "host" else grad}


def exact_synthesis(case, seed, target_maps):
    """The same L-BFGS with torch's optimiser on the model's loss."""
    model = Statistics(case["nside"], case["j"])
    shape = (case["batch"], 1, -1)
    with torch.no_grad():
        t, var = model(target_maps.reshape(shape), moments=True)
    t, var = t[:, 0].mean(dim=0), var[:, 0].mean(dim=0)
    top = 12 * case["nside"] ** 2
    counts = [top, top]
    for n in range(case["j"]):
        counts += [top >> (2 * n)] * (2 * L + (n + 1) * L * L + (n + 1) * (n + 2) // 2 * L ** 3)
    w = torch.tensor(counts, dtype=torch.float64, device=device()) / var
    w = torch.where(torch.isfinite(w), w, w[torch.isfinite(w)].max()) / w.numel()
    x = white(case["nside"], case["batch"], 3 * seed).requires_grad_()
    losses = []
    search = torch.optim.LBFGS([x], lr=1.0, max_iter=case["iters"], tolerance_grad=1e-12, tolerance_change=1e-15,
                               history_size=10, line_search_fn="strong_wolfe")

    def closure():
        search.zero_grad()
        loss = (w * (model(x.reshape(shape))[:, 0].mean(dim=0) - t).abs().square()).sum()
        loss.backward()
        losses.append(loss.item())
        return loss

    search.step(closure)
    return {"losses": np.array(losses), "x": x.detach()}
