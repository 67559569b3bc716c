"""The work this framework is measured on: line integral convolution calls
through the public entry points, and the equalization that follows them.

A case is a dict of plain values:

  kind "convolve"  one ``rlic_amd.convolve`` call on ROCm tensors, or, with
                   ``where`` = "host", on NumPy arrays (uploaded, computed
                   and downloaded by the call)
  kind "batch"     one ``rlic_amd.batch.convolve_batch`` call on ``fields``
                   fields of uneven sizes, kernels, modes and boundaries
  kind "serve"     ``requests`` requests of mixed types and sizes submitted
                   to a running ``rlic_amd.serve.Server`` and stepped until done
  kind "equalize"  global histogram equalization of a LIC-like image, the
                   post-step an image gets before it is shown

The sizes, kernels and boundary sets are those of the repository's workloads
(``rlic_amd/workloads.py``): 256^2 to 16384^2 single fields, sides of 32 to
2048 in batches, kernels of 17 to 257 taps, 1 to 20 passes.
"""

import math
import random

import numpy as np
import torch

import rlic_amd
from rlic_amd.batch import convolve_batch
from rlic_amd.equalize import equalize_histogram
from rlic_amd.serve import Server

_DTYPES = {"f32": torch.float32, "f64": torch.float64}


# ---------------------------------------------------------------- the cases

def _single(name, ny, nx, dtype, length, iterations=1, *, weights="triangular",
            mode="velocity", bx="closed", by="closed", holes=0, where="device"):
    return dict(name=name, kind="convolve", ny=ny, nx=nx, dtype=dtype, length=length,
                iterations=iterations, weights=weights, mode=mode, bx=bx, by=by, holes=holes,
                where=where)


def listed():
    return [
        # a thumbnail: the smallest calls, launches and host time
        _single("thumb_97x61_f32", 97, 61, "f32", 17),
        # an image of the README example's size and kernel, its field already on the
        # device
        _single("readme_256_f64", 256, 256, "f64", 65, bx="periodic", by="periodic"),
        # the same as the README calls it: NumPy in, NumPy out
        _single("readme_256_f64_host", 256, 256, "f64", 65, bx="periodic", by="periodic",
                where="host"),
        # a figure-sized image of odd sides, several passes, a kernel longer
        # than any staged box, double as NumPy users have it
        _single("odd_1021x1537_f64", 1021, 1537, "f64", 151, 4, by="periodic"),
        # the same in float with holes (masked data: lines end early)
        _single("masked_2111x1500_f32", 2111, 1500, "f32", 201, 3, weights="boxcar",
                bx="periodic", holes=1),
        # the headline field
        _single("plain_4096_f32", 4096, 4096, "f32", 129, 5, weights="gaussian", bx="periodic"),
        # large polarization fields, one pass
        _single("polar_8192_f64", 8192, 8192, "f64", 257, mode="polarization"),
        _single("polar_16384_f32", 16384, 16384, "f32", 257, mode="polarization"),
        # many small fields at once: per-field host work and one launch
        dict(name="batch_64_small", kind="batch", dtype="f32", fields=64, lo=32, hi=256, pick=1),
        # uneven fields of the batch workload
        dict(name="batch_48_uneven", kind="batch", dtype="f32", fields=48, lo=128, hi=2048,
             pick=4),
        # a burst of requests of both types on a running server
        dict(name="serve_24", kind="serve", requests=24, lo=128, hi=2048, pick=5),
        # a LIC image made ready for display
        dict(name="equalize_4096_f32", kind="equalize", ny=4096, nx=4096, dtype="f32", bins=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi):
    """Two log-uniform sides with an aspect ratio of at most 4."""
    while True:
        ny, nx = _log_int(rng, lo, hi), _log_int(rng, lo, hi)
        if 0.25 <= ny / nx <= 4.0:
            return ny, nx


#: No drawn case does more lane-steps (float64 ones counted twice) than the
#: largest listed one.
_MOST_STEPS = 16384 * 16384 * 256


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choices(("device", "host", "batch", "serve", "equalize"), (11, 2, 3, 2, 2))[0]
    dtype = rng.choice(("f32", "f64"))
    if kind == "equalize":
        ny, nx = _sides(rng, 256, 8192)
        return dict(kind="equalize", ny=ny, nx=nx, dtype=dtype, bins=_log_int(rng, 64, 4096))
    if kind == "batch":
        lo, hi = rng.choice(((32, 256), (128, 2048)))
        return dict(kind="batch", dtype=dtype, fields=rng.randint(8, 64), lo=lo, hi=hi,
                    pick=rng.randrange(1 << 20))
    if kind == "serve":
        return dict(kind="serve", requests=rng.randint(8, 32), lo=128, hi=2048,
                    pick=rng.randrange(1 << 20))
    while True:
        ny, nx = _sides(rng, 32, 1024 if kind == "host" else 16384)
        length = rng.randrange(17, 258, 2) if rng.random() < 0.8 else rng.randint(16, 256)
        iterations = rng.choice((1, 1, 1, rng.randint(2, 10)))
        if ny * nx * (length - 1) * iterations * (2 if dtype == "f64" else 1) <= _MOST_STEPS:
            break
    case = _single("", ny, nx, dtype, length, iterations,
                   weights=rng.choice(("triangular", "boxcar", "gaussian")),
                   mode=rng.choice(("velocity", "polarization")),
                   bx=rng.choice(("periodic", "closed")), by=rng.choice(("periodic", "closed")),
                   holes=int(rng.random() < 0.2), where=kind)
    del case["name"]
    return case


# --------------------------------------------------------------- the inputs

def _weights(kind, length):
    if kind == "boxcar":
        return np.ones(length)
    if kind == "gaussian":
        return np.exp(-0.5 * ((np.arange(length) - (length - 1) / 2) / (length / 4)) ** 2)
    return 1 - np.abs(np.linspace(-1, 1, length))


def _modes(rng, ny, nx, device, n=8, kmax=16):
    """A sum of plane waves: wavenumbers 1..kmax, N(0, 1) amplitudes."""
    jj = torch.arange(nx, device=device, dtype=torch.float64) * (2 * math.pi / nx)
    ii = torch.arange(ny, device=device, dtype=torch.float64) * (2 * math.pi / ny)
    rows, cols = [], []
    for _ in range(n):
        kx, ky = rng.randint(1, kmax), rng.randint(1, kmax)
        a, phi = rng.gauss(0, 1), rng.uniform(0, 2 * math.pi)
        # a cos(x + y) = a cos(y) cos(x) - a sin(y) sin(x)
        rows += [a * torch.cos(ky * ii), -a * torch.sin(ky * ii)]
        cols += [torch.cos(kx * jj + phi), torch.sin(kx * jj + phi)]
    return torch.stack(rows, 1) @ torch.stack(cols, 0)


def _field(ny, nx, dtype, mode, seed, device, holes=False):
    """texture, u, v of one field."""
    rng = random.Random(seed)
    gen = torch.Generator(device=device).manual_seed(seed)
    t = _DTYPES[dtype]
    texture = torch.rand((ny, nx), generator=gen, device=device, dtype=t)
    u = _modes(rng, ny, nx, device)
    v = _modes(rng, ny, nx, device)
    if mode == "polarization":  # two half-planes of opposite sense
        u *= 0.3
        u += torch.where(torch.arange(nx, device=device) < nx / 2, -1.0, 1.0)
    u, v = u.to(t), v.to(t)
    if holes:
        ii = torch.arange(ny, device=device)[:, None]
        jj = torch.arange(nx, device=device)[None, :]
        for _ in range(24):
            ci, cj = rng.randrange(ny), rng.randrange(nx)
            r = rng.uniform(0.01, 0.06) * min(ny, nx)
            hole = (ii - ci) ** 2 + (jj - cj) ** 2 < r * r
            u[hole] = math.nan
            v[hole] = math.nan
    return texture, u, v


def _calls(case):
    """The convolve calls a case makes, as "convolve" cases."""
    if case["kind"] == "convolve":
        return [case]
    rng = random.Random(case["pick"])
    n, most = (case["fields"], 10) if case["kind"] == "batch" else (case["requests"], 20)
    calls = []
    for k in range(n):
        ny, nx = _sides(rng, case["lo"], case["hi"])
        dtype = case["dtype"] if case["kind"] == "batch" else ("f32", "f64")[k % 2]
        calls.append(_single("", ny, nx, dtype, rng.randrange(17, 258, 2), rng.randint(1, most),
                             weights=rng.choice(("triangular", "boxcar")),
                             mode=rng.choice(("velocity", "polarization")),
                             bx=rng.choice(("periodic", "closed")),
                             by=rng.choice(("periodic", "closed"))))
    return calls


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _arguments(call, seed, device):
    """The arguments of one convolve call, as tensors on ``device``."""
    texture, u, v = _field(call["ny"], call["nx"], call["dtype"], call["mode"], seed, device,
                           bool(call["holes"]))
    kernel = torch.from_numpy(_weights(call["weights"], call["length"]))
    return (texture, u, v), dict(kernel=kernel.to(device=device, dtype=_DTYPES[call["dtype"]]),
                                 uv_mode=call["mode"],
                                 boundaries={"x": call["bx"], "y": call["by"]},
                                 iterations=call["iterations"])


def _image(case, seed, device):
    """Noise averaged along rows: the value distribution of a LIC image."""
    gen = torch.Generator(device=device).manual_seed(seed)
    x = torch.rand((case["ny"], case["nx"]), generator=gen, device=device,
                   dtype=_DTYPES[case["dtype"]])
    out = x.clone()
    for k in range(1, 8):
        out += x.roll(k, 1)
    return out


def prepare(case, seed):
    device = _device()
    if case["kind"] == "equalize":
        return case, _image(case, seed, device)
    calls = [_arguments(c, seed * 1009 + k, device) for k, c in enumerate(_calls(case))]
    if case["kind"] == "serve":
        return case, (Server(64 << 30), calls)
    if case["kind"] == "batch":
        return case, [dict(texture=t, u=u, v=v, **kw) for (t, u, v), kw in calls]
    args, kw = calls[0]
    if case["where"] == "host":
        args = tuple(a.cpu().numpy() for a in args)
        kw["kernel"] = kw["kernel"].cpu().numpy()
    return case, (args, kw)


def run(state):
    case, held = state
    if case["kind"] == "equalize":
        return equalize_histogram(held, case["bins"])
    if case["kind"] == "batch":
        return convolve_batch(held)
    if case["kind"] == "serve":
        server, calls = held
        requests = [server.submit(*args, **kw) for args, kw in calls]
        server.run()
        return [r.result for r in requests]
    args, kw = held
    return rlic_amd.convolve(*args, **kw)


# ----------------------------------------------------------------- the work

def work(case):
    """Inputs read once and outputs written once.  Operations: 12 for each
    step of a first pass (two step times of a subtraction and a division, a
    comparison, one position update of a product and a sum, the weighted
    sum), 2 for each step of a later one (its cells are known)."""
    if case["kind"] == "equalize":
        n = case["ny"] * case["nx"]
        return {"bytes": 2 * n * (4 if case["dtype"] == "f32" else 8), "flops": 3 * n}
    total = {"bytes": 0, "flops": 0}
    for c in _calls(case):
        size, n = 4 if c["dtype"] == "f32" else 8, c["ny"] * c["nx"]
        total["bytes"] += size * (4 * n + c["length"])
        total["flops"] += n * (c["length"] - 1) * (12 + 2 * (c["iterations"] - 1))
    return total


# -------------------------------------------------------- the exact results

def _walk(u, v, nx, ny, start, length, mode, px, py):
    """The cells that the lines from ``start`` visit: (steps, pixels) indices,
    ny * nx where a line has ended, in the order they are summed.  The step
    rule is evaluated in the field's own type, which defines the line."""
    kmid = length // 2
    lines = torch.full((length - 1, start.numel()), ny * nx, dtype=torch.int32,
                       device=start.device)
    row = 0
    for forward, steps in ((True, length - 1 - kmid), (False, kmid)):
        at = start.clone()
        i, j = at // nx, at % nx
        fx = torch.full(at.shape, 0.5, dtype=u.dtype, device=u.device)
        fy = fx.clone()
        alive = torch.ones(at.shape, dtype=torch.bool, device=u.device)
        last_u = last_v = None
        for _ in range(steps):
            pu, pv = u[at], v[at]
            alive = alive & ~(pu.isnan() | pv.isnan())
            if mode == "polarization":
                if last_u is not None:
                    flip = pu * last_u + pv * last_v < 0
                    pu, pv = torch.where(flip, -pu, pu), torch.where(flip, -pv, pv)
                last_u, last_v = pu, pv
            mu, mv = (pu, pv) if forward else (-pu, -pv)
            tx = (torch.where(mu.signbit(), fx, (0.5 - fx) * 2 + fx) / mu).abs()
            ty = (torch.where(mv.signbit(), fy, (0.5 - fy) * 2 + fy) / mv).abs()
            xs = tx < ty
            moves = alive & ((mu != 0) | (mv != 0))
            # the fraction across the other axis, rounded once
            fx_y = (ty.double() * mu.double() + fx.double()).to(u.dtype)
            fy_x = (tx.double() * mv.double() + fy.double()).to(u.dtype)
            fx = torch.where(xs, (mu < 0).to(u.dtype), fx_y)
            fy = torch.where(xs, fy_x, (mv < 0).to(u.dtype))
            j = j + torch.where(moves & xs, torch.where(mu >= 0, 1, -1), 0)
            i = i + torch.where(moves & ~xs, torch.where(mv >= 0, 1, -1), 0)
            j = j.remainder(nx) if px else j.clamp(0, nx - 1)
            i = i.remainder(ny) if py else i.clamp(0, ny - 1)
            at = i * nx + j
            lines[row] = torch.where(alive, at, ny * nx)
            row += 1
    return lines


def _exact_call(call, args, kw):
    texture, u, v = args
    ny, nx = texture.shape
    n, length = ny * nx, call["length"]
    kmid = length // 2
    order = [*range(kmid + 1, length), *range(kmid - 1, -1, -1)]
    weights = kw["kernel"].double().tolist()
    u, v = u.reshape(-1), v.reshape(-1)
    px, py = call["bx"] == "periodic", call["by"] == "periodic"
    x = torch.cat([texture.reshape(-1).double(), torch.zeros(1, device=texture.device,
                                                              dtype=torch.float64)])
    # as many pixels at a time as keep their lines within 16 GiB
    chunk = max(1, min(n, (1 << 32) // max(1, length - 1)))
    keep = None
    for _ in range(call["iterations"]):
        out = torch.zeros_like(x)
        for a in range(0, n, chunk):
            start = torch.arange(a, min(a + chunk, n), device=x.device, dtype=torch.int32)
            lines = keep if keep is not None else _walk(u, v, nx, ny, start, length, call["mode"],
                                                        px, py)
            acc = x[a:a + chunk][:start.numel()] * weights[kmid]
            for s, k in enumerate(order):
                acc += weights[k] * x[lines[s]]
            out[a:a + start.numel()] = acc
            keep = lines if chunk >= n else None
        x = out
        x[n] = 0
    return x[:n].reshape(ny, nx)


def exact(case, seed):
    device = _device()
    if case["kind"] == "equalize":
        x = _image(case, seed, device).double()
        lo, hi = x.min(), x.max()
        bins = ((x - lo) * (case["bins"] / (hi - lo))).floor().clamp(max=case["bins"] - 1).long()
        counts = torch.bincount(bins.reshape(-1), minlength=case["bins"])
        return counts.cumsum(0).double()[bins] / x.numel()
    results = []
    for k, c in enumerate(_calls(case)):
        args, kw = _arguments(c, seed * 1009 + k, device)
        results.append(_exact_call(c, args, kw))
    if case["kind"] == "convolve":
        return results[0].cpu().numpy() if case["where"] == "host" else results[0]
    return results
