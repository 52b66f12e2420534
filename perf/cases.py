"""What the library is measured on: one pass through a public entry point per
case, over the sizes, directions, data types and options it is used with.

Kinds of cases
  stencil  one Compute of a cuSten handle on a device-resident grid (x, y, xy;
           periodic and not; FP64 and FP32 storage)
  stream   the same on a host-resident grid, streamed in numTiles strips
  fun      one Compute of a point-function ("Fun") handle
  weno     one Compute of a WENO5 advection handle
  batch    several steps of many uneven periodic grids advanced together
  pent     one implicit step of many pentadiagonal systems: refill and factor
           the matrices (refactor) and solve, or solve with kept factors
  ch       several steps of one Cahn-Hilliard simulation, then its fields
  serve    a parameter sweep of Cahn-Hilliard requests through a server, from
           the first submit to the last result in the caller's memory

`exact` restates each pass in plain 64-bit torch; periodic pentadiagonal
solves are circulant there and go through an FFT.
"""
import math

import numpy as np
import torch

from custen_amd import api, workloads

DEV = "cuda"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a small call: the cache-resident grid of the 1024 x 1024 benchmark,
        # fourth-order d2/dx2; the launch is a large part of it
        dict(name="x_p_1024", kind="stencil", dir="x", periodic=True, f32=False, nx=1024, ny=1024,
             H=5, V=1),
        # the headline: 13-point biharmonic on a large periodic grid
        dict(name="xy_p_8192", kind="stencil", dir="xy", periodic=True, f32=False, nx=8192,
             ny=8192, H=5, V=5),
        # an ordinary solver grid with boundaries, whose node counts are odd
        # (cells + 1): unaligned rows, ragged strips, a write window
        dict(name="xy_np_odd", kind="stencil", dir="xy", periodic=False, f32=False, nx=4099,
             ny=3001, H=5, V=5),
        # FP32 storage of a large field
        dict(name="xy_p_f32_8192", kind="stencil", dir="xy", periodic=True, f32=True, nx=8192,
             ny=8192, H=5, V=5),
        # a wide filter window, the widest with a kernel of its own
        dict(name="xy_np_9x9_4096", kind="stencil", dir="xy", periodic=False, f32=False, nx=4096,
             ny=4096, H=9, V=9),
        # a field larger than the caller wants in HBM at once: y derivative of
        # pinned host data in four tiles
        dict(name="y_np_host", kind="stream", dir="y", periodic=False, f32=False, nx=8192,
             ny=4096, H=1, V=9, tiles=4, pinned=True),
        # the Laplacian of u^3 - u, the point function of the Cahn-Hilliard
        # program, on its largest grid
        dict(name="fun_cube_2048", kind="fun", func="xy_cube_minus", periodic=True, nx=2048,
             ny=2048),
        # advection of a field by a velocity field
        dict(name="weno_4096", kind="weno", nx=4096, ny=4096, single=True),
        # an ensemble of uneven grids, ten steps between two outputs
        dict(name="batch_128", kind="batch", grids=128, sizes="square", f32=False, H=5, steps=10),
        # variable-coefficient implicit hyperdiffusion lines: matrices change
        # every step
        dict(name="pent_4096x1022", kind="pent", m=1022, systems=4096, refactor=True),
        # one simulation, fifty steps between two snapshots
        dict(name="ch_1024", kind="ch", n=1024, steps=50),
        # a sweep of eight simulations of the four benchmark sizes
        dict(name="serve_8", kind="serve", sizes="256,512,1024,2048,256,512,1024,2048", steps=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stencil"] * 6 + ["stream", "fun", "weno", "batch", "pent", "ch", "serve"])
    if kind in ("stencil", "stream"):
        d = rng.choice(["x", "y", "xy", "xy"])
        c = dict(kind=kind, dir=d, periodic=rng.random() < 0.5, f32=rng.random() < 0.3, H=1, V=1)
        if d == "xy":
            c["H"], c["V"] = rng.choice([(3, 3), (5, 5), (5, 5), (7, 7), (9, 9), (3, 5), (5, 3)])
        else:
            c["H" if d == "x" else "V"] = rng.choice([3, 5, 7, 9, 11, 13])
        if kind == "stream":
            tiles = rng.choice([1, 2, 4, 8])
            c.update(nx=_log_int(rng, 200, 8192), ny=tiles * _log_int(rng, 32, 4096 // tiles),
                     tiles=tiles, pinned=rng.random() < 0.7)
        else:
            c.update(nx=_log_int(rng, 60, 8192), ny=_log_int(rng, 60, 8192))
        return c
    if kind == "fun":
        f = rng.choice(["xy_cube_minus", "xy_cube_minus", "xy_weighted_sum",
                        "x_central_difference", "y_central_difference9"])
        return dict(kind=kind, func=f, periodic=rng.random() < 0.7, nx=_log_int(rng, 60, 4096),
                    ny=_log_int(rng, 60, 4096))
    if kind == "weno":
        return dict(kind=kind, nx=_log_int(rng, 60, 4096), ny=_log_int(rng, 60, 4096),
                    single=rng.random() < 0.7)
    if kind == "batch":
        return dict(kind=kind, grids=_log_int(rng, 2, 96), sizes="uneven", f32=rng.random() < 0.3,
                    H=rng.choice([3, 5, 5]), steps=rng.randint(1, 12))
    if kind == "pent":
        m = _log_int(rng, 30, 2046)
        return dict(kind=kind, m=m, systems=_log_int(rng, 16, 4_000_000 // m),
                    refactor=rng.random() < 0.5)
    if kind == "ch":
        return dict(kind=kind, n=_log_int(rng, 48, 1500), steps=rng.randint(1, 50))
    sizes = [_log_int(rng, 64, 1400) for _ in range(rng.randint(2, 4))]
    sizes += [rng.choice(sizes) for _ in range(rng.randint(0, 4))]
    return dict(kind="serve", sizes=",".join(map(str, sizes)), steps=rng.randint(5, 40))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _uniform(shape, seed, lo=-1.0, hi=1.0, dtype=torch.float64):
    g = torch.Generator(device=DEV).manual_seed(seed)
    t = torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)
    return t.mul_(hi - lo).add_(lo).to(dtype)


def _second_difference(points, n):
    """Central d2/dx2 weights of `points` points on n cells of a 2 pi domain."""
    p = points // 2
    f = math.factorial
    w = [2.0 * (-1) ** (k + 1) * f(p) ** 2 / (k * k * f(p - k) * f(p + k)) for k in range(1, p + 1)]
    w = np.array(w[::-1] + [-2.0 * sum(w)] + w)
    return w / (2 * math.pi / n) ** 2


def _binomial(points):
    w = np.array([math.comb(points - 1, k) for k in range(points)], dtype=np.float64)
    return w / w.sum()


def _stencil_weights(c):
    if c["dir"] == "x":
        return _second_difference(c["H"], c["nx"])
    if c["dir"] == "y":
        return _second_difference(c["V"], c["ny"])
    if (c["H"], c["V"]) == (5, 5):
        return workloads.biharmonic_weights(c["nx"])
    if (c["H"], c["V"]) == (3, 3):
        return workloads.laplacian9_weights(c["nx"])
    return np.outer(_binomial(c["V"]), _binomial(c["H"])).ravel()


def _step_weights(H):
    """One stable explicit (hyper)diffusion step."""
    w = workloads.laplacian9_weights(2048) if H == 3 else -workloads.biharmonic_weights(2048)
    w = 0.2 * w / np.abs(w).max()
    w[H * H // 2] += 1.0
    return w


def _batch_shapes(c, seed):
    if c["sizes"] == "square":
        return [(s, s) for s in workloads.batch_sizes(c["grids"], 4)]
    r = np.random.default_rng(1000 + c["grids"])
    lo, hi = math.log(40), math.log(1500)
    return [(int(math.exp(a)), int(math.exp(b))) for a, b in r.uniform(lo, hi, (c["grids"], 2))]


def _hyperdiffusion(m, systems, seed):
    """I + sigma D2^T D2 (D2 the second difference on m points), one sigma per
    system: the five diagonals, interleaved (5, m, systems)."""
    sigma = torch.exp(_uniform((systems,), seed + 1, math.log(0.5), math.log(50.0)))
    pat = torch.zeros(5, m, dtype=torch.float64)
    for j in range(m - 2):  # row j of D2: points j, j + 1, j + 2
        for a, va in enumerate((1.0, -2.0, 1.0)):
            for b, vb in enumerate((1.0, -2.0, 1.0)):
                pat[2 + b - a, j + a] += va * vb
    t = pat.to(DEV)[:, :, None] * sigma
    t[2] += 1.0
    return t.contiguous()


def _ch_field(n, seed):
    return np.random.default_rng(seed).uniform(-0.1, 0.1, (n, n))


class _Handle:
    """A cuSten handle and the arrays it works on."""

    def __init__(self, variant, keep, out):
        self.h = api.cuSten_t()
        self.variant, self.keep, self.out = variant, keep, out
        self.compute = getattr(api, "custenCompute2DF32" if variant == "F32"
                               else f"cuStenCompute{variant}")
        self.destroy = getattr(api, "custenDestroy2DF32" if variant == "F32"
                               else f"cuStenDestroy{variant}")

    def __del__(self):
        if self.h.plan:
            self.destroy(self.h)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("stencil", "stream"):
        dt = torch.float32 if c["f32"] else torch.float64
        inp = _uniform((c["ny"], c["nx"]), seed, dtype=dt)
        out = torch.zeros_like(inp)
        w = torch.from_numpy(_stencil_weights(c)).to(DEV)
        place = api.DEVICE
        if kind == "stream":
            place = api.HOST
            inp, out = inp.cpu(), out.cpu()
            if c["pinned"]:
                inp, out = inp.pin_memory(), out.pin_memory()
        H, V, nx, ny = c["H"], c["V"], c["nx"], c["ny"]
        L, T = H // 2, V // 2
        tiles = c.get("tiles", 1)
        if c["f32"]:
            s = _Handle("F32", (inp, w), out)
            d = {"x": 0, "y": 1, "xy": 2}[c["dir"]]
            api.custenCreate2DF32(s.h, 0, tiles, nx, ny, d, int(c["periodic"]), out, inp, w,
                                  H, L, L, V, T, T)
        else:
            s = _Handle("2D" + c["dir"].upper() + ("p" if c["periodic"] else "np"), (inp, w), out)
            shape = (H, L, L, V, T, T) if c["dir"] == "xy" else \
                (H, L, L) if c["dir"] == "x" else (V, T, T)
            getattr(api, f"cuStenCreate{s.variant}")(s.h, 0, tiles, nx, ny, 32, 32, out, inp, w,
                                                     *shape)
        s.place = place
        return s
    if kind == "fun":
        inp = _uniform((c["ny"], c["nx"]), seed)
        out = torch.zeros_like(inp)
        coe = torch.from_numpy(_fun_coefficients(c)).to(DEV)
        f = api.custenGetBuiltinFunction(c["func"])
        p = "pFun" if c["periodic"] else "npFun"
        d = c["func"].split("_")[0].upper()
        s = _Handle(f"2D{d}{p}", (inp, coe), out)
        shape = {"X": (3, 1, 1, 1, f), "Y": (9, 4, 4, 9, f), "XY": (3, 1, 1, 3, 1, 1, f)}[d]
        if s.variant == "2DYnpFun":
            shape = (9, 4, 4, f)
        getattr(api, f"cuStenCreate{s.variant}")(s.h, 0, 1, c["nx"], c["ny"], 32, 32, out, inp,
                                                 coe, *shape)
        s.place = api.DEVICE
        return s
    if kind == "weno":
        q, u, v = _weno_fields(c, seed)
        s = _Handle("2DXYWENOADVp", (q, u, v), torch.zeros_like(q))
        api.cuStenCreate2DXYWENOADVp(s.h, 0, 1, c["nx"], c["ny"], 32, 32, 2 * math.pi / c["nx"],
                                     2 * math.pi / c["ny"], u, v, s.out, q)
        api.custenSetWenoSquares(s.h, c["single"])
        s.place = api.DEVICE
        return s
    if kind == "batch":
        shapes = _batch_shapes(c, seed)
        offs, total = _offsets(shapes)
        dt = torch.float32 if c["f32"] else torch.float64
        a = _uniform((total,), seed, dtype=dt)
        b = torch.zeros_like(a)
        views = [[t[o:o + ny * nx].view(ny, nx) for o, (ny, nx) in zip(offs, shapes)]
                 for t in (a, b)]
        H = c["H"]
        w = torch.from_numpy(_step_weights(H)).to(DEV)
        batch = api.Batch(views[1], views[0], w, H, H // 2, H, H // 2, f32=c["f32"])
        return dict(batch=batch, steps=c["steps"], sides=(a, b))
    if kind == "pent":
        t = _hyperdiffusion(c["m"], c["systems"], seed)
        s = dict(m=c["m"], systems=c["systems"], matrix=t if c["refactor"] else None,
                 factors=t.clone(), b=_uniform((c["m"], c["systems"]), seed + 2))
        if not c["refactor"]:
            api.custenPentFactorBatch(*s["factors"], c["m"], c["systems"])
        return s
    if kind == "ch":
        return dict(steps=c["steps"],
                    solver=api.CHSolver(api.ch_params(c["n"]), _ch_field(c["n"], seed)))
    return dict(steps=c["steps"], requests=[(api.ch_params(n), f) for n, f in _sweep(c, seed)])


def _fun_coefficients(c):
    if c["func"].startswith("xy"):
        return workloads.laplacian9_weights(c["nx"])
    if c["func"].startswith("x"):
        return np.array([1.0 / (2 * math.pi / c["nx"]) ** 2])
    return _second_difference(9, c["ny"])


def _weno_fields(c, seed):
    """A field with fronts and a shear flow with both signs in x and y."""
    ny, nx = c["ny"], c["nx"]
    y = torch.arange(ny, device=DEV, dtype=torch.float64)[:, None] * (2 * math.pi / ny)
    x = torch.arange(nx, device=DEV, dtype=torch.float64)[None, :] * (2 * math.pi / nx)
    q = torch.tanh(8.0 * torch.sin(x + 0.3 * seed % 6.0) * torch.cos(2 * y)) + \
        _uniform((ny, nx), seed, -1e-3, 1e-3)
    u = torch.sin(y) * torch.cos(x) + 0.1
    v = torch.cos(y + 0.5) * torch.sin(3 * x)
    return q, u.contiguous(), v.contiguous()


def _offsets(shapes):
    offs, total = [], 0
    for ny, nx in shapes:
        offs.append(total)
        total += (ny * nx + 63) // 64 * 64
    return offs, total


def _sweep(c, seed):
    return [(int(n), _ch_field(int(n), seed * 100 + k)) for k, n in enumerate(c["sizes"].split(","))]


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    if isinstance(state, _Handle):
        state.compute(state.h, state.place)
        return state.out
    if "batch" in state:
        b = state["batch"]
        b.run(state["steps"])
        cur = b.parity
        return state["sides"][cur], state["sides"][1 - cur]
    if "factors" in state:
        f, m, n = state["factors"], state["m"], state["systems"]
        if state["matrix"] is not None:
            f.copy_(state["matrix"])
            api.custenPentFactorBatch(f[0], f[1], f[2], f[3], f[4], m, n)
        api.custenPentSolveBatch(f[0], f[1], f[2], f[3], f[4], state["b"], m, n)
        return f, state["b"]
    if "solver" in state:
        state["solver"].run(state["steps"])
        return state["solver"].field()
    srv = api.CHServer(budget_bytes=32 << 30, max_slots=64)
    ids = [srv.submit(p, state["steps"], c0) for p, c0 in state["requests"]]
    srv.run_until_idle()
    out = [srv.result(i) for i in ids]
    srv.close()
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without: each input read once, each output written once
# ---------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind in ("stencil", "stream", "fun"):
        pts = c["nx"] * c["ny"]
        if kind == "fun":
            taps = 3 if c["func"].startswith("x_") else 9
        else:
            taps = c["H"] * c["V"]
        return dict(bytes=pts * (8 if c.get("f32") else 16), flops=2 * taps * pts)
    if kind == "weno":
        pts = c["nx"] * c["ny"]
        return dict(bytes=32 * pts, flops=2 * 100 * pts)
    if kind == "batch":
        pts = sum(ny * nx for ny, nx in _batch_shapes(c, 0))
        return dict(bytes=pts * (8 if c["f32"] else 16), flops=2 * c["H"] ** 2 * pts * c["steps"])
    if kind == "pent":
        pts = c["m"] * c["systems"]
        if c["refactor"]:
            return dict(bytes=8 * 12 * pts, flops=(10 + 9) * pts)
        return dict(bytes=8 * 7 * pts, flops=9 * pts)
    if kind == "ch":
        pts = c["n"] ** 2
        return dict(bytes=4 * 8 * pts, flops=110 * pts * c["steps"])
    pts = sum(int(n) ** 2 for n in c["sizes"].split(","))
    return dict(bytes=2 * 8 * pts, flops=110 * pts * c["steps"])


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch
# ---------------------------------------------------------------------------
def _apply(u, w, H, L, V, T):
    """Periodic stencil sum."""
    out = torch.zeros_like(u)
    for j in range(V):
        for i in range(H):
            if w[j * H + i] != 0.0:
                out += float(w[j * H + i]) * torch.roll(u, (T - j, L - i), (0, 1))
    return out


def _exact_stencil(u, w, H, V, periodic):
    full = _apply(u, w, H, H // 2, V, V // 2)
    if periodic:
        return full
    out = torch.zeros_like(u)
    L, T, R, B = H // 2, V // 2, u.shape[1] - H // 2, u.shape[0] - V // 2
    out[T:B, L:R] = full[T:B, L:R]
    return out


def _weno_flux(v):
    v1, v2, v3, v4, v5 = v
    p1 = v1 / 3 - v2 * (7 / 6) + v3 * (11 / 6)
    p2 = -v2 / 6 + v3 * (5 / 6) + v4 / 3
    p3 = v3 / 3 + v4 * (5 / 6) - v5 / 6
    s1 = (13 / 12) * (v1 - 2 * v2 + v3) ** 2 + 0.25 * (v1 - 4 * v2 + 3 * v3) ** 2
    s2 = (13 / 12) * (v2 - 2 * v3 + v4) ** 2 + 0.25 * (v2 - v4) ** 2
    s3 = (13 / 12) * (v3 - 2 * v4 + v5) ** 2 + 0.25 * (3 * v3 - 4 * v4 + v5) ** 2
    a1, a2, a3 = 0.1 / (s1 + 1e-6) ** 2, 0.6 / (s2 + 1e-6) ** 2, 0.3 / (s3 + 1e-6) ** 2
    return (a1 * p1 + a2 * p2 + a3 * p3) / (a1 + a2 + a3)


def _exact_weno(q, vel, dim):
    n = q.shape[dim]
    inv = 1.0 / (2 * math.pi / n)
    # d[k] = q[c + k - 3] - q[c + k - 4]
    d = [None] + [(torch.roll(q, 3 - k, dim) - torch.roll(q, 4 - k, dim)) * inv
                  for k in range(1, 7)]
    pos = _weno_flux(d[1:6])
    neg = _weno_flux([d[k] for k in (6, 5, 4, 3, 2)])
    return vel * torch.where(vel > 0, pos, neg)


def _exact_pent(t, b):
    """Factors and solutions of interleaved systems, as the entry points lay
    them out (factored dl, d, du, dw in place of the matrix)."""
    ds, dl, d, du, dw = (x.clone() for x in t)
    m = d.shape[0]
    x = b.clone()
    for i in range(m):
        if i > 1:
            dl[i] -= ds[i] * du[i - 2]
            d[i] -= ds[i] * dw[i - 2]
        if i > 0:
            d[i] -= dl[i] * du[i - 1]
            if i < m - 1:
                du[i] -= dl[i] * dw[i - 1]
            x[i] -= dl[i] * x[i - 1]
            if i > 1:
                x[i] -= ds[i] * x[i - 2]
        x[i] /= d[i]
        if i < m - 1:
            du[i] /= d[i]
        if i < m - 2:
            dw[i] /= d[i]
    x[m - 2] -= du[m - 2] * x[m - 1]
    for i in range(m - 3, -1, -1):
        x[i] -= du[i] * x[i + 1] + dw[i] * x[i + 2]
    return torch.stack([ds, dl, d, du, dw]), x


def _exact_ch(c0, steps):
    n = c0.shape[0]
    dx = 2 * math.pi / n
    dt = 0.1 * dx
    s = 2 * dt * 0.01 / (3 * dx ** 4)
    snl = (dt / 3) * (2 / dx ** 2)
    lin = [0, 0, -1, 0, 0, 0, -2, 8, -2, 0, -1, 8, -20, 8, -1, 0, -2, 8, -2, 0, 0, 0, -1, 0, 0]
    lin = [s * v for v in lin]
    nl = [snl * v for v in (0, 1, 0, 1, -4, 1, 0, 1, 0)]
    theta = torch.arange(n, device=DEV, dtype=torch.float64) * (2 * math.pi / n)
    inv = 1.0 / (1.0 + s * (2 - 2 * torch.cos(theta)) ** 2)
    inv = inv[:, None] * inv[None, :]
    c = torch.from_numpy(c0).to(DEV)
    old = c.clone()
    for _ in range(steps):
        bar = 2 * c - old
        r = _apply(bar, lin, 5, 2, 5, 2) - (2 / 3) * (c - old) + _apply(c ** 3 - c, nl, 3, 1, 3, 1)
        c, old = bar + torch.fft.ifft2(torch.fft.fft2(r) * inv).real, c
    return c, old


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("stencil", "stream"):
        u = _uniform((c["ny"], c["nx"]), seed,
                     dtype=torch.float32 if c["f32"] else torch.float64).double()
        return _exact_stencil(u, _stencil_weights(c), c["H"], c["V"], c["periodic"])
    if kind == "fun":
        u = _uniform((c["ny"], c["nx"]), seed)
        w = _fun_coefficients(c)
        if c["func"] == "xy_cube_minus":
            u = u ** 3 - u
        if c["func"].startswith("xy"):
            return _exact_stencil(u, w, 3, 3, c["periodic"])
        if c["func"].startswith("x"):
            return _exact_stencil(u, [w[0], -2.0 * w[0], w[0]], 3, 1, c["periodic"])
        return _exact_stencil(u, w, 1, 9, c["periodic"])
    if kind == "weno":
        q, u, v = _weno_fields(c, seed)
        return _exact_weno(q, u, 1) + _exact_weno(q, v, 0)
    if kind == "batch":
        shapes = _batch_shapes(c, seed)
        offs, total = _offsets(shapes)
        a = _uniform((total,), seed, dtype=torch.float32 if c["f32"] else torch.float64).double()
        w = _step_weights(c["H"])
        sides = [a, torch.zeros_like(a)]
        for k in range(c["steps"]):
            for o, (ny, nx) in zip(offs, shapes):
                sl = slice(o, o + ny * nx)
                sides[(k + 1) & 1][sl] = _apply(sides[k & 1][sl].view(ny, nx), w, c["H"],
                                                c["H"] // 2, c["H"], c["H"] // 2).view(-1)
        cur = c["steps"] & 1
        return sides[cur], sides[1 - cur]
    if kind == "pent":
        return _exact_pent(_hyperdiffusion(c["m"], c["systems"], seed),
                           _uniform((c["m"], c["systems"]), seed + 2))
    if kind == "ch":
        return _exact_ch(_ch_field(c["n"], seed), c["steps"])
    return [_exact_ch(f, c["steps"])[0] for _, f in _sweep(c, seed)]
