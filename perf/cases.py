"""The workloads whose speed this repository watches.

``listed()`` names twelve calls a user of the engine makes, from one small
plane to a batched ensemble; ``draw(rng)`` gives others of the same ranges.
``prepare`` makes what a program holds before the call (inputs on the GPU,
the transform, a batch), ``run`` is one pass through the public entry
points, ``work`` the bytes and operations a pass cannot do without, and
``exact`` the same results in 64 bits from plain torch.

Kinds of case:
  transform  one call of a SphericalHarmonicTransform or
             VorticityDivergenceOperator method on a level stack
  roundtrip  a TransformBatch of one or more members' vorticity, divergence,
             temperature and ln ps to the grid and back, replayed as a graph
  ensemble   EnsembleSynthesis: members' spectra in, every grid field out
  sample     fields, gradients or winds at scattered points
  vertical   the semi-implicit column operators
"""
from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "gpuwm-global_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from arwen_spectral import (EnsembleSynthesis, LNPS_REFERENCE, SphericalHarmonicTransform,  # noqa: E402
                            TransformBatch, VorticityDivergenceOperator)
from arwen_spectral import sampling, semi_implicit  # noqa: E402
from arwen_spectral.constants import EARTH_RADIUS_M  # noqa: E402

# coefficient amplitude of each field class at n = 1 (vorticity and
# divergence in 1/s, temperature anomaly in K, ln ps anomaly, moisture)
SCALE = {"vorticity": 1e-5, "divergence": 2e-6, "temperature": 10.0, "lnps": 1e-2, "qv": 1e-3}
ENSEMBLE_FIELDS = ("u", "v", "theta", "qv", "lnps", "psi", "chi")
TAU, DT, ALPHA = 900.0, 600.0, 0.6  # seconds, seconds, off-centring


def listed():
    return [
        # one surface field of a small model: launches and latency only
        dict(name="inverse_plane_t63", kind="transform", op="inverse", T=63, nlat=64, nlon=128,
             count=1, precision="float32"),
        # ln ps back to spectral space in every step of the T383 dycore
        dict(name="forward_plane_t383", kind="transform", op="forward", T=383, nlat=384, nlon=768,
             count=1, precision="bf16x6"),
        # temperature and both its gradients, one level stack, every step
        dict(name="inverse_gradient_t383", kind="transform", op="inverse_with_gradient", T=383,
             nlat=384, nlon=768, count=40, precision="bf16x6"),
        # analysis of a 64-level stack on the dealiased T255 grid
        dict(name="forward_t255_l64", kind="transform", op="forward", T=255, nlat=384, nlon=768,
             count=64, precision="float32"),
        # winds from vorticity and divergence, and back, one level stack
        dict(name="wind_t383", kind="transform", op="wind", T=383, nlat=384, nlon=768, count=40,
             precision="bf16x6"),
        dict(name="vordiv_t383", kind="transform", op="vordiv", T=383, nlat=384, nlon=768,
             count=40, precision="bf16x6"),
        # gradients on a default-sized odd grid (161 x 322): an equator row,
        # a longitude count with prime factors 7 and 23, a ragged level count
        dict(name="gradient_t106_ragged", kind="transform", op="gradient", T=106, nlat=161,
             nlon=322, count=19, precision="float32"),
        # the 121-field round trip of the benchmark
        dict(name="roundtrip_t383", kind="roundtrip", T=383, nlat=384, nlon=768, levels=40,
             members=1, precision="bf16x6"),
        # sixteen members' grid fields for the assimilation
        dict(name="ensemble_t127_m16", kind="ensemble", T=127, nlat=192, nlon=384, levels=40,
             members=16, precision="bf16x6"),
        # a level stack at 30,000 scattered points
        dict(name="sample_t383", kind="sample", op="scalar", T=383, nlat=384, nlon=768, count=40,
             points=30000, precision="float64"),
        # the semi-implicit stage solve and the half map of a T383 L40 step
        dict(name="solve_t383_l40", kind="vertical", op="solve", T=383, nlat=384, nlon=768,
             levels=40),
        dict(name="half_map_t383_l40", kind="vertical", op="half", T=383, nlat=384, nlon=768,
             levels=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_grid(rng, T):
    """Latitudes of the linear or the dealiased grid; longitudes rounded up
    to an even number, a multiple of 16 or a multiple of 64."""
    f = rng.choice((1.0, 1.5))
    nlat = math.ceil(f * (T + 1))
    step = rng.choice((2, 16, 64, 64))
    return nlat, -(-math.ceil(2 * f * (T + 1)) // step) * step


def draw(rng):
    kind = rng.choice(("transform",) * 5 + ("roundtrip", "ensemble", "sample", "vertical"))
    T = _log_int(rng, 21, 383)
    nlat, nlon = _draw_grid(rng, T)
    precision = rng.choice(("float32", "bf16x6"))
    # no more than about the listed cases' planes, by the triangle's size
    room = (384 * 385) / ((T + 1) * (T + 2))
    if kind == "transform":
        op = rng.choice(("inverse", "inverse_exp", "inverse_with_gradient", "gradient", "forward",
                         "forward_about", "wind", "vordiv", "waist"))
        return dict(kind=kind, op=op, T=T, nlat=nlat, nlon=nlon,
                    count=_log_int(rng, 1, min(64, 1 + 64 * room)), precision=precision)
    if kind == "roundtrip":
        return dict(kind=kind, T=T, nlat=nlat, nlon=nlon, levels=_log_int(rng, 5, 40),
                    members=_log_int(rng, 1, max(1.0, min(8.0, room))), precision=precision)
    if kind == "ensemble":
        T = min(T, 213)
        nlat, nlon = _draw_grid(rng, T)
        room = (128 * 129) / ((T + 1) * (T + 2))
        return dict(kind=kind, T=T, nlat=nlat, nlon=nlon, levels=_log_int(rng, 5, 40),
                    members=_log_int(rng, 2, max(2.0, min(16.0, 16 * room))), precision=precision)
    if kind == "sample":
        return dict(kind=kind, op=rng.choice(("scalar", "scalar", "gradient", "wind")), T=T,
                    nlat=nlat, nlon=nlon, count=_log_int(rng, 1, 20),
                    points=_log_int(rng, 300, 30000),
                    precision=rng.choice(("float64", "float64", "float32")))
    return dict(kind="vertical", op=rng.choice(("solve", "apply", "half", "tendencies")), T=T,
                nlat=nlat, nlon=nlon, levels=_log_int(rng, 5, 64 if T < 256 else 40))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


@functools.lru_cache(maxsize=None)
def _transform(T, nlat, nlon, precision):
    """A program makes its transform once and keeps it."""
    return SphericalHarmonicTransform.create(T, nlat=nlat, nlon=nlon, dealias_factor=1.0,
                                             precision=precision)


def _tr(case):
    precision = case.get("precision", "float32")
    if case["kind"] in ("sample", "vertical"):
        precision = "float32"
    return _transform(case["T"], case["nlat"], case["nlon"], precision)


def _red(T, lead, scale, seed):
    """Red-spectrum coefficients scale n^-1.5 (N + iN)/sqrt(2), m = 0 real,
    zero above the triangle and at n = 0, complex64."""
    dev, t1 = _device(), T + 1
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))
    n = torch.arange(t1, device=dev, dtype=torch.float32)
    amp = torch.where(n > 0, n.clamp(min=1) ** -1.5, torch.zeros_like(n)) * (scale / math.sqrt(2.0))
    x = torch.randn((*lead, t1, t1, 2), generator=gen, device=dev) * amp[:, None, None]
    x *= torch.ones((t1, t1), device=dev).tril()[..., None]
    x[..., :, 0, 1] = 0.0
    return torch.view_as_complex(x)


def _fields(case, seed):
    """The spectral fields of a transform, roundtrip or ensemble case."""
    T, kind = case["T"], case["kind"]
    s = 1000 * int(seed)
    if kind == "ensemble":
        lead = (case["members"], case["levels"])
        return {"vorticity": _red(T, lead, SCALE["vorticity"], s + 1),
                "divergence": _red(T, lead, SCALE["divergence"], s + 2),
                "theta": _red(T, lead, SCALE["temperature"], s + 3),
                "qv": _red(T, lead, SCALE["qv"], s + 4),
                "log_surface_pressure": _red(T, lead[:1], SCALE["lnps"], s + 5)}
    if kind == "roundtrip":
        lead = (case["members"], case["levels"])
        return {"vorticity": _red(T, lead, SCALE["vorticity"], s + 1),
                "divergence": _red(T, lead, SCALE["divergence"], s + 2),
                "temperature": _red(T, lead, SCALE["temperature"], s + 3),
                "lnps": _red(T, lead[:1], SCALE["lnps"], s + 4)}
    lead = (case["count"],)
    if case["op"] in ("wind", "vordiv"):
        return {"vorticity": _red(T, lead, SCALE["vorticity"], s + 1),
                "divergence": _red(T, lead, SCALE["divergence"], s + 2)}
    name = "lnps" if case["op"] == "inverse_exp" else "temperature"
    return {"field": _red(T, lead, SCALE[name], s + 1)}


def _grid_inputs(case, seed):
    """float32 grid fields of an analysis case, from the 64-bit synthesis below."""
    f, ex = _fields(case, seed), _exact_transform(case)
    if case["op"] == "vordiv":
        return tuple(g.float().contiguous() for g in ex.wind(f["vorticity"], f["divergence"]))
    g = ex.inverse(f["field"])
    if case["op"] == "forward_about":
        g = g + _theta_offsets(case)[:, None, None]
    return (g.float().contiguous(),)


def _theta_offsets(case):
    """Whole-kelvin reference temperatures per level."""
    return torch.linspace(215.0, 305.0, case["count"], device=_device(), dtype=torch.float64).round()


def _operator(L, seed):
    """A well-posed vertical operator: M = V diag(c^2) V^-1 with wave speeds
    of 10 to 330 m/s, C of full column rank, B = -M C^+ (so M = -B C)."""
    rng = np.random.default_rng(int(seed))
    q, _ = np.linalg.qr(rng.standard_normal((L, L)))
    v = q * rng.uniform(0.5, 2.0, L)
    c2 = np.sort(rng.uniform(10.0, 330.0, L))[::-1] ** 2
    vi = np.linalg.inv(v)
    m = (v * c2) @ vi
    c = rng.standard_normal((L + 1, L)) / math.sqrt(L)
    return -m @ np.linalg.pinv(c), c, m, v, vi, c2


def _vertical_inputs(case, seed):
    """Columns and float32 operator matrices, as the semi-implicit scheme builds them."""
    T, L, op = case["T"], case["levels"], case["op"]
    s, dev = 1000 * int(seed), _device()
    out = {"d": _red(T, (L,), SCALE["divergence"], s + 1),
           "theta": _red(T, (L,), SCALE["temperature"], s + 2),
           "lnps": _red(T, (), SCALE["lnps"], s + 3)}
    b, c, m, v, vi, c2 = _operator(L, seed)
    n = np.arange(T + 1.0)
    k2 = n * (n + 1.0) / EARTH_RADIUS_M ** 2
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev)  # noqa: E731
    mats = {"b": up(b), "c": up(c), "k2": up(k2)}
    if op in ("solve", "apply"):
        f = (TAU if op == "solve" else ALPHA * DT) ** 2 * k2
        mats["inverse"] = up((v[None] / (1.0 + f[:, None] * c2)[:, None, :]) @ vi)
        if op == "apply":
            mats["structure"] = up(m)
    if op == "half":
        # Crank-Nicolson half steps of each mode frequency: p + i q omega = sqrt(g)
        def half(freq):
            y = freq * DT
            root = np.sqrt((1 + 1j * (1 - ALPHA) * y) / (1 - 1j * ALPHA * y))
            return root.real, np.where(freq > 0, root.imag / np.where(freq > 0, freq, 1.0), 0.5 * DT)
        p, qq = half(np.sqrt(k2)[:, None] * np.sqrt(c2))
        mats["p_d"], mats["q_d"] = up((v * p[:, None, :]) @ vi), up((v * qq[:, None, :]) @ vi)
        # C V / c and -V^-1 B / c carry the modes of C B; its null space has frequency 0
        right, left = c @ v / np.sqrt(c2), -(vi @ b) / np.sqrt(c2)[:, None]
        null = np.eye(L + 1) - right @ left
        mats["p_x"] = up((right * p[:, None, :]) @ left + null)
        mats["q_x"] = up((right * qq[:, None, :]) @ left + 0.5 * DT * null)
    out.update(mats)
    return out


def _points(case, seed):
    rng = np.random.default_rng(int(seed) + 77)
    return (np.degrees(np.arcsin(rng.uniform(-0.9999, 0.9999, case["points"]))),
            rng.uniform(0.0, 360.0, case["points"]))


def _sample_fields(case, seed):
    s, lead = 1000 * int(seed), (case["count"],)
    if case["op"] == "wind":
        return (_red(case["T"], lead, SCALE["vorticity"], s + 1),
                _red(case["T"], lead, SCALE["divergence"], s + 2))
    return (_red(case["T"], lead, SCALE["temperature"], s + 1),)


# --------------------------------------------------------------------------
# What is timed
# --------------------------------------------------------------------------

def _prepare_transform(case, seed):
    t, op = _tr(case), case["op"]
    if op in ("forward", "forward_about", "vordiv", "waist"):
        x = _grid_inputs(case, seed)
    else:
        x = tuple(_fields(case, seed).values())
    vec = VorticityDivergenceOperator(t)
    if op == "forward_about":
        g = _theta_offsets(case)
        go = g.float()
        co = (g * math.sqrt(4.0 * math.pi)).to(torch.complex64)
        return lambda: t.forward_about(x[0], go, co)
    return {"inverse": lambda: t.inverse(x[0]),
            "inverse_exp": lambda: t.inverse_about(
                x[0], LNPS_REFERENCE * math.sqrt(4.0 * math.pi), exp=True),
            "inverse_with_gradient": lambda: t.inverse_with_gradient(x[0]),
            "gradient": lambda: t.gradient(x[0]),
            "forward": lambda: t.forward(x[0]),
            "waist": lambda: t.contract_waist(t.fourier_waist(x[0])),
            "wind": lambda: vec.wind_from_vordiv(*x),
            "vordiv": lambda: vec.vordiv_from_wind(*x)}[op]


def _prepare_roundtrip(case, seed):
    t, f = _tr(case), _fields(case, seed)
    dev = _device()
    grid = lambda x: torch.empty((*x.shape[:-2], *t.grid.shape), device=dev)  # noqa: E731
    u, v, temp, ps = (grid(f[n]) for n in ("vorticity", "divergence", "temperature", "lnps"))
    back = {n: torch.empty_like(x) for n, x in f.items()}
    batch = TransformBatch([
        ("wind", t, (f["vorticity"], f["divergence"]), (u, v)),
        ("inverse", t, f["temperature"], temp),
        ("inverse", t, f["lnps"], ps),
        ("vordiv", t, (u, v), (back["vorticity"], back["divergence"])),
        ("forward", t, temp, back["temperature"]),
        ("forward", t, ps, back["lnps"])])
    batch.set_config(split_acc=0)
    batch.autotune(reps=2)
    batch.capture()

    def call():
        batch.launch()
        return u, v, temp, ps, back
    return call


def _prepare_ensemble(case, seed):
    t, f = _tr(case), _fields(case, seed)
    members = [{n: x[k] for n, x in f.items()} for k in range(case["members"])]
    ens = EnsembleSynthesis(t, case["members"], case["levels"], ENSEMBLE_FIELDS)
    ens.batch.autotune(reps=2)
    ens.run(graph=True)

    def call():
        ens.load(members)
        return ens.run(graph=True)
    return call


def _prepare_sample(case, seed):
    t, x = _tr(case), _sample_fields(case, seed)
    lat, lon = _points(case, seed)
    fn = {"scalar": sampling.sample_scalar, "gradient": sampling.sample_gradient,
          "wind": sampling.sample_wind}[case["op"]]
    return lambda: fn(t, *x, lat, lon, precision=case["precision"], as_device=True)


def _prepare_vertical(case, seed):
    t, i = _tr(case), _vertical_inputs(case, seed)
    a = (t, i["d"], i["theta"], i["lnps"], i["b"], i["c"])
    return {"solve": lambda: semi_implicit.vertical_solve_shifted(*a, i["inverse"], i["k2"], TAU),
            "apply": lambda: semi_implicit.vertical_apply(*a, i["structure"], i["inverse"],
                                                          i["k2"], DT, ALPHA),
            "half": lambda: semi_implicit.vertical_half_apply(
                *a, i["p_d"], i["q_d"], i["p_x"], i["q_x"], i["k2"]),
            "tendencies": lambda: semi_implicit.vertical_linear_tendencies(*a, i["k2"], 0.7)
            }[case["op"]]


def prepare(case, seed):
    return {"transform": _prepare_transform, "roundtrip": _prepare_roundtrip,
            "ensemble": _prepare_ensemble, "sample": _prepare_sample,
            "vertical": _prepare_vertical}[case["kind"]](case, seed)


def run(state):
    return state()


# --------------------------------------------------------------------------
# Work
# --------------------------------------------------------------------------

def work(case):
    """Triangles of the coefficients and whole grid fields once each; each
    Legendre table once as float32 (north half); 4 operations per table
    value and plane, and the longitude FFTs."""
    T, nlat, nlon, kind = case["T"], case["nlat"], case["nlon"], case["kind"]
    tri, full, g = (T + 1) * (T + 2) / 2, (T + 1.0) ** 2, float(nlat * nlon)
    table, half = 4.0 * tri * math.ceil(nlat / 2), nlat / 2
    fft = 2.5 * g * math.log2(nlon)

    def transform(coeffs_in, grids, planes, tables, coeffs_out=0.0):
        return (8 * tri * coeffs_in + 8 * full * coeffs_out + 4 * g * grids + table * tables,
                4 * half * tri * planes + fft * grids)

    if kind == "transform":
        n = case["count"]
        b, f = {"inverse": lambda: transform(n, n, n, 1),
                "inverse_exp": lambda: transform(n, n, n, 1),
                "inverse_with_gradient": lambda: transform(n, 3 * n, 2 * n, 2),
                "gradient": lambda: transform(n, 2 * n, 2 * n, 2),
                "forward": lambda: transform(0, n, n, 1, n),
                "forward_about": lambda: transform(0, n, n, 1, n),
                "waist": lambda: transform(0, n, n, 1, n),
                "wind": lambda: transform(2 * n, 2 * n, 2 * n, 1),
                "vordiv": lambda: transform(0, 2 * n, 2 * n, 1, 2 * n)}[case["op"]]()
        if case["op"] == "waist":  # the waist is itself a result of the first call
            b += 2 * 8.0 * n * nlat * (T + 1)
        return {"bytes": b, "flops": f}
    if kind == "roundtrip":
        n = case["members"] * (3 * case["levels"] + 1)
        b, f = transform(n, 2 * n, 2 * n, 2, n)
        return {"bytes": b, "flops": f}
    if kind == "ensemble":
        n = case["members"] * case["levels"]
        fields = 6 * n + case["members"]
        b, f = transform(4 * n + case["members"], fields, fields, 1)
        return {"bytes": b, "flops": f}
    if kind == "sample":
        two = 2 if case["op"] != "scalar" else 1
        cols = case["count"] * (2 if case["op"] == "wind" else 1)
        return {"bytes": 8 * tri * cols + 8.0 * case["points"] * (3 + two * case["count"]),
                "flops": case["points"] * tri * (4.0 * cols * two + 4.0 * two)}
    L = case["levels"]
    mats = {"solve": L * L, "apply": L * L, "half": 2 * (L * L + (L + 1) ** 2),
            "tendencies": 0}[case["op"]]
    prods = {"solve": 3, "apply": 4, "half": 6, "tendencies": 2}[case["op"]]
    return {"bytes": (2 * L + 1) * 8 * (tri + full) + 4.0 * (T + 1) * mats,
            "flops": 4.0 * prods * L * L * tri}


# --------------------------------------------------------------------------
# 64-bit results from plain torch
# --------------------------------------------------------------------------

class _Exact:
    """The spherical-harmonic transform in float64: dense tables P[m, n, j]
    and dP/dphi at the Gauss nodes, products and longitude sums by matmul."""

    def __init__(self, T, nlat, nlon):
        mu, w = np.polynomial.legendre.leggauss(nlat)
        dev = _device()
        self.T, self.nlat, self.nlon, self.a = T, nlat, nlon, EARTH_RADIUS_M
        self.mu = torch.from_numpy(mu).to(dev)
        self.w = torch.from_numpy(w).to(dev)
        self.cos = torch.sqrt(1.0 - self.mu ** 2)
        self.m = torch.arange(T + 1, device=dev, dtype=torch.float64)
        self.P, self.dP = self.tables(self.mu)
        lam = torch.arange(nlon, device=dev, dtype=torch.float64) * (2.0 * math.pi / nlon)
        ang = torch.outer(self.m, lam)
        self.c, self.s = torch.cos(ang), torch.sin(ang)

    def tables(self, x):
        """P[m, n, j] = normalized P_n^m(x_j) (0 for n < m) and dP/dphi."""
        T, dev = self.T, x.device
        root = torch.sqrt(1.0 - x ** 2)
        P = torch.zeros((T + 1, T + 1, x.numel()), device=dev, dtype=torch.float64)
        d = torch.full_like(x, 1.0 / math.sqrt(4.0 * math.pi))
        for m in range(T + 1):
            if m:
                d = -math.sqrt((2 * m + 1) / (2.0 * m)) * root * d
            P[m, m] = d
        m = torch.arange(T + 1, device=dev, dtype=torch.float64)[:, None]
        for n in range(1, T + 1):
            mm = m[:n]
            g = torch.sqrt((4.0 * n * n - 1.0) / (n * n - mm * mm))
            h = torch.sqrt(((n - 1.0) ** 2 - mm * mm).clamp(min=0) / (4.0 * (n - 1.0) ** 2 - 1.0))
            prev2 = P[:n, n - 2] if n > 1 else torch.zeros_like(P[:n, 0])
            P[:n, n] = g * (x * P[:n, n - 1] - h * prev2)
        dP = torch.zeros_like(P)
        for n in range(1, T + 1):
            mm = m[:n + 1]
            e = torch.sqrt((n * n - mm * mm) * (2.0 * n + 1.0) / (2.0 * n - 1.0))
            dP[:n + 1, n] = root * (n * x * P[:n + 1, n] - e * P[:n + 1, n - 1]) / (x * x - 1.0)
        return P, dP

    def waist(self, c, table):
        """(F, n, m) coefficients -> X (F, j, m)."""
        c = c.to(torch.complex128).reshape(-1, self.T + 1, self.T + 1)
        F = c.shape[0]
        a = torch.cat([c.real, c.imag]).permute(2, 0, 1).contiguous()
        x = torch.bmm(a, table)  # (m, 2F, j)
        return torch.complex(x[:, :F], x[:, F:]).permute(1, 2, 0)

    def grid(self, X):
        two = torch.where(self.m > 0, 2.0, 1.0)
        return ((X.real * two) @ self.c - (X.imag * two) @ self.s)

    def inverse(self, c):
        return self.grid(self.waist(c, self.P)).reshape(*c.shape[:-2], self.nlat, self.nlon)

    def gradient(self, c):
        lead = c.shape[:-2]
        east = self.grid(self.waist(c * (1j * self.m), self.P)) / (self.a * self.cos[:, None])
        north = self.grid(self.waist(c, self.dP)) / self.a
        shape = (*lead, self.nlat, self.nlon)
        return east.reshape(shape), north.reshape(shape)

    def inverse_laplacian(self, c):
        n = self.m[:, None]
        lam = -n * (n + 1.0) / self.a ** 2
        return torch.where(n > 0, c.to(torch.complex128) / torch.where(n > 0, lam, 1.0), 0.0)

    def wind(self, vort, div):
        pe, pn = self.gradient(self.inverse_laplacian(vort))
        ce, cn = self.gradient(self.inverse_laplacian(div))
        return ce - pn, pe + cn

    def fourier(self, g):
        g = g.double()
        return torch.complex(g @ self.c.T, -(g @ self.s.T)) / self.nlon

    def contract(self, X, table):
        """X (F, j, m) -> sum_j table[m, n, j] X -> (F, n, m)."""
        F = X.shape[0]
        a = torch.cat([X.real, X.imag]).permute(2, 0, 1).contiguous()
        y = torch.bmm(a, table.transpose(1, 2).contiguous())
        return torch.complex(y[:, :F], y[:, F:]).permute(1, 2, 0)

    def forward(self, g):
        X = self.fourier(g.reshape(-1, self.nlat, self.nlon))
        c = self.contract(X * (2.0 * math.pi * self.w)[:, None], self.P)
        c = c.clone()
        c[..., 0] = c[..., 0].real.to(c.dtype)
        return c.reshape(*g.shape[:-2], self.T + 1, self.T + 1)

    def vordiv(self, u, v):
        U = self.fourier(u.reshape(-1, self.nlat, self.nlon))
        V = self.fourier(v.reshape(-1, self.nlat, self.nlon))
        w = (2.0 * math.pi / self.a * self.w)[:, None]
        zonal = 1j * self.m * w / self.cos[:, None]
        div = self.contract(U * zonal, self.P) - self.contract(V * w, self.dP)
        vort = self.contract(V * zonal, self.P) + self.contract(U * w, self.dP)
        out = []
        for c in (vort, div):
            c = c * torch.ones((self.T + 1,) * 2, device=c.device, dtype=torch.float64).tril()
            c[..., 0] = c[..., 0].real.to(c.dtype)
            out.append(c.reshape(*u.shape[:-2], self.T + 1, self.T + 1))
        return tuple(out)


@functools.lru_cache(maxsize=4)
def _exact_tables(T, nlat, nlon):
    return _Exact(T, nlat, nlon)


def _exact_transform(case):
    return _exact_tables(case["T"], case["nlat"], case["nlon"])


def _exact_one(case, seed):
    ex, op = _exact_transform(case), case["op"]
    if op in ("forward", "waist"):
        return ex.forward(*_grid_inputs(case, seed))
    if op == "forward_about":
        off = _theta_offsets(case)
        c = ex.forward(_grid_inputs(case, seed)[0].double() - off[:, None, None])
        c[:, 0, 0] += off * math.sqrt(4.0 * math.pi)
        return c
    if op == "vordiv":
        return ex.vordiv(*_grid_inputs(case, seed))
    f = tuple(x.to(torch.complex128) for x in _fields(case, seed).values())
    if op == "inverse":
        return ex.inverse(f[0])
    if op == "inverse_exp":
        return torch.exp(ex.inverse(f[0]) + LNPS_REFERENCE)
    if op == "inverse_with_gradient":
        return (ex.inverse(f[0]), *ex.gradient(f[0]))
    if op == "gradient":
        return ex.gradient(f[0])
    return ex.wind(*f)


def _exact_sample(case, seed):
    """Point blocks: dense tables at the block's points, one product per order."""
    ex, op, T = _exact_transform(case), case["op"], case["T"]
    lat, lon = _points(case, seed)
    dev = _device()
    x = torch.from_numpy(np.sin(np.deg2rad(lat))).to(dev)
    cosl = torch.from_numpy(np.cos(np.deg2rad(lat))).to(dev)
    lam = torch.from_numpy(np.deg2rad(lon)).to(dev)
    f = [c.to(torch.complex128) for c in _sample_fields(case, seed)]
    if op == "wind":
        f = [ex.inverse_laplacian(c) for c in f]
    two = torch.where(ex.m > 0, 2.0, 1.0)[:, None]
    parts = []
    step = max(64, int(2e9 / (8.0 * (T + 1) ** 2)))
    for p0 in range(0, case["points"], step):
        s = slice(p0, p0 + step)
        P, dP = ex.tables(x[s])
        ang = torch.outer(ex.m, lam[s])
        e = torch.complex(torch.cos(ang), torch.sin(ang)) * two  # (m, p)

        def at(c, table):
            return (ex.waist(c, table).permute(0, 2, 1) * e).real.sum(1)
        if op == "scalar":
            parts.append((at(f[0], P),))
            continue
        g = [(at(c * (1j * ex.m), P) / (ex.a * cosl[s]), at(c, dP) / ex.a) for c in f]
        parts.append(g[0] if op == "gradient"
                     else (g[1][0] - g[0][1], g[0][0] + g[1][1]))
    out = tuple(torch.cat(p, dim=1) for p in zip(*parts))
    return out[0] if op == "scalar" else out


def _exact_vertical(case, seed):
    i, op = _vertical_inputs(case, seed), case["op"]
    d = i["d"].to(torch.complex128)
    x = torch.cat([i["theta"], i["lnps"][None]]).to(torch.complex128)
    mats = {k: v.double().to(torch.complex128) for k, v in i.items()
            if k not in ("d", "theta", "lnps", "k2")}
    k2 = i["k2"].double()[None, :, None]

    def mul(a, y):  # constant matrix on the level axis
        return (a @ y.reshape(y.shape[0], -1)).reshape(-1, *y.shape[1:])

    def per(a, y):  # per-degree matrix (n, i, j) on (j, n, m)
        return torch.bmm(a, y.permute(1, 0, 2).contiguous()).permute(1, 0, 2)
    if op == "tendencies":
        dn, xn = 0.7 * k2 * mul(mats["b"], x), 0.7 * mul(mats["c"], d)
    elif op == "half":
        dn = per(mats["p_d"], d) + per(mats["q_d"], k2 * mul(mats["b"], x))
        xn = per(mats["p_x"], x) + per(mats["q_x"], mul(mats["c"], d))
    elif op == "solve":
        dn = per(mats["inverse"], d + TAU * k2 * mul(mats["b"], x))
        xn = x + TAU * mul(mats["c"], dn)
    else:
        dn = per(mats["inverse"], d + DT * k2 * mul(mats["b"], x)
                 - ALPHA * (1 - ALPHA) * DT * DT * k2 * mul(mats["structure"], d))
        xn = x + DT * mul(mats["c"], (1 - ALPHA) * d + ALPHA * dn)
    dn, xn = dn.clone(), xn.clone()
    if op != "tendencies":
        dn[:, 0, 0], xn[:, 0, 0] = d[:, 0, 0], x[:, 0, 0]
    tri = torch.ones(dn.shape[-2:], device=dn.device, dtype=torch.float64).tril()
    for y in (dn, xn):
        y *= tri
        y[..., 0] = y[..., 0].real.to(y.dtype)
    return dn, xn[:-1], xn[-1]


def exact(case, seed):
    kind = case["kind"]
    if kind == "transform":
        return _exact_one(case, seed)
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind == "vertical":
        return _exact_vertical(case, seed)
    ex, f = _exact_transform(case), _fields(case, seed)
    if kind == "roundtrip":
        u, v = ex.wind(f["vorticity"], f["divergence"])
        return (u, v, ex.inverse(f["temperature"]), ex.inverse(f["lnps"]),
                {n: x.to(torch.complex128) for n, x in f.items()})
    out = {n: [] for n in ENSEMBLE_FIELDS}
    for k in range(case["members"]):
        u, v = ex.wind(f["vorticity"][k], f["divergence"][k])
        out["u"].append(u)
        out["v"].append(v)
        for n, s in (("theta", "theta"), ("qv", "qv"), ("lnps", "log_surface_pressure")):
            out[n].append(ex.inverse(f[s][k].to(torch.complex128)))
        for n, s in (("psi", "vorticity"), ("chi", "divergence")):
            out[n].append(ex.inverse(ex.inverse_laplacian(f[s][k])))
    return {n: torch.stack(x) for n, x in out.items()}
