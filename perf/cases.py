"""Performance cases of the single-GPU FFT path: what a program that uses this
package runs, from 64^3 transforms to 512^3 ones, each through the plan classes
of pencil_fft_hip with caller-owned device buffers.

listed() names the cases, draw() gives more of the same families, prepare()
makes a case's inputs and plans, run() is one pass and returns every output,
work() the bytes and flops a pass cannot do without, exact() the outputs in
64 bits (dense transform matrices along each axis, or torch.fft on the host
for lines too long for a matrix).
"""
import math
import os
import sys
import tempfile

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "pencil-rs_amd"))

import pencil_fft_hip as pf  # noqa: E402
import pseudo_spectral  # noqa: E402

K = pf.R2rKind
DTYPES = {"f32": (torch.float32, torch.complex64), "f64": (torch.float64, torch.complex128)}
# axis transforms by name; "fft" and "rfft" only appear in mixed plans
KINDS = {"dct1": K.DctI, "dct2": K.DctII, "dct3": K.DctIII, "dct4": K.DctIV, "dst1": K.DstI, "dst2": K.DstII,
         "dst3": K.DstIII, "dst4": K.DstIV, "dht": K.Dht, "fft": pf.AxisTransform.FFT, "rfft": pf.AxisTransform.RFFT}
R2R_NAMES = ("dct1", "dct2", "dct3", "dct4", "dst1", "dst2", "dst3", "dst4", "dht")
# edge lengths of uneven batches
BATCH_EDGES = (48, 60, 64, 84, 96, 112, 128, 160)
NU, DT = 0.01, 1e-3  # the pseudo-spectral model's defaults


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # A small complex transform and its inverse: the call a program with
        # many small grids makes, where launches and latency count.
        {"name": "c2c_64_f64", "kind": "c2c", "shape": "64x64x64", "dtype": "f64", "extra": 1, "permute": True},
        # The headline: a 512^3 real field to its half spectrum and back, as
        # one evaluation of a spectral operator does, in both precisions.
        {"name": "r2c_512_f32", "kind": "r2c", "shape": "512x512x512", "dtype": "f32", "extra": 1, "permute": True},
        {"name": "r2c_512_f64", "kind": "r2c", "shape": "512x512x512", "dtype": "f64", "extra": 1, "permute": True},
        # A ragged grid (edges 2, 3, 5-smooth, one of them odd) of a
        # three-component vector field, without the memory permutation.
        {"name": "r2c_ragged_f32", "kind": "r2c", "shape": "180x225x200", "dtype": "f32", "extra": 3,
         "permute": False},
        # Non-periodic boundary conditions: cosine and sine kinds per axis.
        {"name": "r2r_f32", "kind": "r2r", "shape": "256x384x240", "dtype": "f32", "transforms": "dct2,dst1,dct4"},
        # Real Hartley transforms in double precision.
        {"name": "dht_f64", "kind": "r2r", "shape": "256x384x240", "dtype": "f64", "transforms": "dht,dht,dht"},
        # A channel: two periodic axes and one Chebyshev (Gauss-Lobatto,
        # DCT-I) axis, the Fourier-Fourier-Chebyshev layout of wall-bounded
        # flows.
        {"name": "mixed_channel_f64", "kind": "mixed", "shape": "192x160x129", "dtype": "f64",
         "transforms": "fft,rfft,dct1"},
        # 96 independent uneven problems with three components each, one
        # autotuned batch replayed as a graph.
        {"name": "batch_96_f32", "kind": "batch", "count": 96, "extra": 3, "shapes_seed": 20261202},
        # The gradient of 20 pseudo-spectral steps with respect to the initial
        # field: forward and adjoint transforms, pointwise steps, a checkpoint
        # every 5 steps.
        {"name": "gradient_256_f32", "kind": "gradient", "n": 256, "dtype": "f32", "steps": 20, "every": 5},
        # Batched 1D lines: long power-of-two signals ...
        {"name": "lines_65536_f32", "kind": "lines", "n": 65536, "batch": 128, "dtype": "f32", "real": False},
        # ... and lines of a prime length.
        {"name": "lines_10007_f32", "kind": "lines", "n": 10007, "batch": 838, "dtype": "f32", "real": False},
        # A memory-axis permutation between two stages of a user's own route
        # (z, y, x -> x, z, y).
        {"name": "transpose_c64", "kind": "transpose", "shape": "256x384x240", "element": 8, "src": "210",
         "dst": "021"},
    ]


def _edge(rng, around, styles=("pow2", "smooth", "odd", "any")):
    """An edge length near `around`: a power of two, a 7-smooth length, an
    odd 7-smooth length, or any length."""
    style = rng.choice(styles)
    want = max(16.0, around * 2.0 ** rng.uniform(-0.5, 0.5))
    if style == "any":
        return int(round(want))
    best = None
    for v in range(16, 1025):
        r = v
        for p in ((2,) if style == "pow2" else (2, 3, 5, 7)):
            while r % p == 0:
                r //= p
        if r != 1 or (style == "odd" and v % 2 == 0):
            continue
        if best is None or abs(math.log(v / want)) < abs(math.log(best / want)):
            best = v
    return best


def _shape(rng, lo, hi, styles=("pow2", "smooth", "odd", "any")):
    """Three edges whose product is about 2^lo .. 2^hi."""
    side = 2.0 ** (rng.uniform(lo, hi) / 3)
    return "x".join(str(_edge(rng, side, styles)) for _ in range(3))


def draw(rng):
    kind = rng.choice(("c2c", "r2c", "r2c", "r2r", "mixed", "batch", "gradient", "lines", "lines", "transpose"))
    dtype = rng.choice(("f32", "f64"))
    if kind == "c2c":
        return {"kind": kind, "shape": _shape(rng, 15, 24), "dtype": dtype, "extra": rng.choice((1, 1, 3)),
                "permute": rng.random() < 0.7}
    if kind == "r2c":
        return {"kind": kind, "shape": _shape(rng, 15, 25), "dtype": dtype, "extra": rng.choice((1, 1, 3)),
                "permute": rng.random() < 0.7}
    if kind == "r2r":
        names = ["dht"] * 3 if rng.random() < 0.4 else [rng.choice(R2R_NAMES) for _ in range(3)]
        return {"kind": kind, "shape": _shape(rng, 15, 25), "dtype": dtype, "transforms": ",".join(names)}
    if kind == "mixed":
        return {"kind": kind, "shape": _shape(rng, 15, 24), "dtype": dtype,
                "transforms": "fft,rfft," + rng.choice(R2R_NAMES)}
    if kind == "batch":
        return {"kind": kind, "count": int(round(2 ** rng.uniform(3, 6.58))), "extra": rng.choice((1, 3)),
                "shapes_seed": rng.randrange(1 << 30)}
    if kind == "gradient":
        return {"kind": kind, "n": _edge(rng, 2 ** rng.uniform(5, 8), ("pow2", "smooth", "smooth", "odd")),
                "dtype": dtype, "steps": rng.randrange(4, 21), "every": rng.randrange(2, 6)}
    if kind == "lines":
        n = int(round(2 ** rng.uniform(8, 20)))
        style = rng.choice(("pow2", "smooth", "any"))
        if style == "pow2":
            n = 1 << (n.bit_length() - 1)
        elif style == "smooth":
            n = max(1, n // 240) * 240 if n < 30000 else 2 ** int(math.log2(n / 225)) * 225
        total = 2 ** rng.uniform(18, 23)
        return {"kind": kind, "n": n, "batch": max(1, int(total / n)), "dtype": dtype, "real": rng.random() < 0.4}
    orders = ("012", "021", "102", "120", "201", "210")
    src = rng.choice(orders)
    return {"kind": kind, "shape": _shape(rng, 15, 25), "element": rng.choice((2, 4, 8, 16)), "src": src,
            "dst": rng.choice([o for o in orders if o != src])}


# ------------------------------------------------------------------- inputs
def _dims(case):
    return tuple(int(v) for v in case["shape"].split("x"))


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(n, dtype, seed):
    return torch.rand(n, generator=_generator(seed), device="cuda", dtype=dtype) * 2 - 1


def _normal(n, dtype, seed):
    return torch.randn(n, generator=_generator(seed), device="cuda", dtype=dtype)


def _field(case, seed):
    """The input of a route or line case, flat."""
    rdt, cdt = DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "lines":
        return _normal(case["n"] * case["batch"], rdt if case["real"] else cdt, seed)
    n = math.prod(_dims(case)) * case.get("extra", 1)
    if kind == "c2c":
        return torch.view_as_complex(_uniform(2 * n, rdt, seed).view(-1, 2))
    if kind in ("r2r", "mixed"):
        return _uniform(n, rdt, seed)
    return _normal(n, rdt, seed)


def _batch_shapes(case):
    import random

    rng = random.Random(case["shapes_seed"])
    return [tuple(rng.choice(BATCH_EDGES) for _ in range(3)) for _ in range(case["count"])]


def _batch_layout(case):
    """(offset, elements) of every problem in one buffer, each problem at a
    multiple of 64 elements, and the buffer's length."""
    parts, at = [], 0
    for s in _batch_shapes(case):
        n = math.prod(s) * case["extra"]
        parts.append((at, n))
        at += (n + 63) // 64 * 64
    return parts, at


def _batch_input(case, seed):
    parts, total = _batch_layout(case)
    return parts, total, _normal(total, torch.complex64, seed)


def _transpose_input(case, seed):
    n = math.prod(_dims(case))
    if case["element"] == 2:
        return torch.randint(-32768, 32768, (n,), generator=_generator(seed), device="cuda", dtype=torch.int16)
    return _normal(n, {4: torch.float32, 8: torch.complex64, 16: torch.complex128}[case["element"]], seed)


def _initial_field(case, seed):
    """White noise smoothed by exp(-|k|^2 / 64), in 64 bits."""
    n = case["n"]
    x = _normal(n ** 3, torch.float64, seed).view(n, n, n)
    s = _filter_matrix(n, lambda k: math.exp(-k * k / 64.0))
    return _along(x, [s, s, s]).contiguous().view(-1).to(DTYPES[case["dtype"]][0])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        parts, total, flat = _batch_input(case, seed)
        # a tuning cache of this process alone: it measures its own kernels
        os.environ["PFH_TUNE_CACHE"] = os.path.join(tempfile.gettempdir(), f"pfh_tuning_{os.getpid()}.txt")
        out = torch.zeros(total, dtype=torch.complex64, device="cuda")
        shapes = _batch_shapes(case)
        plan = pf.BatchC2cPlan(shapes, autotune=True, extra_shapes=[(case["extra"],)] * len(shapes))
        return {"kind": kind, "plan": plan, "srcs": [flat[a:a + n] for a, n in parts],
                "dsts": [out[a:a + n] for a, n in parts], "ws": plan.allocate_workspace(), "out": out}
    if kind == "gradient":
        model = pseudo_spectral.PseudoSpectralModel(case["n"], dtype=DTYPES[case["dtype"]][0], nu=NU, dt=DT,
                                                    steps=case["steps"], checkpoint_every=case["every"])
        return {"kind": kind, "model": model, "u0": _initial_field(case, seed)}
    if kind == "transpose":
        x = _transpose_input(case, seed)
        plan = pf.LocalTransposePlan(_dims(case), [int(c) for c in case["src"]], [int(c) for c in case["dst"]],
                                     case["element"])
        return {"kind": kind, "plan": plan, "x": x, "y": torch.empty_like(x)}
    rdt, cdt = DTYPES[case["dtype"]]
    x = _field(case, seed)
    if kind == "lines":
        n, batch = case["n"], case["batch"]
        plan = pf.LocalR2cPlan(n, dtype=rdt) if case["real"] else pf.LocalC2cPlan(n, dtype=cdt)
        out = batch * (n // 2 + 1 if case["real"] else n)
        flags = None
    else:
        dims = _dims(case)
        if kind == "c2c":
            plan = pf.C2cPlan(dims, dtype=cdt, extra_shape=_extra(case), permute_dims=case["permute"])
        elif kind == "r2c":
            plan = pf.R2cPlan(dims, dtype=rdt, extra_shape=_extra(case), permute_dims=case["permute"])
        elif kind == "r2r":
            plan = pf.R2rPlan(dims, [KINDS[t] for t in case["transforms"].split(",")], dtype=rdt)
        else:
            plan = pf.MixedR2cPlan(dims, [KINDS[t] for t in case["transforms"].split(",")], dtype=rdt)
        out = plan.output_elements()
        # spectra that this program made itself: their status is read later
        flags = pf.EXEC_DEFER_STATUS
    complex_out = kind in ("c2c", "r2c", "mixed", "lines")
    return {"kind": kind, "plan": plan, "x": x, "y": torch.empty(out, dtype=cdt if complex_out else rdt, device="cuda"),
            "back": torch.empty_like(x), "ws": plan.allocate_workspace(), "flags": flags}


def _extra(case):
    return (case["extra"],) if case["extra"] > 1 else ()


# --------------------------------------------------------------------- runs
def run(state):
    """One pass: a transform and its normalized inverse (routes and lines), a
    batch's forward, a loss and its gradient, or a permutation."""
    kind, plan = state["kind"], state.get("plan")
    if kind == "batch":
        plan.forward(state["srcs"], state["dsts"], state["ws"], use_graph=True)
        return state["out"]
    if kind == "gradient":
        loss, grad = state["model"].gradient(state["u0"])
        return [loss, grad]
    if kind == "transpose":
        return plan.execute(state["x"], state["y"])
    plan.forward(state["x"], state["y"], state["ws"])
    if state["flags"] is None:
        plan.inverse(state["y"], state["back"], state["ws"])
    else:
        plan.inverse(state["y"], state["back"], state["ws"], flags=state["flags"])
    return [state["y"], state["back"]]


def work(case):
    """Each input read once and each output written once; 5 n log2 n flops per
    complex line of n points, half of that per real one."""
    kind = case["kind"]
    if kind == "batch":
        n = [math.prod(s) * case["extra"] for s in _batch_shapes(case)]
        flops = sum(5 * v * math.log2(v / case["extra"]) for v in n)
        return {"bytes": 16 * sum(n), "flops": flops}
    if kind == "transpose":
        return {"bytes": 2 * case["element"] * math.prod(_dims(case)), "flops": 0}
    real = 4 if case["dtype"] == "f32" else 8
    if kind == "gradient":
        n, steps = case["n"], case["steps"]
        # per step: forward sweep, recomputed step and reverse sweep, two
        # transforms each; the field, its gradient and the checkpoints
        fields = 2 + 2 * math.ceil(steps / case["every"])
        return {"bytes": fields * n ** 3 * real, "flops": 6 * steps * 2.5 * n ** 3 * math.log2(n ** 3)}
    if kind == "lines":
        n, batch = case["n"], case["batch"]
        x = n * real * (1 if case["real"] else 2)
        y = (n // 2 + 1 if case["real"] else n) * 2 * real
        return {"bytes": 2 * batch * (x + y), "flops": 2 * batch * (2.5 if case["real"] else 5) * n * math.log2(n)}
    dims, extra = _dims(case), case.get("extra", 1)
    n = math.prod(dims) * extra
    flops = 2 * 2.5 * n * math.log2(n / extra)
    if kind == "c2c":
        return {"bytes": 4 * n * 2 * real, "flops": 2 * flops}
    if kind == "r2r":
        return {"bytes": 4 * n * real, "flops": flops}
    axis = 2 if kind == "r2c" else 1
    half = n // dims[axis] * (dims[axis] // 2 + 1)
    return {"bytes": 2 * (n * real + half * 2 * real), "flops": flops}


# -------------------------------------------------------------------- exact
def _index(n):
    return torch.arange(n, dtype=torch.int64, device="cuda")


def _turns(p, q, fn):
    """fn(pi p / q) of integer arrays, reduced to one turn before the multiplication."""
    return fn((p % (2 * q)).double() * (math.pi / q))


def _matrix(name, n):
    """The unnormalized transform matrix [output, input] of one axis in 64
    bits, by the definitions of FFTW's kinds."""
    j, cos, sin = _index(n), torch.cos, torch.sin
    k = j[:, None]
    if name in ("fft", "rfft"):
        if name == "rfft":
            k = k[: n // 2 + 1]
        return torch.complex(_turns(2 * j * k, n, cos), -_turns(2 * j * k, n, sin))
    if name == "dht":
        return _turns(2 * j * k, n, cos) + _turns(2 * j * k, n, sin)
    if name == "dct1":
        m = 2 * _turns(j * k, n - 1, cos)
        m[:, 0] *= 0.5
        m[:, -1] *= 0.5
        return m
    if name == "dct2":
        return 2 * _turns((2 * j + 1) * k, 2 * n, cos)
    if name == "dct3":
        m = 2 * _turns(j * (2 * k + 1), 2 * n, cos)
        m[:, 0] *= 0.5
        return m
    if name == "dct4":
        return 2 * _turns((2 * j + 1) * (2 * k + 1), 4 * n, cos)
    if name == "dst1":
        return 2 * _turns((j + 1) * (k + 1), n + 1, sin)
    if name == "dst2":
        return 2 * _turns((2 * j + 1) * (k + 1), 2 * n, sin)
    if name == "dst3":
        m = 2 * _turns((j + 1) * (2 * k + 1), 2 * n, sin)
        m[:, -1] *= 0.5
        return m
    return 2 * _turns((2 * j + 1) * (2 * k + 1), 4 * n, sin)  # dst4


def _filter_matrix(n, fn):
    """The circulant matrix of the periodic filter fn(k) on an axis of n points."""
    j = _index(n)
    k = torch.where(j <= n // 2, j, j - n).tolist()
    f = torch.tensor([fn(v) for v in k], dtype=torch.float64, device="cuda")
    row = (_turns(2 * j[:, None] * j, n, torch.cos) * f).sum(1) / n
    return row[(j[:, None] - j) % n]


def _along(x, matrices):
    """The matrices applied along the last axes of x, the last axis first."""
    for a in range(len(matrices) - 1, -1, -1):
        m, axis = matrices[a], x.dim() - len(matrices) + a
        moved = x.movedim(axis, -1)
        flat = moved.reshape(-1, moved.shape[-1])
        if m.is_complex() and not flat.is_complex():
            t = m.t()
            y = torch.complex(flat @ t.real.contiguous(), flat @ t.imag.contiguous())
        else:
            y = flat @ m.t().contiguous().to(flat.dtype)
        x = y.reshape(*moved.shape[:-1], m.shape[0]).movedim(-1, axis)
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "transpose":
        x = _transpose_input(case, seed)
        src, dst = [int(c) for c in case["src"]], [int(c) for c in case["dst"]]
        dims = _dims(case)
        y = x.view([dims[a] for a in src]).permute([src.index(a) for a in dst]).reshape(-1)
        if case["element"] == 2:
            return y
        return y.to(torch.complex128 if y.is_complex() else torch.float64)
    if kind == "gradient":
        n, steps = case["n"], case["steps"]
        gamma = 0.1 * DT
        a = _filter_matrix(n, lambda k: math.exp(-NU * DT * k * k))
        u = _initial_field(case, seed).double().view(n, n, n)
        ws = []
        for _ in range(steps):
            w = _along(u, [a, a, a]).contiguous()
            ws.append(w)
            u = w + gamma * w * w
        g = 2.0 * u
        for w in reversed(ws):
            g = _along(g * (1 + 2 * gamma * w), [a, a, a])
        return [float((u * u).sum()), g.reshape(-1)]
    if kind == "batch":
        parts, total, flat = _batch_input(case, seed)
        host = flat.cpu()
        out = torch.zeros(total, dtype=torch.complex128)
        for (at, n), s in zip(parts, _batch_shapes(case)):
            x = host[at:at + n].to(torch.complex128).view(-1, *s)
            y = torch.fft.fftn(x, dim=(1, 2, 3)).permute(0, 3, 2, 1)
            out[at:at + n] = y.reshape(-1)
        return out
    x = _field(case, seed)
    wide = x.to(torch.complex128 if x.is_complex() else torch.float64)
    if kind == "lines":
        lines = wide.view(case["batch"], case["n"]).cpu()
        y = torch.fft.rfft(lines) if case["real"] else torch.fft.fft(lines)
        return [y.reshape(-1), wide]
    dims = _dims(case)
    names = {"c2c": ["fft"] * 3, "r2c": ["fft", "fft", "rfft"]}.get(kind) or case["transforms"].split(",")
    field = wide.view(case.get("extra", 1), *dims)
    y = _along(field, [_matrix(t, n) for t, n in zip(names, dims)])
    if case.get("permute", True):
        y = y.permute(0, 3, 2, 1)  # output memory order: the axes reversed
    return [y.reshape(-1), wide]
