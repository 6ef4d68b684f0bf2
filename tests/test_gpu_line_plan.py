"""GPU parity of the compile-time line plans (pfh_line.hip): every planned
length on row lines with a partial last tile, and routes whose stages take
column sides with partial tiles, in every mode, against numpy / the oracle.
Bounds: the suite's 2e-6 (f32) and 1e-12 (f64) relative L2, which hold for
these lengths with a rounding error of a few eps per radix pass; 4x over the
three stages of a route."""
import numpy as np
import pytest
import torch

import oracle as O
import pencil_fft_hip as pf
from util import complex_of, rel_l2, tol, uniform_complex, uniform_real

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64]
OPS = [O.FORWARD, O.INVERSE, O.BACKWARD, O.ADJ_FORWARD, O.ADJ_INVERSE, O.ADJ_BACKWARD]


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


LENGTHS = [n for n in range(8, 513) if _smooth(n)] + [385]


def _tdev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("dt", DTYPES)
def test_every_length_c2c_and_half_length_real(gpu, dt):
    rng = np.random.default_rng(31)
    for n in LENGTHS:
        lines = 256 // n * 2 + 7  # a partial last tile
        x = uniform_complex(rng, (lines, n), complex_of(dt))
        plan = pf.LocalC2cPlan(n, dtype=torch.from_numpy(x).dtype)
        got = _host(plan.forward(_tdev(x)))
        assert rel_l2(got, np.fft.fft(x.astype(np.complex128))) <= tol(dt), n
        got = _host(plan.inverse(_tdev(x)))
        assert rel_l2(got, np.fft.ifft(x.astype(np.complex128))) <= tol(dt), n
        r = uniform_real(rng, (lines, 2 * n), dt)
        rplan = pf.LocalR2cPlan(2 * n, dtype=torch.from_numpy(r).dtype)
        spec = rplan.forward(_tdev(r))
        assert rel_l2(_host(spec), np.fft.rfft(r.astype(np.float64))) <= tol(dt), n
        assert rel_l2(_host(rplan.inverse(spec)), r) <= 2 * tol(dt), n


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("kind", list(range(1, 10)))
def test_real_kinds_on_row_lines(gpu, kind, dt):
    """n, n / 2, 2n, n - 1 or n + 1 is a planned length: even and odd lines,
    both parities of the half length, forward and inverse."""
    rng = np.random.default_rng(kind)
    for n in (16, 17, 19, 24, 30, 45, 50, 64, 65, 63, 75, 126, 129, 180, 225, 240, 256, 384, 385, 512):
        x = uniform_real(rng, (11, n), dt)
        td = torch.from_numpy(x).dtype
        plan = pf.LocalDhtPlan(n, dtype=td) if kind == 9 else pf.LocalR2rPlan(n, kind, dtype=td)
        for op, fn in ((O.FORWARD, plan.forward), (O.INVERSE, plan.inverse)):
            ref = O.r2r_lines(x.astype(np.float64), kind, op)
            assert rel_l2(_host(fn(_tdev(x))), ref) <= tol(dt), (n, kind, op)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("kind", [4, 8])
@pytest.mark.parametrize("m", [70, 72, 75, 84, 96, 98, 105, 112, 120, 128])
def test_type_four_lines_on_either_plan(gpu, m, kind, dt):
    """DCT-IV / DST-IV lines of 2m points: the plan that every kind shares where
    12 divides m, the one with twice the threads elsewhere; one partial tile
    and several."""
    rng = np.random.default_rng(m)
    for lines in (3, 67):
        x = uniform_real(rng, (lines, 2 * m), dt)
        plan = pf.LocalR2rPlan(2 * m, kind, dtype=torch.from_numpy(x).dtype)
        for op, fn in ((O.FORWARD, plan.forward), (O.INVERSE, plan.inverse)):
            ref = O.r2r_lines(x.astype(np.float64), kind, op)
            assert rel_l2(_host(fn(_tdev(x))), ref) <= tol(dt), (lines, op)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("permute", [True, False])
@pytest.mark.parametrize("kinds", [(1, 2, 3), (4, 5, 6), (7, 8, 9), (9, 1, 5)])
def test_real_kinds_on_column_sides(gpu, kinds, permute, dt):
    shape = (25, 36, 49)
    rng = np.random.default_rng(sum(kinds))
    td = torch.float32 if dt == np.float32 else torch.float64
    plan = pf.R2rPlan(shape, list(kinds), dtype=td, extra_shape=(2,), permute_dims=permute)
    x = uniform_real(rng, 2 * int(np.prod(shape)), dt)
    for op in OPS:
        ref = O.transform(O.KIND_R2R, x.astype(np.float64), op, shape=shape, extra=2, r2r=list(kinds),
                          permute_dims=permute)
        assert rel_l2(_host(plan.execute(op, _tdev(x))), ref) <= 4 * tol(dt), op


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("permute", [True, False])
@pytest.mark.parametrize("shape", [(35, 27, 90), (50, 15, 28), (9, 200, 18)])
def test_complex_and_half_complex_routes(gpu, shape, permute, dt):
    rng = np.random.default_rng(shape[0])
    td = torch.float32 if dt == np.float32 else torch.float64
    cd = torch.complex64 if dt == np.float32 else torch.complex128
    n = 3 * int(np.prod(shape))
    for kind, plan in ((O.KIND_C2C, pf.C2cPlan(shape, dtype=cd, extra_shape=(3,), permute_dims=permute)),
                       (O.KIND_R2C, pf.R2cPlan(shape, dtype=td, extra_shape=(3,), permute_dims=permute))):
        x = uniform_complex(rng, n, complex_of(dt)) if kind == O.KIND_C2C else uniform_real(rng, n, dt)
        wide = x.astype(np.complex128 if kind == O.KIND_C2C else np.float64)
        spec = O.transform(kind, wide, O.FORWARD, shape=shape, extra=3, permute_dims=permute)
        for op in OPS:
            fwd_like = op in (O.FORWARD, O.ADJ_INVERSE, O.ADJ_BACKWARD)
            src = x if fwd_like else spec.astype(complex_of(dt))
            ref = O.transform(kind, src.astype(np.complex128 if np.iscomplexobj(src) else np.float64), op,
                              shape=shape, extra=3, permute_dims=permute)
            assert rel_l2(_host(plan.execute(op, _tdev(src))), ref) <= 4 * tol(dt), (kind, op)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("n", [16500, 20160, 32768, 65536, 100000, 122500, 1031, 2 * 1031, 10007])
def test_pieces_of_long_lines(gpu, n, dt):
    """Splits whose pieces have line plans (16500: one of them does not),
    Bluestein lines, odd line counts and partial last tiles; equal chunks."""
    rng = np.random.default_rng(n)
    for lines in (1, 5):
        x = uniform_complex(rng, (lines, n), complex_of(dt))
        plan = pf.LocalC2cPlan(n, dtype=torch.from_numpy(x).dtype)
        ref = np.fft.fft(x.astype(np.complex128))
        assert rel_l2(_host(plan.forward(_tdev(x))), ref) <= tol(dt), lines
        assert rel_l2(_host(plan.inverse(_tdev(ref.astype(complex_of(dt))))), x) <= tol(dt), lines


@pytest.mark.parametrize("dt", DTYPES)
def test_odd_real_lines(gpu, dt):
    """Odd R2C / C2R lines on the line plans, both directions and adjoints'
    weights (route operations), row and column sides."""
    rng = np.random.default_rng(41)
    for n in (9, 15, 35, 63, 105, 225, 343, 441, 945):
        r = uniform_real(rng, (9, n), dt)
        plan = pf.LocalR2cPlan(n, dtype=torch.from_numpy(r).dtype)
        spec = plan.forward(_tdev(r))
        assert rel_l2(_host(spec), np.fft.rfft(r.astype(np.float64))) <= tol(dt), n
        assert rel_l2(_host(plan.inverse(spec)), r) <= 2 * tol(dt), n
    for shape, permute in (((21, 10, 45), True), ((12, 35, 27), False)):
        plan = pf.R2cPlan(shape, dtype=torch.from_numpy(r).dtype, permute_dims=permute)
        x = uniform_real(rng, int(np.prod(shape)), dt)
        spec = O.transform(O.KIND_R2C, x.astype(np.float64), O.FORWARD, shape=shape, permute_dims=permute)
        for op in OPS:
            fwd_like = op in (O.FORWARD, O.ADJ_INVERSE, O.ADJ_BACKWARD)
            src = x if fwd_like else spec.astype(complex_of(dt))
            ref = O.transform(O.KIND_R2C, src.astype(np.complex128 if np.iscomplexobj(src) else np.float64), op,
                              shape=shape, permute_dims=permute)
            assert rel_l2(_host(plan.execute(op, _tdev(src))), ref) <= 4 * tol(dt), (shape, op)


BLUE = [17, 19, 22, 26, 33, 37, 51, 61, 74, 89, 97, 101, 121, 127, 131, 143, 194, 233, 251, 257, 319, 401, 461, 511]


@pytest.mark.parametrize("dt", DTYPES)
def test_lengths_without_a_plan(gpu, dt):
    """Bluestein inside the workgroup: primes and lengths with a prime factor
    from 11 on, every complex and real mode, rows with a partial last tile.
    The two extra transforms and three products stay within twice the bound."""
    rng = np.random.default_rng(43)
    cd = complex_of(dt)
    for n in BLUE:
        x = uniform_complex(rng, (13, n), cd)
        plan = pf.LocalC2cPlan(n, dtype=torch.from_numpy(x).dtype)
        assert rel_l2(_host(plan.forward(_tdev(x))), np.fft.fft(x.astype(np.complex128))) <= 2 * tol(dt), n
        assert rel_l2(_host(plan.inverse(_tdev(x))), np.fft.ifft(x.astype(np.complex128))) <= 2 * tol(dt), n
        for rn in (n, 2 * n):
            r = uniform_real(rng, (13, rn), dt)
            rplan = pf.LocalR2cPlan(rn, dtype=torch.from_numpy(r).dtype)
            spec = rplan.forward(_tdev(r))
            assert rel_l2(_host(spec), np.fft.rfft(r.astype(np.float64))) <= 2 * tol(dt), rn
            assert rel_l2(_host(rplan.inverse(spec)), r) <= 4 * tol(dt), rn
    for n in (17, 34, 97, 110, 131, 202, 233, 466):
        x = uniform_real(rng, (11, n), dt)
        td = torch.from_numpy(x).dtype
        for kind in range(1, 10):
            plan = pf.LocalDhtPlan(n, dtype=td) if kind == 9 else pf.LocalR2rPlan(n, kind, dtype=td)
            for op, fn in ((O.FORWARD, plan.forward), (O.INVERSE, plan.inverse)):
                ref = O.r2r_lines(x.astype(np.float64), kind, op)
                assert rel_l2(_host(fn(_tdev(x))), ref) <= 2 * tol(dt), (n, kind, op)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("permute", [True, False])
def test_routes_without_a_plan(gpu, permute, dt):
    rng = np.random.default_rng(47)
    td = torch.float32 if dt == np.float32 else torch.float64
    cd = torch.complex64 if dt == np.float32 else torch.complex128
    for kind, shape, r2r in ((O.KIND_C2C, (37, 22, 29), None), (O.KIND_R2C, (26, 41, 34), None),
                             (O.KIND_R2C, (33, 17, 53), None), (O.KIND_R2R, (31, 46, 38), [2, 5, 9]),
                             (O.KIND_R2R, (23, 58, 39), [3, 1, 8])):
        n = int(np.prod(shape))
        if kind == O.KIND_C2C:
            plan = pf.C2cPlan(shape, dtype=cd, permute_dims=permute)
        elif kind == O.KIND_R2C:
            plan = pf.R2cPlan(shape, dtype=td, permute_dims=permute)
        else:
            plan = pf.R2rPlan(shape, r2r, dtype=td, permute_dims=permute)
        x = uniform_complex(rng, n, complex_of(dt)) if kind == O.KIND_C2C else uniform_real(rng, n, dt)
        kw = {"r2r": r2r} if r2r else {}
        wide = x.astype(np.complex128 if kind == O.KIND_C2C else np.float64)
        spec = O.transform(kind, wide, O.FORWARD, shape=shape, permute_dims=permute, **kw)
        for op in OPS:
            fwd_like = op in (O.FORWARD, O.ADJ_INVERSE, O.ADJ_BACKWARD)
            src = x if fwd_like or kind == O.KIND_R2R else spec.astype(complex_of(dt))
            ref = O.transform(kind, src.astype(np.complex128 if np.iscomplexobj(src) else np.float64), op, shape=shape,
                              permute_dims=permute, **kw)
            assert rel_l2(_host(plan.execute(op, _tdev(src))), ref) <= 6 * tol(dt), (kind, shape, op)


@pytest.mark.parametrize("tiles", [63, 64, 127, 128, 129, 257, 1023, 1024, 1025, 1300])
def test_tile_runs_cover_every_line(gpu, tiles):
    """Runs of tiles per XCD: tile counts around the multiples of a round of
    runs, on k_line_plan (15), k_line_blue (17) and the generic kernel (11)."""
    rng = np.random.default_rng(tiles)
    for n, per in ((15, 256 // 3), (17, 256 // 9), (11, 128)):
        lines = tiles * per - 1
        x = uniform_complex(rng, (lines, n), np.complex64)
        got = _host(pf.LocalC2cPlan(n, dtype=torch.complex64).forward(_tdev(x)))
        ref = np.fft.fft(x.astype(np.complex128))
        per_line = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
        assert per_line.max() <= 4 * tol(np.float32), (n, int(per_line.argmax()))
