"""Forms that the fused step chooses between, against the FP64 device path's
unfused potential or the oracle at the sizes where the choice changes."""
import numpy as np
import pytest

import libdft_amd as L
from oracle import pyoracle as po
from tests import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("cbf", [1.0, 0.5], ids=["cbf1", "cbf05"])
@pytest.mark.parametrize("shape", [(128, 128, 128), (256, 128, 128), (64, 512, 128)], ids=lambda s: "x".join(map(str, s)))
def test_potential_forms_agree(shape, cbf, prec):
    """dft_ot_potential (U*q4 summed in k space above 2^21 points, transformed by
    itself up to there) against dft_ot_potential2 on the same density and
    velocities, which always transforms it: FP64 to rounding, FP32 to 2e-5 of the
    largest value (the bound of the potential tests)."""
    step = 0.8
    lib = L.lib()
    w = L.Wave(shape, step, prec)
    f = L.Functional(9, w, 2, 4)
    f.p.c_bfpot = cbf
    w.set(inputs.smooth_modulated(shape, step, f.p.rho0, 0.3))
    a, b = L.CField(shape, step, prec), L.CField(shape, step, prec)
    f.potential(a)
    rho, v = L.RField(shape, step, prec), [L.RField(shape, step, prec) for _ in range(3)]
    lib.grid_wf_density(w.h, rho.h)
    lib.grid_wf_velocity(w.h, v[0].h, v[1].h, v[2].h, L.DFT_EPS)
    lib.dft_ot_potential2(f.h, b.h, rho.h, v[0].h, v[1].h, v[2].h)
    got, want = a.get(), b.get()
    for g, x in ((got.real, want.real), (got.imag, want.imag)):
        assert np.abs(g - x).max() <= (1e-12 if prec == L.GRID_FP64 else 2e-5) * np.abs(want).max()
    for x in (a, b, rho, *v, f, w):
        x.free()


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(4, 8, 16), (8, 4, 64), (16, 16, 8), (32, 8, 4), (64, 4, 16), (128, 8, 8), (256, 4, 8),
                                   (512, 8, 4)], ids=lambda s: "x".join(map(str, s)))
def test_propagation_every_x_length(shape, prec):
    """grid_wf_propagate at every length of the x axis (the kinetic pass and its
    mirrored inverse) against the oracle, in real and imaginary time."""
    step = 0.7
    psi = inputs.smooth_modulated(shape, step, 3e-3, 0.3)
    x = inputs.splitmix64_uniform(int(np.prod(shape)) * 2, 7).reshape(shape + (2,))
    psi = psi * (1 + 0.1 * (x[..., 0] + 1j * x[..., 1]))
    V = 1e-4 * (x[..., 1] + 0.3j * x[..., 0])
    for dt in (150.0, -90j):
        w, p = L.Wave(shape, step, prec), L.CField(shape, step, prec)
        w.set(psi), p.set(V)
        L.lib().grid_wf_propagate(w.h, p.h, L.Complex.of(dt))
        want = po.propagate(psi, V, dt, step)
        assert np.abs(w.get() - want).max() <= (1e-12 if prec == L.GRID_FP64 else 5e-6) * np.abs(want).max()
        w.free(), p.free()


@pytest.mark.parametrize("model", [0, 1, 9], ids=["plain", "kc", "full"])
@pytest.mark.parametrize("shape", [(8, 4, 16), (16, 8, 4), (64, 16, 32), (32, 64, 128)], ids=lambda s: "x".join(map(str, s)))
def test_potential_nyquist_tiles(shape, model):
    """The x-middle's Nyquist tiles where ny is below, at and above a tile's columns,
    and grids whose tile count is no multiple of 8, against the oracle (FP64)."""
    step = 1.1
    o = po.OracleOT(model, shape, step, 2, 4)
    psi = inputs.smooth_modulated(shape, step, o.p.rho0, 0.3)
    w = L.Wave(shape, step, L.GRID_FP64)
    w.set(psi)
    f, p = L.Functional(model, w, 2, 4), L.CField(shape, step, L.GRID_FP64)
    f.potential(p)
    want = o.potential(psi)
    assert np.abs(p.get() - want).max() <= 1e-10 * np.abs(want).max()
    p.free(), f.free(), w.free()


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("model", [1, 9], ids=["kc", "full"])
@pytest.mark.parametrize("shape", [(4, 4, 4), (4, 512, 8), (512, 4, 16), (8, 4, 512)], ids=lambda s: "x".join(map(str, s)))
def test_kc_term1_differences(shape, model, prec):
    """KC term 1 = c rst sum_d D_d J_d, its z part formed on the line and its x and y
    parts by stencils of the next stage, where those wrap within a block, across the
    longest axes and on lines of several wavefronts, against the oracle (which has no
    potential for a box smaller than the Lennard-Jones core: NaN on both sides)."""
    step = 0.9
    o = po.OracleOT(model, shape, step, 2, 4)
    psi = inputs.smooth_modulated(shape, step, o.p.rho0, 0.3)
    w = L.Wave(shape, step, prec)
    w.set(psi)
    f, p = L.Functional(model, w, 2, 4), L.CField(shape, step, prec)
    f.potential(p)
    got, want = p.get(), o.potential(psi)
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), ok) and ok.all() == (min(shape) < max(shape))
    got, want = got[ok], want[ok]
    assert np.abs(got - want).max(initial=0) <= (1e-10 if prec == L.GRID_FP64 else 2e-5) * np.abs(want).max(initial=0)
    p.free(), f.free(), w.free()


def test_potential_forms_agree_512():
    """The k-space sum of U*q4 where an FP64 x line has 512 points."""
    test_potential_forms_agree((512, 64, 128), 1.0, L.GRID_FP64)


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("model", [0, 1, 8, 9, 10, 11], ids=["plain", "kc", "bf", "full", "hd-bf", "hd-full"])
@pytest.mark.parametrize("shape", [(4, 512, 8), (512, 4, 16), (8, 4, 512), (32, 16, 64)], ids=lambda s: "x".join(map(str, s)))
def test_energy_density_of_a_wave_function(shape, model, prec):
    """dft_ot_energy_density (stages fused into the z transforms) at short and long
    axes, lines of part of a wavefront and of several, against the oracle."""
    step = 0.9
    o = po.OracleOT(model, shape, step, 2, 4)
    psi = inputs.smooth_modulated(shape, step, o.p.rho0, 0.3)
    w, e = L.Wave(shape, step, prec), L.RField(shape, step, prec)
    w.set(psi)
    f = L.Functional(model, w, 2, 4)
    f.energy_density(e)
    want = o.energy_density(psi)
    assert np.abs(e.get() - want).max() <= (1e-10 if prec == L.GRID_FP64 else 2e-5) * np.abs(want).max()
    f.free(), e.free(), w.free()


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("model", [0, 1, 3], ids=["plain", "kc", "hd-kc"])
@pytest.mark.parametrize("shape", [(4, 512, 8), (512, 4, 16), (8, 4, 512), (32, 16, 64)], ids=lambda s: "x".join(map(str, s)))
def test_energy_gradient_stages(shape, model, prec):
    """dft_ot_energy_gradient through the z stages, at short and long axes, against
    the oracle, with the bounds of the potential, whose stages these are."""
    step = 0.9
    o = po.OracleOT(model, shape, step, 2, 4)
    psi = inputs.smooth_modulated(shape, step, o.p.rho0, 0.3)
    rho = np.abs(psi) ** 2
    w, r, g = L.Wave(shape, step, prec), L.RField(shape, step, prec), L.RField(shape, step, prec)
    r.set(rho)
    f = L.Functional(model, w, 2, 4)
    L.lib().dft_ot_energy_gradient(f.h, g.h, r.h)
    want = o.energy_gradient(rho)
    assert np.abs(g.get() - want).max() <= (1e-10 if prec == L.GRID_FP64 else 2e-5) * np.abs(want).max()
    for x in (f, r, g, w):
        x.free()


def test_reverse_pass_work_space_is_reusable():
    """The reverse passes' kept work space: repeated and interleaved calls of two
    functionals, a sweep with more checkpoints than the one before, and two threads
    on functionals of their own give the results of a first call, bit for bit."""
    import threading

    def setup(shape, model, seed):
        w = L.Wave(shape, 0.9, L.GRID_FP64)
        f = L.Functional(model, w, 2, 4)
        w.set(inputs.smooth_modulated(shape, 0.9, f.p.rho0, 0.3, seed))
        vb, out = L.CField(shape, 0.9, L.GRID_FP64), L.CField(shape, 0.9, L.GRID_FP64)
        vb.set(inputs.smooth_modulated(shape, 0.9, 1.0, 0.5, seed + 1))
        return w, f, vb, out

    def vjp(s):
        assert L.lib().dft_ot_potential_vjp_psi(s[1].h, s[3].h, s[2].h, s[0].h) == 0
        return s[3].get()

    def sweep(s, k, every):
        return s[1].adjoint_well(-1e-4, 4.0, (0.0, 0.0, 0.0), 0.0, 100.0, k, every)

    a, b = setup((16, 16, 32), 9, 5), setup((32, 16, 16), 1, 9)
    first = vjp(a), vjp(b), sweep(a, 3, 2), sweep(a, 7, 3), sweep(b, 3, 2)
    again = vjp(a), vjp(b), sweep(a, 3, 2), sweep(a, 7, 3), sweep(b, 3, 2)
    for x, y in zip(first, again):
        assert np.array_equal(np.asarray(x, dtype=object), np.asarray(y, dtype=object)) if isinstance(x, tuple) else np.array_equal(x, y)
    got = {}
    ts = [threading.Thread(target=lambda k=k, s=s: got.__setitem__(k, [vjp(s) for _ in range(3)])) for k, s in enumerate((a, b))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in (0, 1):
        assert all(np.array_equal(x, first[k]) for x in got[k])
    for s in (a, b):
        for x in (s[2], s[3], s[1], s[0]):
            x.free()


@pytest.mark.parametrize("prec", [L.GRID_FP64, L.GRID_FP32], ids=["fp64", "fp32"])
def test_reverse_passes_follow_the_model(prec):
    """The functional's model flags are read by every call: reverse passes of one
    functional with the backflow flag cleared and set between them, in both orders,
    give bit for bit what a functional gives whose first reverse pass they are."""
    shape, step = (16, 16, 32), 0.9
    w = L.Wave(shape, step, prec)
    vb, out = L.CField(shape, step, prec), L.CField(shape, step, prec)
    vb.set(inputs.smooth_modulated(shape, step, 1.0, 0.5, 6))

    def fresh():
        f = L.Functional(9, w, 2, 4)
        w.set(inputs.smooth_modulated(shape, step, f.p.rho0, 0.3, 5))
        return f

    def vjp(f, model):
        f.p.model = model
        assert L.lib().dft_ot_potential_vjp_psi(f.h, out.h, vb.h, w.h) == 0
        return out.get()

    def sweep(f, model):
        f.p.model = model
        return np.array([x for y in f.adjoint_well(-1e-4, 4.0, (0.0, 0.0, 0.0), 0.0, 100.0, 3, 2) for x in np.ravel(y)])

    calls = [(c, m) for m in (9, 1) for c in (vjp, sweep)]
    want = {}
    for c, m in calls:
        f = fresh()
        want[c, m] = c(f, m)
        f.free()
    assert not np.array_equal(want[vjp, 9], want[vjp, 1]) and not np.array_equal(want[sweep, 9], want[sweep, 1])
    for order in (calls, calls[::-1]):
        f = fresh()
        for c, m in order + order:
            assert np.array_equal(c(f, m), want[c, m]), (c.__name__, m)
        f.free()
    for x in (vb, out, w):
        x.free()


def test_kept_work_spaces_are_bounded():
    """The work spaces that reverse passes leave with their functionals: 16 GiB in all
    (19 of 1 GiB each here), the last used among them, results as before; dft_ot_trim
    gives all of it back, and the next call does without."""
    import ctypes

    shape, step, lib = (128, 128, 128), 0.9, L.lib()
    GiB, slack = 1 << 30, 1 << 28

    def free():
        a, b = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert lib.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0  # of the HIP runtime the library is linked with
        return a.value

    w = L.Wave(shape, step, L.GRID_FP64)
    vb, out = L.CField(shape, step, L.GRID_FP64), L.CField(shape, step, L.GRID_FP64)
    fs = [L.Functional(9, w, 1, 1) for _ in range(19)]
    w.set(inputs.smooth_modulated(shape, step, fs[0].p.rho0, 0.3, 5))
    vb.set(inputs.smooth_modulated(shape, step, 1.0, 0.5, 6))

    def vjp(f):
        assert lib.dft_ot_potential_vjp_psi(f.h, out.h, vb.h, w.h) == 0
        return out.get()

    want = vjp(fs[0])
    lib.dft_ot_trim()
    base = free()
    vjp(fs[0])
    one = base - free()
    assert one > GiB - slack
    for f in fs:
        vjp(f)
        assert base - free() <= 16 * GiB + slack
    kept = base - free()
    assert kept > 16 * GiB - one - slack
    assert np.array_equal(vjp(fs[-1]), want) and abs(base - free() - kept) <= slack
    assert np.array_equal(vjp(fs[0]), want) and base - free() <= 16 * GiB + slack
    lib.dft_ot_trim()
    assert abs(base - free()) <= slack
    assert np.array_equal(vjp(fs[1]), want)
    for x in (*fs, vb, out, w):
        x.free()


@pytest.mark.parametrize("model", [0, 1, 9], ids=["plain", "kc", "full"])
@pytest.mark.parametrize("shape", [(8, 4, 16), (16, 8, 4), (64, 16, 32), (32, 64, 128)], ids=lambda s: "x".join(map(str, s)))
def test_potential_nyquist_tiles_fp32(shape, model):
    """test_potential_nyquist_tiles in FP32, whose tiles have column counts of their
    own, with the bound of the FP32 potential tests."""
    step = 1.1
    o = po.OracleOT(model, shape, step, 2, 4)
    psi = inputs.smooth_modulated(shape, step, o.p.rho0, 0.3)
    w = L.Wave(shape, step, L.GRID_FP32)
    w.set(psi)
    f, p = L.Functional(model, w, 2, 4), L.CField(shape, step, L.GRID_FP32)
    f.potential(p)
    want = o.potential(psi)
    assert np.abs(p.get() - want).max() <= 2e-5 * np.abs(want).max()
    p.free(), f.free(), w.free()
