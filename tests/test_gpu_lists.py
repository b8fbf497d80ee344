"""The stage on source lists (the form that runs when no mapping is fixed)
against the fused per-element kernels and the per-sweep path, bit for bit:
every basis size the fused stage provides, both interpolation families, the
level-sum cap, FP32 storage, the single operators, and grids on both sides of
the size at which the kernels change (16,384 elements): above it two sources are
in flight instead of four, and the lanes of a target share table blocks."""
import ctypes

import numpy as np
import pytest

import pyadg
import pyoracle
import workloads
from common import first_diff, ic_params, init_both, oracle_run_linear, problem

pytestmark = pytest.mark.gpu


def _steps(s, prob, variant, steps, form=1):
    s.set_kernel_variant(variant)
    s.restore_state(0)
    p = pyadg.Problem.from_buffer_copy(prob)
    p.form, p.max_steps, p.t_start = form, steps, 0.0
    s.run_hyperbolic(p)
    return s.num_elem, s.get()


def _same(a, b, what):
    assert a[0] == b[0], f"{what}: {a[0]} and {b[0]} elements"
    assert np.array_equal(a[1], b[1]), f"{what}: " + first_diff(a[1], b[1])


@pytest.mark.parametrize("dim,k,m,nmax", [(1, 2, 3, 7), (1, 1, 1, 1), (2, 1, 4, 5), (2, 2, 1, 4), (2, 3, 2, 4),
                                          (3, 1, 1, 3), (3, 2, 2, 3), (3, 3, 4, 3), (4, 1, 3, 3), (4, 2, 3, 2),
                                          (4, 3, 4, 1)])
def test_basis_sizes(dim, k, m, nmax):
    print(f"[case] lists dim={dim} k={k} m={m} nmax={nmax}", flush=True)
    s = pyadg.Solution(dim, k, m, nmax, True, nmax)
    s.init_adaptive_intp_builtin(ic_params(1, shift=0.13), 1e10)
    s.save_state(0)
    for flux in (pyadg.FLUX_BURGERS, pyadg.FLUX_VARCOEF):
        p = problem(flux_kind=flux, flux_param=0.4, alpha=[1.3] * dim, wave_speed=[1.0] * dim, cfl=0.05, t_final=1.0,
                    adaptive=0, eps=0.0, eta=0.0, max_steps=0, t_start=0.0)
        got = _steps(s, p, -1, 2)
        _same(got, _steps(s, p, 1, 2), f"flux {flux}, per-element kernels")
        _same(got, _steps(s, p, -1, 2, form=0), f"flux {flux}, per-sweep path")


@pytest.mark.parametrize("herm,fp32,cap", [(1, 0, -1), (0, 1, -1), (0, 0, 3), (1, 1, 4)])
def test_family_precision_cap(herm, fp32, cap):
    print(f"[case] lists herm={herm} fp32={fp32} cap={cap}", flush=True)
    ws = [workloads.c2_burgers(seed=i, nmax=6, level_init=5) for i in (3, 4, 5)]
    s = workloads.make_batch(ws)
    s.set_interpolation(herm)
    s.set_precision(fp32)
    s.set_level_sum_cap(cap)
    s.save_state(0)
    _same(_steps(s, ws[0].problem, -1, 3), _steps(s, ws[0].problem, 3, 3), "per-element kernels")
    # the other family on the same grid rebuilds the lists of its tables
    s.set_interpolation(1 - herm)
    _same(_steps(s, ws[0].problem, -1, 1), _steps(s, ws[0].problem, 3, 1), "other family")


@pytest.mark.parametrize("batch", [60, 110])
def test_few_and_many_elements(batch):
    print(f"[case] lists batch={batch}", flush=True)
    ws = [workloads.c2_burgers(seed=i + 1, nmax=6, level_init=5) for i in range(batch)]
    s = workloads.make_batch(ws)
    assert (s.num_elem > 16384) == (batch == 110), s.num_elem
    s.save_state(0)
    p = pyadg.Problem.from_buffer_copy(ws[0].problem)
    p.adaptive = 0
    _same(_steps(s, p, -1, 1), _steps(s, p, 3, 1), "fixed grid")
    # refinement and coarsening grow and shrink the lists
    _same(_steps(s, ws[0].problem, -1, 2), _steps(s, ws[0].problem, 3, 2), "adaptive")


def _many(dim, k, m, nmax):
    """A batch of more than 16,384 elements with coefficients that fall off with the level."""
    s = pyadg.Solution(dim, k, m, nmax, True, nmax)
    batch = 16384 // s.num_elem + 2
    s.init_batch(batch)
    lev = np.concatenate([s.instance_grid(i)[0] for i in range(batch)])
    u = np.random.default_rng(dim * 100 + k * 10 + m).standard_normal((len(lev), s.K))
    s.set(pyadg.FIELD_UCOE, (u * 0.2 * 2.0 ** (-1.5 * lev.sum(axis=1))[:, None]).reshape(-1))
    assert s.num_elem > 16384
    return s, batch


# phases where the lanes of a target share table blocks: blocks of 4, 6, 9, 12, 16 and 20 values (whole and half
# 16-byte pieces, single words), one and two pieces a lane, FP32 halves; and the widths that are not shared
@pytest.mark.parametrize("dim,k,m,nmax,fp32,herm", [
    (1, 2, 3, 7, 0, 0), (2, 1, 1, 6, 0, 0), (2, 2, 2, 6, 0, 0), (2, 3, 3, 5, 0, 0), (2, 3, 4, 5, 1, 0), (2, 2, 3, 5, 1, 1),
    (2, 2, 3, 6, 0, 1), (3, 1, 1, 4, 0, 0), (3, 2, 2, 4, 0, 0), (3, 2, 2, 4, 1, 0), (3, 2, 3, 4, 0, 0), (3, 2, 3, 4, 1, 0),
    (3, 3, 3, 3, 0, 0), (3, 1, 4, 4, 1, 0), (4, 1, 2, 3, 0, 0), (4, 1, 2, 3, 1, 0), (4, 2, 1, 2, 0, 0)])
def test_many_elements_of_every_block(dim, k, m, nmax, fp32, herm):
    print(f"[case] lists, many elements dim={dim} k={k} m={m} nmax={nmax} fp32={fp32} herm={herm}", flush=True)
    s, batch = _many(dim, k, m, nmax)
    s.set_interpolation(herm)
    s.set_precision(fp32)
    s.save_state(0)
    flux = pyadg.FLUX_BURGERS if dim < 3 else pyadg.FLUX_VARCOEF
    p = problem(flux_kind=flux, flux_param=0.4, alpha=[1.3] * dim, wave_speed=[1.0] * dim, cfl=0.05, t_final=1.0,
                adaptive=0, eps=0.0, eta=0.0, max_steps=0, t_start=0.0)
    got = _steps(s, p, -1, 1)
    _same(got, _steps(s, p, 1, 1), "per-element kernels")
    if not fp32:
        _same(got, _steps(s, p, -1, 1, form=0), "per-sweep path")


@pytest.mark.parametrize("dim,cap", [(2, -1), (2, 4), (3, 3)])
def test_many_elements_with_caps_and_instance_constants(dim, cap):
    print(f"[case] lists, many elements dim={dim} cap={cap}, constants per instance", flush=True)
    s, batch = _many(dim, 2, 3, 6 if dim == 2 else 4)
    s.set_level_sum_cap(cap)
    s.save_state(0)
    r = np.random.default_rng(5)
    s.set_instance_params(coef_scale=r.uniform(0.5, 1.5, (batch, dim)), alpha=r.uniform(0.5, 2.0, (batch, dim)))
    for flux in (pyadg.FLUX_BURGERS, pyadg.FLUX_VARCOEF_SCALED):
        p = problem(flux_kind=flux, flux_param=0.4, alpha=[1.3] * dim, wave_speed=[1.0] * dim, cfl=0.05, t_final=1.0,
                    adaptive=0, eps=0.0, eta=0.0, max_steps=0, t_start=0.0)
        got = _steps(s, p, -1, 1)
        _same(got, _steps(s, p, 3, 1), f"flux {flux}, per-element kernels")
        _same(got, _steps(s, p, -1, 1, form=0), f"flux {flux}, per-sweep path")


@pytest.mark.parametrize("dim,k,m,cap", [(1, 1, 2, -1), (2, 3, 3, -1), (3, 2, 3, 3), (4, 1, 2, -1),
                                         (2, 2, 4, -1), (3, 2, 1, -1)])
def test_single_operators_match_oracle(dim, k, m, cap):
    """Operators on lists, added to what the right-hand side holds, against
    the oracle; the constant-coefficient operator with both signs of speed."""
    print(f"[case] list operators dim={dim} k={k} m={m} cap={cap}", flush=True)
    nmax = 5 if dim < 3 else 4
    g = pyadg.Solution(dim, k, m, nmax, True, nmax)
    o = pyoracle.Oracle(dim, k, m, nmax, True, nmax)
    init_both(g, o, ic_params(1, shift=0.21), 1e10)
    speeds, alpha = [0.7, -1.3, 0.4, -0.2][:dim], [1.2, 0.9, 1.1, 0.8][:dim]
    for s in (g, o):
        s.set_level_sum_cap(cap)
        s.eval_up()
        s.flux(pyadg.FLUX_VARCOEF, [0.3])
        s.fp_to_coe()
        s.rhs_zero()
        s.rhs_linear(speeds)
        s.rhs_lagr_vol()
        s.rhs_lagr_flx()
        s.rhs_penalty(alpha)
        s.rhs_penalty([2 * a for a in alpha])
    for field in (pyadg.FIELD_UP, pyadg.FIELD_RHS):
        a, b = g.get(field), o.get(field)
        assert np.array_equal(a, b), f"field {field}: " + first_diff(a, b)
    g.run_linear(speeds, 1e-3, 2)
    oracle_run_linear(o, speeds, 1e-3, 2)
    for field in (pyadg.FIELD_UCOE, pyadg.FIELD_RHS, pyadg.FIELD_TN):
        a, b = g.get(field), o.get(field)
        assert np.array_equal(a, b), f"field {field}: " + first_diff(a, b)


def _free_bytes():
    """Free memory of the device, from the runtime that the library uses."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


# 168 thousand 4D elements: point values on lists, right-hand side on lists direction by direction (joined it would take
# 32 GiB); 336 thousand: sweep by sweep but for the penalty; 142 thousand 3D elements: direction by direction
@pytest.mark.parametrize("dim,nmax,batch,flux,gib", [(4, 8, 16, pyadg.FLUX_VARCOEF, 12), (4, 8, 16, pyadg.FLUX_BURGERS, 12),
                                                     (4, 8, 32, pyadg.FLUX_VARCOEF, 2), (3, 7, 84, pyadg.FLUX_VARCOEF, 2),
                                                     (3, 7, 84, pyadg.FLUX_BURGERS, 2)])
def test_operators_of_large_grids_keep_their_memory(dim, nmax, batch, flux, gib):
    """On grids whose phase buffers would take gigabytes (4D, k = 2, m = 3: 84 KB an element and room to grow) the
    operators run direction by direction or sweep by sweep: the same values as on a small grid's lists."""
    print(f"[case] operators of a large grid dim={dim} nmax={nmax} batch={batch} flux={flux}", flush=True)

    def rhs(s):
        s.eval_up()
        s.flux(flux, [0.3])
        s.fp_to_coe()
        s.rhs_zero()
        s.rhs_lagr_vol()
        s.rhs_lagr_flx()
        s.rhs_penalty([1.1] * dim)

    one, many = (pyadg.Solution(dim, 2, 3, nmax, True, nmax) for _ in range(2))
    many.init_batch(batch)
    n = one.num_elem * one.K
    assert many.num_elem == batch * one.num_elem and many.num_elem > 130000
    u = np.random.default_rng(3).standard_normal(n) * 0.1
    one.set(pyadg.FIELD_UCOE, u)
    many.set(pyadg.FIELD_UCOE, np.tile(u, batch))
    many.sync()
    before = _free_bytes()
    rhs(many)
    many.sync()
    assert before - _free_bytes() < gib << 30
    rhs(one)
    want, got = one.get(pyadg.FIELD_RHS), many.get(pyadg.FIELD_RHS).reshape(batch, n)
    for i in range(batch):
        assert np.array_equal(got[i], want), f"instance {i}: " + first_diff(got[i], want)


def test_operators_keep_a_plan_per_flux():
    """Operators of one flux and then another, again and again: nothing is planned anew (a plan's upload waits for
    the device), and the values are those of contexts that keep to one flux."""
    kinds = (pyadg.FLUX_BURGERS, pyadg.FLUX_SINCOS)

    def rhs(s, kind):
        s.eval_up()
        s.flux(kind, [0.6])
        s.fp_to_coe()
        s.rhs_zero()
        s.rhs_lagr_vol()
        s.rhs_lagr_flx()
        return s.get(pyadg.FIELD_RHS)

    sols = [pyadg.Solution(2, 2, 3, 5, True, 5) for _ in range(3)]
    for s in sols:
        s.init_adaptive_intp_builtin(ic_params(1, shift=0.13), 1e10)
    want = [rhs(sols[i], kinds[i]) for i in range(2)]
    for i in range(2):
        rhs(sols[2], kinds[i])
    sols[2].profile(True)
    for turn in range(3):
        for i in range(2):
            got = rhs(sols[2], kinds[i])
            assert np.array_equal(got, want[i]), f"turn {turn}, flux {kinds[i]}: " + first_diff(got, want[i])
    assert sols[2].profile_host()["plan"] == 0.0
