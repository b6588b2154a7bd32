"""One-component 2D rows on the matrix cores (k_plane) against the separate kernels (TMI_PLANE2D=0).

Tolerance: the same FP64 (FP32) products summed in another order; 1e-12 (1e-5) of the row block's
largest value, the parity bounds of the separate kernels themselves.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tramonto_amd.batch import BatchSpec, DeviceBatch, rough_slit_pore_batch_2d  # noqa: E402
from tramonto_amd.device import PREC_MIXED, DeviceProblem  # noqa: E402
from tramonto_amd.problem import (IN_BULK, IN_WALL, PERIODIC, REFLECT, ProblemSpec, SplitMix64, rough_slit_pore_2d,  # noqa: E402
                                  rough_wall_2d, small_case)
from linear_update import check_batch_step, check_update, row_scale  # noqa: E402


def _box(nx, ny, bc, cut=1.5, dx=0.1, func=0, seed=3):
    rho = 0.5 * (1 + 0.2 * SplitMix64(seed).uniform(nx * ny, -1, 1))
    return ProblemSpec(name="box", ndim=2, ncomp=1, nx=[nx, ny], dx=[dx, dx], bc=bc, type_func=func,
                       type_attr=0 if cut else -1, hs_diam=[1.0], sigma_ff=np.ones((1, 1)), eps_ff=np.full((1, 1), 0.8),
                       cut_ff=np.full((1, 1), cut), rho_b=[0.5], rho0=rho[None, :])


SPECS = {
    "2d_periodic": lambda: small_case("2d_periodic"),
    "2d_wall_reflect": lambda: small_case("2d_wall_reflect"),
    "2d_wall_fmt4": lambda: small_case("2d_wall_fmt4"),
    "2d_rough_wall": lambda: small_case("2d_rough_wall"),
    "ragged": lambda: _box(33, 47, [[PERIODIC, PERIODIC], [IN_BULK, REFLECT]], func=2),
    "reflect_both": lambda: _box(17, 31, [[REFLECT, REFLECT], [REFLECT, IN_WALL]]),
    "hard_only": lambda: _box(18, 16, [[IN_BULK, IN_WALL], [PERIODIC, PERIODIC]], cut=0.0),
    "reach_plus_one": lambda: _box(20, 35, [[IN_BULK, IN_BULK], [IN_WALL, IN_BULK]], cut=0.6),   # attraction reach FMT + 1
    "fine": lambda: rough_wall_2d(seed=5, nx=113, ny=112, dx=0.05),   # one 16-wave workgroup per CU
}


def _compare(a, b, blocks, tol):
    for lo, hi in blocks:
        if lo < hi:
            scale = float(a[lo:hi].abs().max())
            assert float((a[lo:hi] - b[lo:hi]).abs().max()) <= tol * scale, (lo, hi)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", list(SPECS) + ["batch", "batch_walls"])
def test_plane_matches_separate_kernels(kind, monkeypatch):
    batch = kind.startswith("batch")
    monkeypatch.setenv("TMI_PRECOND", "diag")
    if batch:
        spec = rough_slit_pore_batch_2d(npores=3, seed=4, nx=53, h_range=(3.0, 5.0))
        if kind == "batch_walls":
            spec = BatchSpec([rough_slit_pore_2d(seed=i, nx=37, ny=ny, eps_ff=0.5) for i, ny in enumerate((33, 48, 49))])
            for p in spec.pores:
                p.bc = [[IN_WALL, IN_WALL], [IN_WALL, IN_WALL]]
        make = lambda: DeviceBatch(spec)   # noqa: E731
    else:
        spec = SPECS[kind]()
        make = lambda: DeviceProblem(spec)   # noqa: E731
    monkeypatch.setenv("TMI_MF_FFT", "0")
    monkeypatch.setenv("TMI_FMT_FFT", "0")
    monkeypatch.setenv("TMI_PLANE2D", "0")
    rows = make()
    for v in ("TMI_MF_FFT", "TMI_FMT_FFT"):
        monkeypatch.delenv(v)
    monkeypatch.setenv("TMI_PLANE2D", "2")   # the matrix-core form without the timing against the others
    plane = make()
    # the forms compared are two forms
    assert rows.row_form()[0] == 0 and plane.row_form() == (2, 16 if kind == "fine" else 8)
    C, R = 1, 8
    x = rows.initial_state()
    blocks = ((0, C), (C, C + R), (C + R, x.shape[0]))
    _compare(x, plane.initial_state(), blocks, 1e-12)
    g = torch.Generator(device="cuda").manual_seed(1)
    noise = lambda: 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1   # noqa: E731
    x[C:] *= 1.0 + 0.01 * noise()[C:]
    Fa, sa = rows.fill_residual(x)
    Fb, sb = plane.fill_residual(x)
    _compare(Fa, Fb, blocks, 1e-12)
    assert abs(sa - sb) <= 1e-12 * abs(sa)
    v = noise()
    _compare(rows.apply_jacobian(x, v), plane.apply_jacobian(x, v), blocks, 1e-12)
    _compare(rows.apply_jacobian(x, v, fp32=True), plane.apply_jacobian(x, v, fp32=True), blocks, 1e-5)
    ms = plane.fill_residual_timed(x, reps=2)   # the stage of the launch that a fill runs
    assert ms[0] > 0 and not ms[1:].any() and (rows.fill_residual_timed(x, reps=2)[[0, 1, 3, 4]] > 0).all()
    # Schur product, right-hand side and back-substitution: one Newton update
    da, _ = rows.schur_solve(x, Fa, rtol=1e-12)
    db, _ = plane.schur_solve(x, Fa, rtol=1e-12)
    _compare(da, db, blocks, 1e-8)
    dm, _ = plane.schur_solve(x, Fa, rtol=1e-8, restart=500, maxit=2500, precision=PREC_MIXED)   # hard systems among them
    check_update(rows, x, Fa, dm, C, row_scale(rows, x, C, g), mixed=True)


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("walls", [False, True])
def test_batched_step_solves_each_piece(walls, mixed, monkeypatch):
    """Batched Schur products of 2D pieces: walls between pieces (and at their x ends), tiles of finished
    pieces skipped."""
    spec = rough_slit_pore_batch_2d(npores=4, seed=4, nx=53, h_range=(3.0, 5.0))
    if walls:
        for p in spec.pores:
            p.bc = [[IN_WALL, IN_WALL], [IN_WALL, IN_WALL]]
    monkeypatch.setenv("TMI_PLANE2D", "0")
    rows = DeviceBatch(spec)
    monkeypatch.setenv("TMI_PLANE2D", "2")
    plane = DeviceBatch(spec)
    assert rows.row_form()[0] == 0 and plane.row_form()[0] == 2
    check_batch_step(plane, rows, mixed, torch.Generator(device="cuda").manual_seed(2))


@pytest.mark.gpu
@pytest.mark.parametrize("env,forms", [({"TMI_MF_FFT": "1"}, (1, None)), ({"TMI_FMT_FFT": "1"}, (None, 2)),
                                       ({"TMI_MF_FFT": "0"}, (0, None)), ({"TMI_FMT_FFT": "0"}, (None, 0))])
def test_forced_forms_leave_the_matrix_core_rows(env, forms, monkeypatch):
    """TMI_MF_FFT and TMI_FMT_FFT force a form of the separate sums, in batches the direct one."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    dp = DeviceProblem(small_case("2d_rough_wall"))
    assert dp.row_form()[0] == 0
    for got, want in zip((dp.info.mf_fft, dp.info.fmt_fft), forms):
        assert want is None or got == want
    if "0" in env.values():
        assert DeviceBatch(rough_slit_pore_batch_2d(npores=2, seed=4, nx=53, h_range=(3.0, 4.0))).row_form()[0] == 0


@pytest.mark.gpu
def test_reference_jacobian_beside_the_matrix_core_rows(monkeypatch):
    """Where the timing picks the matrix-core rows, products with the reference's Jacobian run in the separate
    forms that the timing kept beside them: the same rows as with those forms forced."""
    from tramonto_amd.device import JAC_REFERENCE
    spec = _box(64, 64, [[PERIODIC, PERIODIC], [PERIODIC, PERIODIC]], cut=2.5, func=3)
    plane = DeviceProblem(spec)
    assert plane.row_form()[0] == 2 and (plane.info.mf_fft, plane.info.fmt_fft, plane.info.fft_xreg) == (0, 0, 0)
    with pytest.raises(RuntimeError):
        plane.fft_timed(0, 1)   # no such launches in its fill
    monkeypatch.setenv("TMI_FMT_FFT", "0")
    monkeypatch.setenv("TMI_MF_FFT", "0")
    direct = DeviceProblem(spec)
    x = direct.initial_state()
    g = torch.Generator(device="cuda").manual_seed(4)
    v = 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1
    for p in (plane, direct):
        p.set_jacobian(JAC_REFERENCE)
    _compare(direct.apply_jacobian(x, v), plane.apply_jacobian(x, v), ((0, 1), (1, 9), (9, 10)), 1e-12)
    F, _ = direct.fill_residual(x)
    da, _ = direct.schur_solve(x, F, rtol=1e-12)
    db, _ = plane.schur_solve(x, F, rtol=1e-12)
    _compare(da, db, ((0, 1), (1, 9), (9, 10)), 1e-8)


@pytest.mark.gpu
@pytest.mark.parametrize("cut", [0.0, 2.5])
def test_rows_alone_beside_the_matrix_core_fill(cut, monkeypatch):
    """Initial fields and back-substitution run in whichever form the set-up timed faster for the rows alone
    (hard spheres: mostly the separate kernels beside a matrix-core fill): the forced forms' rows."""
    spec = _box(64, 48, [[PERIODIC, PERIODIC], [IN_WALL, IN_BULK]], cut=cut)
    plane = DeviceProblem(spec)
    assert plane.row_form()[0] == 2
    monkeypatch.setenv("TMI_FMT_FFT", "0")
    monkeypatch.setenv("TMI_MF_FFT", "0")
    direct = DeviceProblem(spec)
    x = direct.initial_state()
    blocks = ((0, 1), (1, 9), (9, x.shape[0]))
    _compare(x, plane.initial_state(), blocks, 1e-12)
    F, _ = direct.fill_residual(x)
    da, _ = direct.schur_solve(x, F, rtol=1e-12)
    db, _ = plane.schur_solve(x, F, rtol=1e-12)
    _compare(da, db, blocks, 1e-8)
