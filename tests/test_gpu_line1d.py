"""1D rows in one launch (k_line) against the separate row kernels (TMI_LINE1D=0).

Tolerance: the same FP64 (FP32) products summed in another order, at most a few hundred terms per row:
1e-12 (1e-5) of the row block's largest value, the parity bounds of the row kernels themselves.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tramonto_amd.batch import DeviceBatch, slit_pore_batch  # noqa: E402
from tramonto_amd.device import PREC_MIXED, DeviceProblem  # noqa: E402
from tramonto_amd.problem import (FMT3, IN_BULK, IN_WALL, PERIODIC, REFLECT, hard_wall_1d, slit_pore_1d,  # noqa: E402
                                  small_case)
from linear_update import check_batch_step, check_update, row_scale  # noqa: E402


def _single(kind):
    if kind == "periodic":   # images one period away on both sides, a span shorter than the attraction's reach
        sp = slit_pore_1d(H=2.0, dx=0.02, cut_fac=0.99, seed=3)
        sp.bc, sp.nwall, sp.vext, sp.zero_tf = [[PERIODIC, PERIODIC]], 0, None, None
        sp.rho0 = np.maximum(sp.rho0, 0.05)
        return sp
    if kind in ("reflect", "reflect_bulk", "reflect_hs"):   # the last: no attraction, the FMT halo twice the density halo
        sp = hard_wall_1d(seed=4, size=3.15 if kind != "reflect_bulk" else 9.6, dx=0.05, rho_b=0.5)
        sp.bc = [[REFLECT, REFLECT]] if kind == "reflect" else [[IN_BULK, REFLECT]]
        sp.nwall, sp.vext, sp.zero_tf = 0, None, None
        sp.rho0 = np.maximum(sp.rho0, 0.3)
        if kind != "reflect_hs":
            sp.type_attr, sp.eps_ff, sp.cut_ff = 0, np.full((1, 1), 0.8), np.full((1, 1), 2.5)
        return sp
    if kind == "three":   # three components, White Bear
        sp = slit_pore_1d(H=7.3, dx=0.05, sig=(1.0, 0.9, 0.7), rho_b=(0.1, 0.1, 0.1), seed=5)
        sp.type_func = FMT3
        return sp
    if kind == "long2":
        return hard_wall_1d(seed=6, size=0.05 * 20000, dx=0.05, rho_b=0.6)
    if kind == "long_rows":   # the rows alone go to the row kernels
        return hard_wall_1d(seed=6, size=0.05 * 140000, dx=0.05, rho_b=0.4)
    if kind == "long4":
        return slit_pore_1d(H=0.05 * 40001, dx=0.05, seed=7)
    return small_case(kind)


def _problems(make, monkeypatch):
    monkeypatch.setenv("TMI_AUTOTUNE", "0")
    monkeypatch.setenv("TMI_LINE1D", "0")
    a = make()
    monkeypatch.setenv("TMI_LINE1D", "1")
    b = make()
    assert a.row_form()[0] == 0 and b.row_form()[0] == 1   # the forms compared are two forms
    return a, b


def _compare(a, b, blocks, tol):
    for lo, hi in blocks:
        if lo < hi:
            scale = float(a[lo:hi].abs().max())
            assert float((a[lo:hi] - b[lo:hi]).abs().max()) <= tol * scale, (lo, hi)


KINDS = ["1d_hw", "1d_reflect_wca", "1d_pore_mix", "1d_reflect_slab", "periodic", "reflect", "reflect_bulk", "reflect_hs",
         "three", "long2", "long4", "long_rows", "batch_small", "batch_large"]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_line_matches_row_kernels(kind, monkeypatch):
    batch = kind.startswith("batch")
    if batch:
        spec = slit_pore_batch(npores=3 if kind == "batch_small" else 60, seed=2)
        rows, line = _problems(lambda: DeviceBatch(spec), monkeypatch)
    else:
        spec = _single(kind)
        rows, line = _problems(lambda: DeviceProblem(spec), monkeypatch)
    C = spec.ncomp
    R = 6
    x = rows.initial_state()
    blocks = ((0, C), (C, C + R), (C + R, x.shape[0]))
    _compare(x, line.initial_state(), blocks, 1e-12)
    g = torch.Generator(device="cuda").manual_seed(1)
    noise = lambda: 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1   # noqa: E731
    x[C:] *= 1.0 + 0.01 * noise()[C:]
    Fa, sa = rows.fill_residual(x)
    Fb, sb = line.fill_residual(x)
    _compare(Fa, Fb, blocks, 1e-12)
    assert abs(sa - sb) <= 1e-12 * abs(sa)
    dev = torch.zeros(1, dtype=torch.float64, device="cuda")
    line.fill_residual_device_norm(x, Fb, dev)
    _compare(Fa, Fb, blocks, 1e-12)
    assert abs(float(dev) - sa) <= 1e-12 * abs(sa)
    v = noise()
    _compare(rows.apply_jacobian(x, v), line.apply_jacobian(x, v), blocks, 1e-12)
    _compare(rows.apply_jacobian(x, v, fp32=True), line.apply_jacobian(x, v, fp32=True), blocks, 1e-5)
    ms = line.fill_residual_timed(x, reps=2)   # the stage of the launch that a fill runs
    assert ms[0] > 0 and not ms[1:].any() and (rows.fill_residual_timed(x, reps=2)[[0, 1, 3, 4]] > 0).all()
    # Schur product, right-hand side and back-substitution: one Newton update
    da, _ = rows.schur_solve(x, Fa, rtol=1e-12)
    db, _ = line.schur_solve(x, Fa, rtol=1e-12)
    _compare(da, db, blocks, 1e-8)
    dm, _ = line.schur_solve(x, Fa, rtol=1e-8, restart=500, maxit=2500, precision=PREC_MIXED)
    check_update(rows, x, Fa, dm, C, row_scale(rows, x, C, g), mixed=True)
    assert line.row_form()[1] == {"long2": 2, "long4": 4, "long_rows": 4, "batch_large": 4}.get(kind, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("npores", [5, 80])   # one and four positions per lane
def test_batched_step_solves_each_pore(npores, mixed, monkeypatch):
    """Batched Schur products: the direction scaled on the way in, workgroups of finished pores skipped."""
    spec = slit_pore_batch(npores=npores, seed=5)
    rows, line = _problems(lambda: DeviceBatch(spec), monkeypatch)
    check_batch_step(line, rows, mixed, torch.Generator(device="cuda").manual_seed(2))


@pytest.mark.gpu
@pytest.mark.parametrize("nodes", [201, 20000, 40000])   # one, two and four positions per lane
def test_pair_without_attraction(nodes, monkeypatch):
    """A binary fluid whose unlike pair has eps = 0: its attraction stencil has no point at all.  The
    residual of both forms against the oracle, products and the first Krylov steps against each other."""
    from oracle.oracle import Oracle
    spec = slit_pore_1d(H=0.02 * (nodes - 1), dx=0.02, seed=8)
    spec.eps_ff = np.array([[1.0, 0.0], [0.0, 0.9]])
    rows, line = _problems(lambda: DeviceProblem(spec), monkeypatch)
    assert line.info.sten_len[2][1] == 0 and line.info.sten_len[2][0] > 0
    o = Oracle.from_spec(spec)
    x = o.init_fields(spec.initial_x())
    rng = np.random.default_rng(3)
    x[2:] *= 1.0 + 0.01 * rng.uniform(-1, 1, x[2:].shape)
    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    v = torch.from_numpy(rng.uniform(-1, 1, x.shape)).cuda()
    blocks = ((0, 2), (2, 8), (8, 10))
    Fo = torch.from_numpy(np.asarray(o.residual(x))).reshape(x.shape).cuda()
    Fa, Fb = rows.fill_residual(xd)[0], line.fill_residual(xd)[0]
    _compare(Fo, Fa, blocks, 1e-12)
    _compare(Fo, Fb, blocks, 1e-12)
    _compare(rows.apply_jacobian(xd, v), line.apply_jacobian(xd, v), blocks, 1e-12)
    _compare(rows.apply_jacobian(xd, v, fp32=True), line.apply_jacobian(xd, v, fp32=True), blocks, 1e-5)
    da, _ = rows.schur_solve(xd, Fo, rtol=1e-30, restart=4, maxit=4)
    db, _ = line.schur_solve(xd, Fo, rtol=1e-30, restart=4, maxit=4)
    _compare(da, db, blocks, 1e-8)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nodes", [2600, 4096, 4097, 8192])   # one workgroup's sweep ends at step 76, 48, 17, 8
def test_long_krylov_cycles(nodes, precision, monkeypatch):
    """Cycles that go on past the basis one workgroup sweeps, restarted ones and ones cut by the iteration limit
    among them: the same steps as the general GMRES (TMI_LINE1D=0).  rtol 1e-9 bounds the distance of two
    updates by the condition of a dense fluid's Schur system, below 1e3; in mixed precision the FP32 product
    carries 1e-6 of the update, and the general solver's basis is FP32 too."""
    from tramonto_amd.device import PREC_FP64
    spec = hard_wall_1d(seed=2, size=0.05 * (nodes - 1), dx=0.05, rho_b=0.8)
    rows, line = _problems(lambda: DeviceProblem(spec), monkeypatch)
    x = rows.initial_state()
    F, _ = rows.fill_residual(x)
    prec, tol = (PREC_FP64, 1e-6) if precision == "fp64" else (PREC_MIXED, 1e-3)
    for restart, maxit in ((200, 400), (30, 400), (200, 55)):
        da, ia = rows.schur_solve(x, F, rtol=1e-9, restart=restart, maxit=maxit, precision=prec)
        db, ib = line.schur_solve(x, F, rtol=1e-9, restart=restart, maxit=maxit, precision=prec)
        assert 50 < ib <= maxit
        if precision == "fp64":
            assert abs(ia - ib) <= 1
        if ia < maxit and ib < maxit:
            assert float((da - db).abs().max()) <= tol * float(da.abs().max())
        elif precision == "fp64":   # cut after the same number of steps
            assert ia == ib and float((da - db).abs().max()) <= tol * float(da.abs().max())
