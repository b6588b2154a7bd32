"""Batched uneven 1D pores on the device against the oracle, pore by pore
(run on an MI355X).

Every pore of a batch is the problem the oracle (and the reference) solves on
its own; the batch must reproduce each pore's residual and Jacobian products
to 1e-12 and each pore's converged profile to 1e-8, with and without graph
replay, and in mixed precision.
"""
import os

import numpy as np
import pytest
import scipy.sparse as sps

torch = pytest.importorskip("torch")

from oracle.oracle import Oracle  # noqa: E402
from tramonto_amd.batch import slit_pore_batch  # noqa: E402

RTOL = 1e-12


@pytest.fixture(scope="module")
def small():
    from tramonto_amd.batch import DeviceBatch
    b = slit_pore_batch(npores=5, seed=3, h_range=(3.0, 5.0))
    oracles = [Oracle.from_spec(p) for p in b.pores]
    return b, oracles, DeviceBatch(b)


@pytest.fixture(scope="module")
def small_rows(small):
    """the same batch through the separate row kernels"""
    from tramonto_amd.batch import DeviceBatch
    b, oracles, _ = small
    old = os.environ.get("TMI_LINE1D")
    os.environ["TMI_LINE1D"] = "0"
    try:
        return b, oracles, DeviceBatch(b)
    finally:
        os.environ.pop("TMI_LINE1D") if old is None else os.environ.update(TMI_LINE1D=old)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def generic_state(b, oracles, seed):
    xs = [o.init_fields(p.initial_x()) for p, o in zip(b.pores, oracles)]
    x = np.concatenate(xs, axis=1)
    rng = np.random.default_rng(seed)
    x[b.ncomp:] *= 1.0 + 0.01 * rng.uniform(-1.0, 1.0, x[b.ncomp:].shape)
    return x


@pytest.mark.gpu
def test_batch_init_fields_per_pore(small):
    b, oracles, db = small
    xg = db.init_fields(dev(b.initial_x())).cpu().numpy()
    for xp, p, o in zip(b.split(xg), b.pores, oracles):
        xo = o.init_fields(p.initial_x())
        assert np.abs(xp - xo).max() < RTOL * np.abs(xo).max()


@pytest.mark.gpu
def test_batch_residual_per_pore(small):
    b, oracles, db = small
    x = generic_state(b, oracles, 21)
    Fg, _ = db.fill_residual(dev(x))
    for Fp, xp, o in zip(b.split(Fg.cpu().numpy()), b.split(x), oracles):
        Fo = o.residual(np.ascontiguousarray(xp))
        assert np.abs(Fp - Fo).max() < RTOL * np.abs(Fo).max()


@pytest.mark.gpu
def test_batch_jvp_per_pore(small):
    b, oracles, db = small
    x = generic_state(b, oracles, 22)
    rng = np.random.default_rng(4)
    v = rng.uniform(-1.0, 1.0, x.shape)
    Jv = db.apply_jacobian(dev(x), dev(v)).cpu().numpy()
    for p, o, xp, vp, Jp in zip(b.pores, oracles, b.split(x), b.split(v), b.split(Jv)):
        r, c, val = o.jacobian_coo(np.ascontiguousarray(xp))
        n = p.nunk * p.nnodes
        J = sps.coo_matrix((val, (r, c)), shape=(n, n)).tocsr()
        ref = (J @ np.ascontiguousarray(vp).reshape(-1)).reshape(p.nunk, p.nnodes)
        assert np.abs(Jp - ref).max() < RTOL * np.abs(ref).max()


@pytest.mark.gpu
def test_batch_transpose_is_unsupported(small):
    b, oracles, db = small
    x = db.initial_state()
    with pytest.raises(RuntimeError, match="not implemented"):
        db.apply_jacobian_transpose(x, x)


@pytest.fixture(scope="module")
def oracle_profiles(small):
    b, oracles, _ = small
    out = []
    for p, o in zip(b.pores, oracles):
        xo, st = o.newton(o.init_fields(p.initial_x()), resid_tol=1e-10)
        assert st["converged"], st
        out.append(xo)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("graph", ["1", "0"])
def test_batch_newton_matches_oracle(graph, small, oracle_profiles, monkeypatch):
    b, oracles, db = small
    monkeypatch.setenv("TMI_BATCH_GRAPH", graph)
    x = db.initial_state()
    st = db.newton(x, resid_tol=1e-10, gmres_tol=1e-9, max_iter=60)
    assert st["converged"], st
    assert st["pore_converged"].all() and (st["pore_resid"] < 1e-10).all()
    assert (st["pore_iters"] > 0).all() and (st["pore_gmres"] > 0).all()
    for xp, xo, p in zip(b.split(x.cpu().numpy()), oracle_profiles, b.pores):
        assert np.abs(xp[: p.ncomp] - xo[: p.ncomp]).max() < 1e-8


@pytest.mark.gpu
def test_batch_newton_mixed_precision(small, oracle_profiles):
    from tramonto_amd.device import PREC_MIXED
    b, oracles, db = small
    x = db.initial_state()
    st = db.newton(x, resid_tol=1e-10, gmres_tol=1e-7, max_iter=60, precision=PREC_MIXED)
    assert st["converged"], st
    for xp, xo, p in zip(b.split(x.cpu().numpy()), oracle_profiles, b.pores):
        assert np.abs(xp[: p.ncomp] - xo[: p.ncomp]).max() < 1e-8


@pytest.mark.gpu
def test_batch_newton_matches_single_pore_solves(small):
    """The batch and one device problem per pore converge to the same profiles."""
    from tramonto_amd.device import DeviceProblem
    b, oracles, db = small
    x = db.initial_state()
    assert db.newton(x, resid_tol=1e-11, gmres_tol=1e-10, max_iter=60)["converged"]
    for xp, p in zip(b.split(x.cpu().numpy()), b.pores):
        dp = DeviceProblem(p)
        xs = dp.initial_state()
        assert dp.newton(xs, resid_tol=1e-11, gmres_tol=1e-10, max_iter=60)["converged"]
        assert np.abs(xp - xs.cpu().numpy()).max() < 1e-9 * max(1.0, np.abs(xp).max())


@pytest.mark.gpu
@pytest.mark.parametrize("per_lane", [4, 8, 16])
@pytest.mark.parametrize("lanes", [64, 128, 256])
def test_every_row_kernel_shape_matches_oracle(small_rows, per_lane, lanes):
    """Every launch shape the 1D autotuner can choose (outputs per lane x lanes per workgroup, for the
    rho-bar, mean-field and Euler-Lagrange row kernels, FP64 and FP32), forced with
    tmi_row_tuning_set: residual and J v per pore against the oracle to 1e-12, the FP32 product
    against FP64 to 1e-5."""
    b, oracles, db = small_rows
    assert db.row_form()[0] == 0   # the row kernels, not all rows in one launch
    db.set_row_tuning(per_lane, lanes)
    tun = db.row_tuning()
    assert all(tun[p][k][:2] == (per_lane, lanes) for p in tun for k in tun[p] if tun[p][k][0])
    try:
        x = generic_state(b, oracles, 30 + per_lane + lanes)
        Fg, _ = db.fill_residual(dev(x))
        for Fp, xp, o in zip(b.split(Fg.cpu().numpy()), b.split(x), oracles):
            Fo = o.residual(np.ascontiguousarray(xp))
            assert np.abs(Fp - Fo).max() < RTOL * np.abs(Fo).max()
        rng = np.random.default_rng(per_lane * lanes)
        v = rng.uniform(-1.0, 1.0, x.shape)
        Jv = db.apply_jacobian(dev(x), dev(v)).cpu().numpy()
        for p, o, xp, vp, Jp in zip(b.pores, oracles, b.split(x), b.split(v), b.split(Jv)):
            r, c, val = o.jacobian_coo(np.ascontiguousarray(xp))
            n = p.nunk * p.nnodes
            J = sps.coo_matrix((val, (r, c)), shape=(n, n)).tocsr()
            ref = (J @ np.ascontiguousarray(vp).reshape(-1)).reshape(p.nunk, p.nnodes)
            assert np.abs(Jp - ref).max() < RTOL * np.abs(ref).max()
        J32 = db.apply_jacobian(dev(x), dev(v), fp32=True).cpu().numpy()
        assert np.abs(J32 - Jv).max() < 1e-5 * np.abs(Jv).max()
    finally:
        db.set_row_tuning(8, 256)


# ---------------------------------------------------------------- 2D pieces
@pytest.fixture(scope="module")
def small2d():
    """four rough slit pores of 64 columns (periodic x, walls at both y ends) and uneven heights"""
    from tramonto_amd.batch import DeviceBatch, rough_slit_pore_batch_2d
    b = rough_slit_pore_batch_2d(npores=4, seed=5, nx=64, h_range=(3.0, 5.0), dx=0.1)
    oracles = [Oracle.from_spec(p) for p in b.pores]
    return b, oracles, DeviceBatch(b)


@pytest.mark.gpu
def test_batch_2d_residual_and_jvp_per_piece(small2d):
    """2D pieces stacked along y between wall rows: each piece's residual and Jacobian product equal
    the oracle's for that piece on its own (1e-12), at a perturbed state."""
    b, oracles, db = small2d
    assert db.info.fmt_fft == 0 and db.info.mf_fft == 0   # batches of 2D pieces keep the direct sums
    x = generic_state(b, oracles, 31)
    Fg, _ = db.fill_residual(dev(x))
    for Fp, xp, o in zip(b.split(Fg.cpu().numpy()), b.split(x), oracles):
        Fo = o.residual(np.ascontiguousarray(xp))
        assert np.abs(Fp - Fo).max() < RTOL * np.abs(Fo).max()
    rng = np.random.default_rng(6)
    v = rng.uniform(-1.0, 1.0, x.shape)
    Jv = db.apply_jacobian(dev(x), dev(v)).cpu().numpy()
    for p, o, xp, vp, Jp in zip(b.pores, oracles, b.split(x), b.split(v), b.split(Jv)):
        r, c, val = o.jacobian_coo(np.ascontiguousarray(xp))
        n = p.nunk * p.nnodes
        J = sps.coo_matrix((val, (r, c)), shape=(n, n)).tocsr()
        ref = (J @ np.ascontiguousarray(vp).reshape(-1)).reshape(p.nunk, p.nnodes)
        assert np.abs(Jp - ref).max() < RTOL * np.abs(ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("graph", ["1", "0"])
def test_batch_2d_newton_matches_single_solves(graph, small2d, monkeypatch):
    """The batched per-piece Newton-Krylov on 2D pieces: every piece converges, to the profile of
    the piece solved as one device problem (1e-8; that path's Newton profiles are pinned to the
    oracle's by the parity suite; the first piece is also checked against the oracle here)."""
    from tramonto_amd.device import DeviceProblem
    b, oracles, db = small2d
    monkeypatch.setenv("TMI_BATCH_GRAPH", graph)
    x = db.initial_state()
    st = db.newton(x, resid_tol=1e-10, gmres_tol=1e-9, gmres_restart=100, gmres_max_iter=2000, max_iter=60)
    print("2D batch:", st["pore_iters"], st["pore_gmres"], st["pore_resid"], flush=True)
    assert st["converged"], st
    assert st["pore_converged"].all() and (st["pore_resid"] < 1e-10).all()
    for k, (xp, p, o) in enumerate(zip(b.split(x.cpu().numpy()), b.pores, oracles)):
        if k == 0:
            xo, sto = o.newton(o.init_fields(p.initial_x()), resid_tol=1e-10)
            assert sto["converged"], sto
            assert np.abs(xp[: p.ncomp] - xo[: p.ncomp]).max() < 1e-8
        dp = DeviceProblem(p)
        xs = dp.initial_state()
        assert dp.newton(xs, resid_tol=1e-11, gmres_tol=1e-10, gmres_restart=100, gmres_max_iter=2000,
                         max_iter=60)["converged"]
        assert np.abs(xp[: p.ncomp] - xs.cpu().numpy()[: p.ncomp]).max() < 1e-8


@pytest.mark.gpu
def test_batch_newton_ignores_unwritten_basis_vectors():
    """The Krylov basis is allocated uninitialised: vectors past a cycle's steps must not enter the
    solution, whatever their memory held before (here NaN, left by freed tensors)."""
    from tramonto_amd.batch import DeviceBatch
    b = slit_pore_batch(npores=3, seed=3, h_range=(3.0, 4.0))
    junk = [torch.full((4 << 20,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(24)]
    torch.cuda.synchronize()
    del junk
    torch.cuda.empty_cache()
    db = DeviceBatch(b)
    x = db.initial_state()
    st = db.newton(x, resid_tol=1e-10, gmres_tol=1e-9, max_iter=60)
    assert st["converged"], st


@pytest.mark.gpu
@pytest.mark.parametrize("nodes,graph", [((1, 2, 3, 40, 900), "1"), ((2049, 2600, 150), "0"), ((4500, 300), "1"),
                                         ((9000, 500, 120), "1")])
def test_batch_newton_segment_lengths(nodes, graph, monkeypatch):
    """One-launch Arnoldi steps over every workgroup shape, and pores too long for one (two components:
    4096, 8192 and 16384 unknowns are the edges): batch and pore-by-pore profiles agree to the
    tolerance of the solves, pores of a few nodes and pores that finish early included."""
    from tramonto_amd.batch import BatchSpec, DeviceBatch
    from tramonto_amd.device import DeviceProblem
    from tramonto_amd.problem import slit_pore_1d
    monkeypatch.setenv("TMI_BATCH_GRAPH", graph)
    pores = [slit_pore_1d(H=0.02 * max(n - 1, 1) if n > 1 else 0.0, dx=0.02, rho_b=(0.1, 0.1), eps_ff=0.5, seed=i)
             for i, n in enumerate(nodes)]
    db = DeviceBatch(BatchSpec(pores))
    for restart in (60, 7):
        x = db.initial_state()
        st = db.newton(x, resid_tol=1e-10, gmres_tol=1e-9, max_iter=60, gmres_restart=restart)
        assert st["converged"], st
    o = db.batch.offsets
    for i, p in enumerate(pores):
        dp = DeviceProblem(p)
        xs = dp.initial_state()
        assert dp.newton(xs, resid_tol=1e-10, gmres_tol=1e-9, max_iter=60, gmres_restart=7)["converged"]
        assert float((xs - x[:, o[i]:o[i + 1]]).abs().max()) < 1e-8


@pytest.mark.gpu
@pytest.mark.parametrize("ndim", [1, 2])
def test_batch_graphs_follow_the_jacobian_mode(ndim, monkeypatch):
    """set_jacobian between two batched solves on one handle: the replayed graphs run the mode in force, as
    direct launches do.  FMT4's reference Jacobian is inexact, so two steps of either mode differ."""
    from tramonto_amd.batch import BatchSpec, DeviceBatch
    from tramonto_amd.device import JAC_EXACT, JAC_REFERENCE
    from tramonto_amd.problem import rough_slit_pore_2d, slit_pore_1d
    pores = [slit_pore_1d(H=3.0, dx=0.05, rho_b=(0.25, 0.25), eps_ff=0.5, seed=i) if ndim == 1 else
             rough_slit_pore_2d(seed=i, nx=53, ny=33, eps_ff=0.5) for i in range(2)]
    for p in pores:
        p.type_func = 3
    db = DeviceBatch(BatchSpec(pores))
    x0 = db.initial_state()

    def two_steps(graph):
        monkeypatch.setenv("TMI_BATCH_GRAPH", graph)
        x = x0.clone()
        db.newton(x, max_iter=2, resid_tol=1e-30, gmres_tol=1e-10)
        return x

    exact = two_steps("1")
    for mode in (JAC_REFERENCE, JAC_EXACT):
        db.set_jacobian(mode)
        graph, direct = two_steps("1"), two_steps("0")
        assert float((graph - direct).abs().max()) < 1e-10
        moved = float((graph - exact).abs().max())
        assert moved > 1e-6 if mode == JAC_REFERENCE else moved < 1e-10
