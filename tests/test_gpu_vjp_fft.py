"""Transpose products as spectral products against the per-point reversed gathers.

Tolerance: both forms are FP64 sums of the same terms; the spectral one carries transform round-off of
a few eps times the largest row (the FFT residual parity bound, 1e-12 of the row block's largest value).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tramonto_amd.problem import periodic_3d, small_case  # noqa: E402

RTOL = 1e-12


def _spec(case):
    if case == "3d_odd_periodic":   # a periodic axis of prime length (padded transform, two images) beside wrapping ones
        return periodic_3d(seed=4, n=(13, 12, 16), dx=0.25, cut=1.2)
    sp = small_case(case)
    if case == "2d_rough_wall":   # rows replaced by V_ext = VEXT_MAX whose densities are not zero
        v = sp.vext.copy()
        v[5::97] = sp.vext_max
        sp.vext = v
    return sp


@pytest.mark.gpu
@pytest.mark.parametrize("env", [{}, {"TMI_FFT_XFUSE": "0"}, {"TMI_FFT_FOLD": "0", "TMI_FFT_XFUSE": "0"}])
@pytest.mark.parametrize("case", ["2d_periodic", "2d_wall_reflect", "2d_rough_wall", "3d_periodic_wb", "3d_mix_bulk",
                                  "3d_odd_periodic", "3d_solute3_small", "3d_x64", "3d_mix3_x128"])
def test_spectral_transpose_matches_gather(case, env, monkeypatch):
    from tramonto_amd.device import DeviceProblem
    spec = _spec(case)
    monkeypatch.setenv("TMI_PRECOND", "diag")
    monkeypatch.setenv("TMI_FMT_FFT", "0")
    monkeypatch.setenv("TMI_MF_FFT", "0")
    direct = DeviceProblem(spec)
    monkeypatch.setenv("TMI_FMT_FFT", "1")
    monkeypatch.setenv("TMI_MF_FFT", "1")
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    fft = DeviceProblem(spec)
    assert fft.info.fmt_fft > 0 and direct.info.fmt_fft == 0
    x = direct.initial_state()
    g = torch.Generator(device="cuda").manual_seed(5)
    x[spec.ncomp:] *= 1.0 + 0.01 * (2 * torch.rand(x[spec.ncomp:].shape, generator=g, device="cuda", dtype=torch.float64) - 1)
    C, R = spec.ncomp, spec.nrb
    for _ in range(2):
        w = 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1
        a, b = direct.apply_jacobian_transpose(x, w), fft.apply_jacobian_transpose(x, w)
        for lo, hi in ((0, C), (C, C + R), (C + R, a.shape[0])):
            if lo == hi:
                continue
            scale = float(a[lo:hi].abs().max())
            err = float((a[lo:hi] - b[lo:hi]).abs().max()) / scale
            assert err < RTOL, (lo, err)
    assert np.isfinite(float(b.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("n,dx,gathers", [(64, 0.1, False), (300, 0.25, True)])
def test_short_2d_stencils_keep_the_gathers(n, dx, gathers, monkeypatch):
    """2D hard spheres: the gathers where the rule expects them to be faster (then the very kernels of a problem
    without spectra, bit for bit), else the spectral products."""
    from tramonto_amd.device import DeviceProblem
    from tramonto_amd.problem import IN_BULK, IN_WALL, PERIODIC, ProblemSpec, SplitMix64
    rho = 0.4 * (1 + 0.2 * SplitMix64(3).uniform(n * n, -1, 1))
    spec = ProblemSpec(name="hs", ndim=2, ncomp=1, nx=[n, n], dx=[dx, dx], bc=[[IN_WALL, IN_BULK], [PERIODIC, PERIODIC]],
                       type_func=0, type_attr=-1, hs_diam=[1.0], sigma_ff=np.ones((1, 1)), eps_ff=np.ones((1, 1)),
                       cut_ff=np.ones((1, 1)), rho_b=[0.4], rho0=rho[None, :])
    chosen = DeviceProblem(spec)
    monkeypatch.setenv("TMI_FMT_FFT", "0")
    direct = DeviceProblem(spec)
    x = direct.initial_state()
    g = torch.Generator(device="cuda").manual_seed(5)
    w = 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1
    a, b = direct.apply_jacobian_transpose(x, w), chosen.apply_jacobian_transpose(x, w)
    for lo, hi in ((0, 1), (1, 9)):
        assert float((a[lo:hi] - b[lo:hi]).abs().max()) <= RTOL * float(a[lo:hi].abs().max())
    assert torch.equal(a, b) == gathers
