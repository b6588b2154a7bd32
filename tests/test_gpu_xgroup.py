"""The fused x pass over groups of mirror lines against its LDS form.

Cases: every register length (32, 64, 128, 256), 2D and 3D, even and odd other axes (groups with
self-mirror lines and a last workgroup that is not full), one to four components (one or several fills of
the spectrum slots, one or several outputs per wave, products that mix even and odd tables).

Tolerance: both forms are FP64 sums of the same terms through transforms of the same length; each carries
round-off of a few eps times the largest row of its block (1e-12, the FFT forms' parity bound), in FP32 of
a few eps32 per transform stage (1e-5).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from tramonto_amd.problem import FMT1, PERIODIC, ProblemSpec, SplitMix64, lorentz_berthelot  # noqa: E402

RTOL, RTOL32 = 1e-12, 1e-5


def _fluid(n, ncomp):
    sig = [1.0, 0.8, 0.9, 0.7][:ncomp]
    rho = [0.3, 0.15, 0.1, 0.1][:ncomp]
    S, E, R = lorentz_berthelot(sig, [0.7] * ncomp, [1.3 * s for s in sig])
    rng = SplitMix64(3)
    N = int(np.prod(n))
    rho0 = np.stack([r * (1.0 + 0.2 * rng.uniform(N, -1.0, 1.0)) for r in rho])
    return ProblemSpec(name="xgroup", ndim=len(n), ncomp=ncomp, nx=list(n), dx=[0.25] * len(n), bc=[[PERIODIC, PERIODIC]] * len(n),
                       type_func=FMT1, type_attr=0, nwall=0, hs_diam=sig, sigma_ff=S, eps_ff=E, cut_ff=R, rho_b=rho,
                       rho0=rho0)


@pytest.mark.gpu
@pytest.mark.parametrize("n,ncomp", [((32, 15, 16), 1), ((64, 16, 15), 2), ((128, 16, 15), 3), ((128, 15, 18), 4),
                                     ((256, 16, 15), 1), ((256, 15, 15), 3), ((32, 27), 2), ((64, 16), 1), ((128, 25), 3),
                                     ((256, 18), 1), ((64, 64, 64), 4),
                                     ((128, 32, 32), 3), ((128, 46, 46), 3)])   # three and two slots for five input pairs
def test_mirror_line_groups_match_lds_form(n, ncomp, monkeypatch):
    from tramonto_amd.device import DeviceProblem
    spec = _fluid(n, ncomp)
    monkeypatch.setenv("TMI_FMT_FFT", "1")
    monkeypatch.setenv("TMI_MF_FFT", "1")
    reg = DeviceProblem(spec)
    monkeypatch.setenv("TMI_FFT_XREG", "0")
    lds = DeviceProblem(spec)
    assert reg.info.fmt_fft == 2 and lds.info.fmt_fft == 2 and reg.info.fft_fold == 1
    # the forms compared are two forms (a product of many pairs on few lines of 128 or 256 keeps the LDS form)
    assert reg.info.fft_xreg == 3 if max(n[1:]) >= 32 else reg.info.fft_xreg & 1
    assert lds.info.fft_xreg == 0
    x = reg.initial_state()
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda: 2 * torch.rand(x.shape, generator=g, device="cuda", dtype=torch.float64) - 1  # noqa: E731
    x[ncomp:] *= 1.0 + 0.01 * rnd()[ncomp:]
    v = rnd()
    pairs = [(reg.fill_residual(x)[0], lds.fill_residual(x)[0], RTOL),
             (reg.apply_jacobian(x, v), lds.apply_jacobian(x, v), RTOL),
             (reg.apply_jacobian(x, v, fp32=True), lds.apply_jacobian(x, v, fp32=True), RTOL32),
             (reg.apply_jacobian_transpose(x, v), lds.apply_jacobian_transpose(x, v), RTOL)]
    C, R = ncomp, spec.nrb
    for i, (a, b, tol) in enumerate(pairs):
        assert bool(torch.isfinite(a).all())
        for lo, hi in ((0, C), (C, C + R), (C + R, a.shape[0])):
            err = float((a[lo:hi] - b[lo:hi]).abs().max()) / max(float(b[lo:hi].abs().max()), 1.0)
            assert err < tol, (i, lo, err)
