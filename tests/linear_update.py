"""Checks of Newton updates by the linear system they solve, J dx = -F, with an FP64 product of another form.

An update solved to a small GMRES tolerance leaves the error E of its Schur product, J dx + F = E dx on the
Euler-Lagrange rows: in FP64 round-off and the solve's tolerance (1e-8 of |F|); in mixed precision the FP32
sums, whose parity bound is 1e-5 of the largest row of J v for |v| <= 1, here doubled for the product's two
chained sums.  The other rows are formed in FP64 whatever the precision.
"""
import torch


def row_scale(product, x, C, gen):
    v = 2 * torch.rand(x.shape, generator=gen, device=x.device, dtype=torch.float64) - 1
    return float(product.apply_jacobian(x, v)[:C].abs().max())


def check_update(product, x, F, dx, C, scale, mixed, parts=None):
    """parts: node ranges that are solved on their own (pores of a batch)."""
    r = product.apply_jacobian(x, dx) + F
    for lo, hi in parts or [(0, x.shape[1])]:
        f, d, e = F[:, lo:hi], dx[:, lo:hi], r[:, lo:hi].abs()
        tol = 1e-8 * float(f.abs().max())
        el = tol + (2e-5 * scale * float(d.abs().max()) if mixed else 0.0)
        assert float(e[:C].max()) <= el, (lo, float(e[:C].max()), el)
        assert float(e[C:].max()) <= tol, (lo, float(e[C:].max()), tol)


def check_batch_step(batch, product, mixed, gen):
    """One undamped step of the batched Newton from a state near the solution, pore by pore (their GMRES
    finish at different steps): x1 - x0 solves each pore's system."""
    from tramonto_amd.device import PREC_FP64, PREC_MIXED
    C, o = batch.spec.ncomp, batch.batch.offsets
    x0 = batch.initial_state()
    assert batch.newton(x0, resid_tol=1e-6, max_iter=80)["converged"]
    x0[:C] *= 1 + 1e-3 * (2 * torch.rand(x0[:C].shape, generator=gen, device=x0.device, dtype=torch.float64) - 1)
    x1 = x0.clone()
    st = batch.newton(x1, max_iter=1, resid_tol=1e-30, gmres_tol=1e-8 if mixed else 1e-11,
                      precision=PREC_MIXED if mixed else PREC_FP64)
    assert len(set(st["pore_gmres"])) > 1
    F, _ = product.fill_residual(x0)
    check_update(product, x0, F, x1 - x0, C, row_scale(product, x0, C, gen), mixed, list(zip(o[:-1], o[1:])))
