"""The step in eight phases (pypde_rbc_phase) against the step with one launch per
operator (which the golden steps pin against the reference), at the sizes where
tiles, chunks and chains end: lengths around multiples of 16 and 32 modes of a
parity, odd lengths (an odd dealiased grid has a middle point that is its own
mirror), the longest lines a phase takes, one instance and enough of them for the
larger tiles, both integrators.

Tolerance: both forms are exact FP64 evaluations of the same step; the Helmholtz and
Poisson operators amplify rounding by up to about N^2, so 1e-12 + 4 N^2 eps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(shape, B, case, integrator, beta):
    import torch
    from pypde_amd.engine import RBCBatch
    params = [dict(ra=1e5 * (1 + b % 5), pr=1.0 + 0.1 * (b % 3), dt=2e-3) for b in range(B)]
    rng = np.random.default_rng(shape[0] * 1000 + shape[1])
    out = []
    for group in (True, False):
        e = RBCBatch(shape, params, case=case, integrator=integrator, beta=beta, group_launches=group)
        assert e.staged == group and (len(e.launches) == 8 * e.nstage) == group
        # neither form sets up the other's operators
        assert hasattr(e, "stage_ops") == group
        assert not group or not (e.fold_x or e.fold_y or e.fold_bf or hasattr(e, "WQy"))
        if group:
            k0, k1 = np.arange(e.N0), np.arange(e.N1)
            fall = np.exp(-8.0 * k0 / e.N0)[:, None] * np.exp(-8.0 * k1 / e.N1)
            X = 0.05 * rng.standard_normal(tuple(e.X.shape)) * fall[:e.M0, :e.M1]
            pres = 0.01 * rng.standard_normal(tuple(e.pres.shape)) * fall
        e.X.copy_(torch.as_tensor(X))
        e.pres.copy_(torch.as_tensor(pres))
        e.ws.fill_(float("nan"))   # nothing is read before the step wrote it
        for _ in range(2):
            e.step_eager()
        out.append([t.cpu().numpy().copy() for t in (e.X[:, 0], e.X[:, 1], e.X[:, 2], e.pres)])
    tol = 1e-12 + 4.0 * max(shape) ** 2 * np.finfo(float).eps
    for name, a, b in zip(("U", "V", "T", "pres"), *out):
        assert np.all(np.isfinite(a)), name
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        assert err < tol, (name, err, tol)


@pytest.mark.parametrize("shape,B", [((8, 8), 1), ((9, 11), 2), ((34, 35), 1), ((36, 66), 2), ((67, 33), 1),
                                     ((66, 98), 1), ((130, 21), 1), ((20, 131), 2), ((259, 18), 1),
                                     ((16, 258), 1), ((514, 12), 1), ((12, 513), 1), ((12, 460), 1),
                                     ((240, 224), 1), ((240, 240), 1), ((12, 260), 3),
                                     ((130, 131), 64)])
def test_phases_match_single_launches(shape, B):
    _run(shape, B, "rbc", "eu", 1.0)


@pytest.mark.parametrize("shape,case,integrator,beta", [((20, 36), "zero", "rk3", 1.0), ((36, 20), "linear", "rk3", 0.5),
                                                        ((68, 64), "linear", "eu", 0.5), ((35, 32), "rbc", "rk3", 1.0)])
def test_phases_match_other_schemes(shape, case, integrator, beta):
    _run(shape, 2, case, integrator, beta)

