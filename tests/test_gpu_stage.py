"""The step in eight phases (pypde_rbc_phase) against the step with one launch per
operator (which the golden steps pin against the reference), at the sizes where
tiles, chunks and chains end: lengths around multiples of 16 and 32 modes of a
parity, odd lengths (an odd dealiased grid has a middle point that is its own
mirror), the longest lines a phase takes, one instance and enough of them for the
larger tiles, both integrators.

Tolerance: both forms are exact FP64 evaluations of the same step; the Helmholtz and
Poisson operators amplify rounding by up to about N^2, so 1e-12 + 4 N^2 eps.  The
pressure correction P is what the pressure is updated by, pres += S P S^T / (dt a),
and small where the flow is nearly free of divergence, while its rounding is that of
the velocities and the pressure it corrects: its error is measured against dt a |pres|
where that is larger than |P|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(shape, B, case, integrator, beta, dealias=True, exact=False):
    import torch
    from pypde_amd.engine import RBCBatch
    params = [dict(ra=1e5 * (1 + b % 5), pr=1.0 + 0.1 * (b % 3), dt=2e-3) for b in range(B)]
    rng = np.random.default_rng(shape[0] * 1000 + shape[1])
    out = []
    for group in (True, False):
        e = RBCBatch(shape, params, case=case, integrator=integrator, beta=beta, dealias=dealias,
                     group_launches=group, exact_solves=exact)
        phases = group and not exact
        assert e.staged == phases and (len(e.launches) == 8 * e.nstage) == phases
        # neither form sets up the other's operators
        assert hasattr(e, "stage_ops") == phases
        assert not phases or not (e.fold_x or e.fold_y or e.fold_bf or hasattr(e, "WQy"))
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
        out.append([t.cpu().numpy().copy() for t in (e.X[:, 0], e.X[:, 1], e.X[:, 2], e.pres, e.P)])
    tol = 1e-12 + 4.0 * max(shape) ** 2 * np.finfo(float).eps
    for name, a, b in zip(("U", "V", "T", "pres", "P"), *out):
        assert np.all(np.isfinite(a)), name
        scale = np.linalg.norm(b)
        if name == "P":
            assert np.all(a[:, 0, 0] == 0.0)   # the gauge
            scale = max(scale, 2e-3 * float(e.ka[-1]) * np.linalg.norm(out[1][3]))
        err = np.linalg.norm(a - b) / scale
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


@pytest.mark.parametrize("shape,B", [
    ((66, 34), 100),    # two x tiles by one per wave; 32 columns of the shortest chains; 16 tiles of y products
    ((140, 20), 90),    # 32 columns of the 8-position chains
    ((12, 256), 50),    # 8 tiles of y products, 8-position chains
    ((12, 513), 12),    # the same, 16-position chains
    ((12, 513), 20),    # 16 tiles of them
    ((514, 512), 1),    # the right-hand side by itself, 16-position chains on both axes
])
def test_phases_larger_forms(shape, B):
    """The kernel forms that larger work takes, at the smallest sizes that reach them."""
    _run(shape, B, "rbc", "eu", 1.0)


@pytest.mark.parametrize("shape,B,integrator,beta,dealias", [
    ((68, 64), 60, "rk3", 0.5, True),    # the right-hand side by itself with explicit diffusion
    ((36, 50), 2, "eu", 1.0, False), ((33, 20), 1, "eu", 1.0, False)])
def test_phases_of_batches_and_without_dealiasing(shape, B, integrator, beta, dealias):
    _run(shape, B, "linear", integrator, beta, dealias)


@pytest.mark.parametrize("shape", [(516, 12), (12, 515)])
def test_more_modes_than_a_phase_holds(shape):
    """One mode past the limit on an axis: refused, as the register recurrences
    hold no more either, but with exact line solves the step runs with grouped
    launches, here against one launch per operator."""
    from pypde_amd._lib import PypdeError
    from pypde_amd.engine import RBCBatch
    with pytest.raises(PypdeError, match="512"):
        RBCBatch(shape, [dict(ra=1e5, pr=1.0, dt=2e-3)])
    _run(shape, 1, "rbc", "eu", 1.0, exact=True)
