"""At shape order 0 a particle sees and feeds its own cell alone.  A state that is not
finite in one cell stays there, through a step of the adjoint problem and through
its VJP: every other cell gets what it gets beside a finite one, to rounding."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("ncell", [(1, 1, 6), (3, 2, 4)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
def test_nonfinite_states_stay_in_their_cell(oracle, nf, prec, ncell, bad):
    """The cells share nothing, so only the order of a cell's own sum can differ:
    1e-12 of the largest entry in FP64; FP32 rounds the summed field and what
    follows from it to 1e-5."""
    import torch
    assert torch.cuda.is_available()
    from emu_amd import adjoint, core
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, nphi=6, st4_amplitude=1e-3, maxError=1e-2, shape_order=0)
    emu = core.Emu(cases.product_params(d))
    c = core.FlavoredNeutrinoContainer.from_aos(emu, oracle.init_particles(cases.oracle_deck(oracle, d)))
    p = adjoint.AdjointProblem(emu, c, dt=1e-12, nsteps=1, precision=prec)
    rng = np.random.default_rng(2)
    n = p.pos0.shape[1]
    at = rng.random((3, n)) * 0.5 * np.array(ncell)[:, None]
    pos = torch.from_numpy(at).to(p.pos0.device)
    cell = tuple(k // 2 for k in ncell)
    there = torch.from_numpy(np.all((at / 0.5).astype(int) == np.array(cell)[:, None], axis=0)).to(pos.device)
    assert 0 < int(there.sum()) < n
    y = p.f0.clone()
    y[:, there] = bad
    g = torch.Generator(device="cpu").manual_seed(5)
    lam = torch.randn(y.shape, generator=g, dtype=torch.float64).to(y)
    tol = 1e-12 if prec == "fp64" else 1e-5
    for f in (lambda s: p.step(pos.clone(), p.Nn_base, s), lambda s: p.step_adjoint(pos, p.Nn_base, s, lam)):
        want, got = f(p.f0)[:, ~there], f(y)[:, ~there]
        assert bool(torch.isfinite(got).all())
        assert float((got - want).abs().max()) <= tol * float(want.abs().max())
