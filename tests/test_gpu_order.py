"""The per-function deposit and gather on particles in box order and in random
order: arrays in order are read through the box list, scattered ones by
records, and both must give the oracle's fields and right-hand sides (bar: the
repository's 1e-12 of each component's range, the rounding of sums over at most
a few thousand particles).  Particle counts around the wave of 64 and the
workgroup of 256; a call of more particles than one batch holds."""
import numpy as np
import pytest

import cases
from test_gpu_parity import random_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from emu_amd import core as c
    return c


@pytest.mark.parametrize("n", [1, 63, 65, 256, 1025, 3000])
@pytest.mark.parametrize("nf", [2, 3])
@pytest.mark.parametrize("ncell", [(3, 4, 5), (1, 1, 9), (1, 5, 4)])
def test_scattered_and_ordered_particles(core, oracle, nf, ncell, n):
    L = tuple(0.5 * k for k in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L)
    prm = cases.oracle_deck(oracle, d).params()
    emu = core.Emu(cases.product_params(d))
    parts, _ = random_case(oracle, nf, ncell, L, n, seed=10 * n + nf)
    grid = oracle.Grid(nf, prm)
    oracle.deposit_to_mesh(nf, prm, parts, grid)
    want_dep = grid.fab().reshape(emu.ncomp, -1).T.copy()
    oracle.fill_boundary(nf, prm, grid)
    want_rhs = parts.copy()
    oracle.interpolate_rhs_from_mesh(nf, prm, want_rhs, grid)
    cell = np.floor(parts["pos"] / 0.5).astype(int)
    in_order = np.lexsort((cell[:, 0], cell[:, 1], cell[:, 2]))
    for order in (np.arange(n), in_order):
        c = core.FlavoredNeutrinoContainer.from_aos(emu, parts[order])
        state = core.MultiFab(emu)
        core.deposit_to_mesh(c, state)
        got = state.data.cpu().numpy().reshape(emu.ncomp, -1).T
        assert cases.max_rel_err(got[:, 3:], want_dep[:, 3:]) < 1e-12
        state.FillBoundary()
        core.interpolate_rhs_from_mesh(c, state)
        got, want = c.to_aos()["rdata"], want_rhs["rdata"][order]
        if n == 1:
            # a lone particle's potential is made of its own states, with which it
            # nearly commutes: its right-hand side is set against the products
            # that cancel, coef (N + Nbar) |f|^2, and the other rows as they are
            K = emu.K
            a = parts["rdata"][0]
            f = np.r_[K["f00_Re"]:K["f00_Re"] + emu.nh, K["f00_Rebar"]:K["f00_Rebar"] + emu.nh]
            coef = 2 ** 0.5 * oracle.GF / 0.5 ** sum(k > 1 for k in ncell) / oracle.hbar
            scale = coef * (a[K["N"]] + a[K["Nbar"]]) * np.abs(a[f]).max() ** 2
            assert np.abs(got[0, f] - want[0, f]).max() < 1e-12 * scale
            got, want = np.delete(got, f, axis=1), np.delete(want, f, axis=1)
        assert cases.max_rel_err(got, want) < 1e-12
        emu.sync()


def test_more_particles_than_a_batch(core):
    """2^25 particles are one batch of the box list; the few past them are a
    second one.  The deposit still sums all of them (partition of unity: the
    cells' N00 add up to the particles'), and the last particles' right-hand
    sides are those of a call on them alone."""
    import torch
    n, tail = (1 << 25) + 77, 100
    emu = core.Emu(cases.product_params(cases.fast_flavor_dict(nf=2, ncell=(8, 8, 8), L=(4.0, 4.0, 4.0))))
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    c = core.FlavoredNeutrinoContainer(emu, n)
    K = emu.K
    c.pos.uniform_(0.0, 4.0, generator=g)
    c.rdata[K["pupz"]:K["pupt"] + 1] = 8e-5
    c.rdata[K["N"]].uniform_(1.0, 2.0, generator=g)
    c.rdata[K["Nbar"]].uniform_(1.0, 2.0, generator=g)
    for k in ("f00_Re", "f00_Rebar"):
        c.rdata[K[k]] = 1.0
        c.rdata[K[k] + 1].uniform_(-0.1, 0.1, generator=g)
    state = core.MultiFab(emu)
    core.deposit_to_mesh(c, state)
    # 2^25 terms summed in two orders: eps sqrt(n) with a margin
    assert float(state.valid()[3].sum()) == pytest.approx(float(c.rdata[K["N"]].sum()), rel=1e-11)
    state.FillBoundary()
    few = core.FlavoredNeutrinoContainer(emu, tail)
    few.pos.copy_(c.pos[:, n - tail:])
    few.rdata.copy_(c.rdata[:, n - tail:])
    core.interpolate_rhs_from_mesh(c, state)
    core.interpolate_rhs_from_mesh(few, state)
    torch.testing.assert_close(c.rdata[:, n - tail:], few.rdata, rtol=1e-12, atol=0.0)
