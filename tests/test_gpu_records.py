"""The per-function deposit and gather on particles so scattered that they cross to box
order as records, for every stencil (1-D to 3-D, shape orders 0 to 2) and particle
counts around the wave of 64 and the workgroup of 256.  The same particles in box
order take the other form; both must give the oracle's fields and right-hand sides
(the repository's 1e-12 of each component's range)."""
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


def boxes_per_wave(cell):
    """What the box list measures, for up to 256 workgroups of 256 particles: one wave
    of each in turn, its first 8 boxes and then every particle of another."""
    total, waves = 0, 0
    for b in range(0, (len(cell) + 255) // 256):
        wave = cell[256 * b + 64 * (b % 4):256 * b + 64 * (b % 4) + 64]
        first = list(dict.fromkeys(wave.tolist()))[:8]
        total += len(first) + int((~np.isin(wave, first)).sum())
        waves += 1
    return total / waves


@pytest.mark.parametrize("n", [63, 64, 65, 257, 1023])
@pytest.mark.parametrize("ncell", [(1, 1, 200), (1, 200, 1), (200, 1, 1), (1, 12, 13), (13, 1, 12), (12, 13, 1), (6, 5, 7)])
@pytest.mark.parametrize("nf, order", [(2, 2), (3, 2), (3, 1), (2, 0)])
def test_every_stencil_through_records(core, oracle, nf, order, ncell, n):
    L = tuple(0.5 * k for k in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, shape_order=order)
    prm = cases.oracle_deck(oracle, d).params()
    emu = core.Emu(cases.product_params(d))
    parts, _ = random_case(oracle, nf, ncell, L, n, seed=10 * n + nf)
    at = np.floor(parts["pos"] / 0.5).astype(int)
    cell = (at[:, 2] * ncell[1] + at[:, 1]) * ncell[0] + at[:, 0]
    assert boxes_per_wave(cell) >= 24
    grid = oracle.Grid(nf, prm)
    oracle.deposit_to_mesh(nf, prm, parts, grid)
    want_dep = grid.fab().reshape(emu.ncomp, -1).T.copy()
    oracle.fill_boundary(nf, prm, grid)
    want_rhs = parts.copy()
    oracle.interpolate_rhs_from_mesh(nf, prm, want_rhs, grid)
    for order_of in (np.arange(n), np.argsort(cell, kind="stable")):
        c = core.FlavoredNeutrinoContainer.from_aos(emu, parts[order_of])
        state = core.MultiFab(emu)
        core.deposit_to_mesh(c, state)
        got = state.data.cpu().numpy().reshape(emu.ncomp, -1).T
        assert cases.max_rel_err(got[:, 3:], want_dep[:, 3:]) < 1e-12
        state.FillBoundary()
        core.interpolate_rhs_from_mesh(c, state)
        assert cases.max_rel_err(c.to_aos()["rdata"], want_rhs["rdata"][order_of]) < 1e-12
        emu.sync()
