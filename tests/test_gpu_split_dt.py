"""The fused step where four waves share a cell, at the computed time step: the
auxiliaries that stage 3 deposits and the bound that stage 4 takes of each cell
(or, with max_adaptive_speedup > 1, a launch of its own), with the crowded cell
first, last and between, and occupancies around a wave's chunk (64) and a
workgroup's round of four chunks (256).  Against the per-function integrator, with the
bars of the occupancy tests (FP64 1e-12, FP32-bulk 2e-5 of each component's range)."""
import pytest

import cases
from test_gpu_edges import placed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from emu_amd import core as c
    return c


@pytest.mark.parametrize("speedup", [0.0, 5.0])
@pytest.mark.parametrize("counts", [(513, 0, 1, 64, 65, 256, 255, 63, 128, 2, 200, 17), (1, 256, 64, 63, 300, 0, 65, 128, 257, 0, 5, 641),
                                    (64, 65, 0, 129, 0, 769, 1, 256, 63, 255, 30, 2)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
@pytest.mark.parametrize("ncell", [(2, 3, 2), (1, 1, 12), (1, 1, 1)])
def test_computed_time_step(core, oracle, nf, prec, ncell, counts, speedup):
    L = tuple(0.5 * n for n in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=32, st4_amplitude=1e-3, flavor_cfl_factor=0.01,
                               max_adaptive_speedup=speedup)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    cells = ncell[0] * ncell[1] * ncell[2]
    occ = dict(enumerate(counts)) if cells > 1 else {0: min(378, 256 + counts[0])}
    parts = placed(oracle, deck, ncell, L, occ, seed=4)
    assert len(parts) > 64 * cells
    c = core.FlavoredNeutrinoContainer.from_aos(emu, parts)
    ref = core.Integrator(emu, core.FlavoredNeutrinoContainer.from_aos(emu, parts))
    st = core.FusedState(emu, c.np, prec)
    st.load(c)
    bar = 1e-12 if prec == "fp64" else 2e-5
    for _ in range(3):
        dt = st.info()["dt"]
        assert dt < 0.4 * 0.5 / oracle.clight # the flavour bound, not the crossing time
        assert dt == pytest.approx(ref.dt, rel=bar)
        st.evolve(1)
        ref.advance()
    st.store(c)
    st.close()
    got, want = cases.by_id(c.to_aos()), cases.by_id(ref.old.to_aos())
    assert cases.max_rel_err(got["rdata"], want["rdata"]) < bar
