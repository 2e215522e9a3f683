"""The fused step where a wave takes two cells side by side (grids of more than 3072
cells; in FP64 two flavours of at most 32 particles a cell): pairs of every kind of
occupancy around a tile (16) and a chunk (64), empty cells, odd numbers of columns
(a last cell by itself) and domains of two and three columns (a pair's box wraps onto
itself), against the oracle with the bars of the occupancy tests (FP64 1e-12,
FP32-bulk 2e-5 of each component's range)."""
import pytest

import cases
from test_gpu_edges import placed, run_fused_against_oracle

pytestmark = pytest.mark.gpu

PAIRS = [(0, 1), (1, 0), (16, 17), (15, 16), (64, 5), (63, 65), (33, 80), (0, 129), (130, 0), (32, 32)]


@pytest.fixture(scope="module")
def core():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from emu_amd import core as c
    return c


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
@pytest.mark.parametrize("ncell", [(17, 13, 15), (2, 40, 40), (3, 33, 33)])
def test_two_cells_per_wave(core, oracle, nf, prec, ncell):
    L = tuple(0.5 * n for n in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=16, st4_amplitude=1e-3)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    cells = ncell[0] * ncell[1] * ncell[2]
    rows = cells // ncell[0]
    occ = {}
    for i, pair in enumerate(PAIRS): # along rows that lie apart, from different columns on
        row, col = (i * 37) % rows, (2 * i) % (ncell[0] - 1)
        occ[row * ncell[0] + col], occ[row * ncell[0] + col + 1] = pair
    occ[cells - 1] = 40
    parts = placed(oracle, deck, ncell, L, occ, seed=6)
    assert cells > 3072 and len(parts) <= 32 * cells
    fixed = 0.3 * 0.5 / oracle.clight
    run_fused_against_oracle(core, oracle, nf, deck.params(), emu, parts, prec, 3, fixed, "auto")


@pytest.mark.parametrize("crowded", [0, 1, 16])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
def test_the_time_step_sees_both_cells(core, oracle, nf, prec, crowded):
    """compute_dt's flavour bound comes from the densest cell: the first of a pair, the
    second, or a last column's cell by itself.  Two steps at the computed dt
    against the per-function path, with the same bars."""
    ncell = (17, 13, 15)
    L = tuple(0.5 * n for n in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=16, st4_amplitude=1e-3, flavor_cfl_factor=0.02)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    row = 7 * 17 * 13 + 5 * 17
    parts = placed(oracle, deck, ncell, L, {row + crowded: 150, 40: 12, 2000: 20}, seed=8)
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
    st.close()
