"""The fused step where four waves share a cell (few cells of more than 64
particles): occupancies around a wave's chunk (64) and a workgroup's round of
four chunks (256), an empty cell and a one-particle one among them, in 3-D and
1-D and one-cell domains, against the oracle with the bars of the occupancy
tests (FP64 1e-12, FP32-bulk 2e-5 of each component's range)."""
import pytest

import cases
from test_gpu_edges import placed, run_fused_against_oracle

pytestmark = pytest.mark.gpu

OCCUPANCY = [257, 0, 1, 64, 65, 256, 255, 513, 300, 128, 600, 63]


@pytest.fixture(scope="module")
def core():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from emu_amd import core as c
    return c


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
@pytest.mark.parametrize("ncell", [(2, 3, 2), (1, 1, 12), (1, 1, 1)])
def test_four_waves_per_cell(core, oracle, nf, prec, ncell):
    L = tuple(0.5 * n for n in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=32, st4_amplitude=1e-3)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    cells = ncell[0] * ncell[1] * ncell[2]
    occ = dict(enumerate(OCCUPANCY[:cells]))
    parts = placed(oracle, deck, ncell, L, occ, seed=4)
    assert len(parts) > 64 * cells
    fixed = 0.3 * 0.5 / oracle.clight if cells > 1 else 0.1 * 0.5 / oracle.clight
    run_fused_against_oracle(core, oracle, nf, deck.params(), emu, parts, prec, 3, fixed, "auto")
