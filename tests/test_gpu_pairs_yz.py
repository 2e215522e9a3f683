"""The fused step on a domain of one column with more than 3072 cells: one cell per wave,
as there is no second one along x.  Occupancies around a tile (16) and a chunk (64),
against the oracle with the bars of the occupancy tests (FP64 1e-12, FP32-bulk 2e-5
of each component's range)."""
import pytest

import cases
from test_gpu_edges import placed, run_fused_against_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def core():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from emu_amd import core as c
    return c


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nf", [2, 3])
def test_one_column(core, oracle, nf, prec):
    ncell, L = (1, 59, 61), (0.5, 29.5, 30.5)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=16, st4_amplitude=1e-3)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    occ = {37 * i: n for i, n in enumerate([1, 15, 16, 17, 63, 64, 65, 130, 33])}
    occ[59 * 61 - 1] = 40
    parts = placed(oracle, deck, ncell, L, occ, seed=6)
    run_fused_against_oracle(core, oracle, nf, deck.params(), emu, parts, prec, 3, 0.3 * 0.5 / oracle.clight, "auto")
