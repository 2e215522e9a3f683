"""The fused step's sort plan at the edges of its rows of 64 cells (a wave each, on the
stages' launches), where it moves to its own stream (more than 32768 cells) and
where a wave takes two rows (2^17 cells and more): particles that change cells, in the
first, last and neighbouring rows, against the oracle with the bars of the occupancy
tests (FP64 1e-12, FP32-bulk 2e-5 of each component's range)."""
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
@pytest.mark.parametrize("ncell", [(1, 1, 63), (1, 1, 64), (4, 4, 4), (5, 13, 1), (1, 1, 129), (8, 16, 16), (32, 32, 32),
                                   (33, 32, 32), (64, 64, 32), (52, 51, 50)])
def test_sort_plan_rows(core, oracle, prec, ncell):
    nf = 2
    L = tuple(0.5 * n for n in ncell)
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=L, nphi=12, st4_amplitude=1e-3)
    deck = cases.oracle_deck(oracle, d)
    emu = core.Emu(cases.product_params(d))
    cells = ncell[0] * ncell[1] * ncell[2]
    at = {0, 1, 62, 63, 64, 65, 127, 128, 129, cells // 2, cells - 65, cells - 64, cells - 2, cells - 1}
    occ = {c: 3 + 17 * (i % 5) for i, c in enumerate(sorted(c for c in at if 0 <= c < cells))}
    parts = placed(oracle, deck, ncell, L, occ, seed=12)
    run_fused_against_oracle(core, oracle, nf, deck.params(), emu, parts, prec, 4, 0.45 * 0.5 / oracle.clight, "auto")
