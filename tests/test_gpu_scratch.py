"""The per-function deposit's and gather's scratch leaves most of the free device memory
to the caller, and a call made while little was free does not keep later ones in
small batches."""
import pytest

import cases

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def test_scratch_takes_a_share_of_the_free_memory():
    """2^23 particles of three flavours: 1.7 GB of deposit scratch in one batch.  With
    1.5 GiB free the calls take a quarter of it at most and go through the particles
    in batches, with the same results (sums in another order: the repository's
    1e-12 of each component's range for the deposit, 1e-12 for the right-hand
    side).  With the memory free again the next call takes all it asks for."""
    import torch
    assert torch.cuda.is_available()
    from emu_amd import core
    n = 1 << 23
    L = (4.0, 4.0, 4.0)
    p = cases.product_params(cases.fast_flavor_dict(nf=3, ncell=(8, 8, 8), L=L))
    emu = core.Emu(p)
    g = torch.Generator(device="cuda").manual_seed(1)
    c = core.FlavoredNeutrinoContainer(emu, n)
    c.pos.uniform_(0.0, 4.0, generator=g)
    c.rdata.uniform_(1.0, 2.0, generator=g)
    F = core.FlavoredNeutrinoContainer(emu, n)
    G = core.FlavoredNeutrinoContainer(emu, n)
    want, got = core.MultiFab(emu), core.MultiFab(emu)

    def calls(e, fab, rhs):
        # the containers belong to a context of the same parameters
        fab.emu = e
        for x in (c, rhs):
            x.emu = e
        core.deposit_to_mesh(c, fab)
        fab.FillBoundary()
        core.rhs_from_mesh(rhs, c, fab)
        e.sync()

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    calls(emu, want, F)
    torch.cuda.empty_cache()
    tight = core.Emu(p)
    filler = torch.empty(free() - 3 * GIB // 2, dtype=torch.uint8, device="cuda")
    before = free()
    assert before < 2 * GIB
    calls(tight, got, G)
    assert before - free() <= before // 4 + (4 << 20)
    del filler
    torch.cuda.empty_cache()
    a, b = (x.data.cpu().numpy().reshape(emu.ncomp, -1).T[:, 3:] for x in (got, want))
    assert cases.max_rel_err(a, b) < 1e-12
    scale = F.rdata.abs().amax(1, keepdim=True)
    assert bool(((G.rdata - F.rdata).abs() <= 1e-12 * scale).all())
    del scale
    torch.cuda.empty_cache()
    before = free()
    calls(tight, got, G)
    assert before - free() > GIB
