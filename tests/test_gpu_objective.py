"""The adjoint objective works in the caller's memory alone: nothing of it is shared
with the context's other calls, and its two ways of summing the particles (through
a cell list in dJdY, or one particle per thread) agree."""
import ctypes

import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def inputs(nf, ncell, n, dtype, seed):
    import torch
    from emu_amd import core
    d = cases.fast_flavor_dict(nf=nf, ncell=ncell, L=tuple(0.5 * k for k in ncell))
    emu = core.Emu(cases.product_params(d))
    g = torch.Generator(device="cuda").manual_seed(seed)
    box = torch.tensor([0.5 * k for k in ncell], dtype=torch.float64, device="cuda")[:, None]
    pos = torch.rand((3, n), dtype=torch.float64, device="cuda", generator=g) * box
    Nn = (1.0 + torch.rand((2, n), dtype=torch.float64, device="cuda", generator=g)).to(dtype)
    Y = torch.randn((2 * nf * nf, n), dtype=torch.float64, device="cuda", generator=g).to(dtype)
    work = torch.empty(2 * int(np.prod(ncell)) + 1, dtype=torch.float64, device="cuda")
    return emu, pos, Nn, Y, work


def objective(emu, pos, Nn, Y, work, dJ):
    import torch
    from emu_amd.capi import check, lib
    fn = lib().emu_adj_objective if Y.dtype == torch.float64 else lib().emu_adj_objective_f32
    J = ctypes.c_double()
    p = [ctypes.c_void_p(t.data_ptr()) if t is not None else None for t in (pos, Nn, Y, dJ, work)]
    check(fn(emu.ctx, pos.shape[1], p[0], p[1], p[2], ctypes.byref(J), p[3], p[4]), "emu_adj_objective", emu.ctx)
    return J.value


@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_objective_takes_no_device_memory(dtype):
    """Of 2^20 particles a cell list is 8 MB, four of hipMalloc's 2 MB steps."""
    import torch
    dtype = getattr(torch, dtype)
    first = inputs(2, (8, 8, 8), 4096, dtype, 1) # the kernels' own memory is taken here
    objective(*first, torch.empty_like(first[3]))
    objective(*first, None)
    args = inputs(2, (8, 8, 8), 1 << 20, dtype, 2)
    dJ = torch.empty_like(args[3])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    objective(*args, dJ)
    objective(*args, None)
    assert torch.cuda.mem_get_info()[0] == free


def test_objective_beside_a_deposit_on_another_stream():
    """A deposit in flight on one stream, then the objective of other arrays on
    another: both give what they give by themselves.  J is a sum over 2^20 / 512 =
    2048 particles and 27 targets a cell in any order; the deposit's bar is the
    repository's 1e-12 of each component's range."""
    import torch
    from emu_amd import core
    emu, pos, Nn, Y, work = inputs(2, (8, 8, 8), 1 << 20, torch.float64, 3)
    c = core.FlavoredNeutrinoContainer(emu, 1 << 21)
    K = emu.K
    g = torch.Generator(device="cuda").manual_seed(4)
    c.pos.uniform_(0.0, 4.0, generator=g)
    c.rdata.uniform_(1.0, 2.0, generator=g)
    want = core.MultiFab(emu)
    core.deposit_to_mesh(c, want)
    dJ_want = torch.empty_like(Y)
    J_want = objective(emu, pos, Nn, Y, work, dJ_want)
    got = core.MultiFab(emu)
    dJ = torch.empty_like(Y)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        emu.bind_stream(a)
        core.deposit_to_mesh(c, got)
        emu.bind_stream(b)
        J = objective(emu, pos, Nn, Y, work, dJ)
        torch.cuda.synchronize()
        assert J == pytest.approx(J_want, rel=1e-11)
        assert float((dJ - dJ_want).abs().max()) < 1e-11 * float(dJ_want.abs().max())
        x, y = (t.data.cpu().numpy().reshape(emu.ncomp, -1).T[:, 3:] for t in (got, want))
        assert cases.max_rel_err(x, y) < 1e-12
    emu.bind_stream()


@pytest.mark.parametrize("form", [((4, 3, 5), 4000), ((1, 1, 9), 700), ((1, 1, 1), 65), ((3, 2, 2), 1), ((32, 32, 32), 90)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("nf", [2, 3])
def test_objective_with_and_without_a_list(nf, dtype, form):
    """dJdY of its own (room for the list, unless the cells are many), none, and in
    place of Y.  A cell's sum of n <= 4000 terms is off by at most n eps = 1e-12 of
    the sum of magnitudes m in either order, so J by 4e-12 of the sum of m^2, which
    is J of |Y|; dJ/dY follows from the same sums (and is rounded to float)."""
    import torch
    ncell, n = form
    args = inputs(nf, ncell, n, getattr(torch, dtype), 5)
    emu, pos, Nn, Y, work = args
    dJ, inplace = torch.empty_like(Y), Y.clone()
    J = objective(*args, dJ)
    most = torch.empty_like(Y)
    tol = 4e-12 * objective(emu, pos, Nn, Y.abs(), work, most)
    assert abs(objective(*args, None) - J) <= tol
    assert abs(objective(emu, pos, Nn, inplace, work, inplace) - J) <= tol
    eps = 4e-12 + (1.2e-7 if dtype == "float32" else 0.0)
    assert ((inplace.double() - dJ.double()).abs() <= eps * most.double()).all()
