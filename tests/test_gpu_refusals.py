"""What the per-function calls refuse on the host, before any kernel reads a particle."""
import ctypes

import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["deposit", "gather", "rhs"])
def test_more_than_int32_particles_are_unsupported(call):
    import torch
    assert torch.cuda.is_available()
    from emu_amd import core
    from emu_amd.capi import lib
    emu = core.Emu(cases.product_params(cases.fast_flavor_dict(nf=2, ncell=(4, 4, 4))))
    a, b = core.FlavoredNeutrinoContainer(emu, 4).view(), core.FlavoredNeutrinoContainer(emu, 4).view()
    a.np = b.np = 1 << 31
    state = core.MultiFab(emu)
    g = state.view()
    code = {"deposit": lambda: lib().emu_deposit_to_mesh(emu.ctx, ctypes.byref(a), ctypes.byref(g)),
            "gather": lambda: lib().emu_interpolate_rhs_from_mesh(emu.ctx, ctypes.byref(a), ctypes.byref(g)),
            "rhs": lambda: lib().emu_rhs_from_mesh(emu.ctx, ctypes.byref(b), ctypes.byref(a), ctypes.byref(g))}[call]()
    assert code == 12
    assert b"more than 2^31 particles" in lib().emu_last_error(emu.ctx)
