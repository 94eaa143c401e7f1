"""The four-column column pass of 2048^2 and 4096^2 (tile 2, 16 values per
thread): bitwise the two-column pass, which runs the steps with a fused
shrinkwrap, over iterates and error traces; several frames, frames idle in a
step, DM's second projection (against one step per call).
"""
import numpy as np
import pytest
import torch

from als_speckle_amd import _capi
from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu

HIO = (_capi.HIO, 0, 0.9, 0.0, 0.0)
KEEP = (_capi.HIO, 0, 0.9, 1.0, 0.0)      # a shrinkwrap that keeps the support: tau 0
DM = (_capi.DM, 0, 0.7, 0.0, 0.0)
IDLE = (_capi.NOOP, 0, 0.0, 0.0, 0.0)


def plan(ctx, n, batch, **kw):
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    p = Plan(ctx, n, batch=batch, shared=False, **kw)
    shape = (batch, n, n) if batch > 1 else (n, n)
    p.set_modulus(n * torch.rand(shape, generator=g, device="cuda"))
    p.set_support((torch.rand(shape, generator=g, device="cuda") > 0.6).float())
    p.set_psi(torch.complex(*[torch.rand(shape, generator=g, device="cuda") for _ in range(2)]))
    return p


@pytest.mark.parametrize("n,batch", [(2048, 1), (2048, 3), (4096, 1)])
def test_equals_the_pass_with_a_fused_shrinkwrap(gpu_ctx, n, batch):
    a, b = plan(gpu_ctx, n, batch), plan(gpu_ctx, n, batch)
    ea = a.iterate([HIO] * 4).cpu().numpy()
    eb = b.iterate([KEEP] * 3 + [HIO]).cpu().numpy()
    assert b.sw_counts() == (3, 0) and torch.equal(a.get_support(), b.get_support())
    assert np.array_equal(ea, eb)
    assert torch.equal(torch.view_as_real(a.get_psi()), torch.view_as_real(b.get_psi()))
    a.close(), b.close()


def test_idle_frames_and_dm(gpu_ctx):
    n = 2048
    a, b = plan(gpu_ctx, n, 2), plan(gpu_ctx, n, 2)
    table = [DM, HIO, DM, IDLE, HIO, DM]          # steps x frames
    ea = a.iterate(table, per_frame=True).cpu().numpy()
    eb = np.concatenate([b.iterate(table[2 * k:2 * k + 2], per_frame=True).cpu().numpy()
                         for k in range(3)])
    assert np.array_equal(ea, eb, equal_nan=True) and np.isnan(ea[1, 1]) and np.isnan(ea).sum() == 1
    assert torch.equal(torch.view_as_real(a.get_psi()), torch.view_as_real(b.get_psi()))
    a.close(), b.close()
