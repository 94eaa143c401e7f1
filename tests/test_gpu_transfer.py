"""The stack transfer functions (spk_prtf, spk_rftf_stack without an ipsf):
row transforms of the estimates themselves, then the summing column pass.

Sizes at the edges: one row, rows that end inside a band of the layout, whole
frames, one frame, one frame past a group, every shape of the transform, the
two-layout size.  Tolerance, relative 2-norm: a complex64 transform is off by
about 3e-7 of the rms |F|; F / |F| of a pixel by that over |F|, whose square
averages to (3e-7)^2 ln(pixels), about 1.2e-6 per frame against values of
0.9: 5e-6.
"""
import numpy as np
import pytest
import torch

from als_speckle_amd.device import Plan
from oracle import phasing_c128 as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,frames,rows,cols,kw", [
    (16, 1, 1, 1, {}), (16, 9, 16, 16, {}), (32, 5, 31, 2, {}), (64, 4, 13, 64, {}),
    (128, 2, 128, 77, {}), (256, 6, 1, 256, dict(tile=2)), (256, 17, 101, 99, dict(tile=8, ept=16)),
    (512, 5, 187, 203, {}), (512, 64, 40, 512, {}), (1024, 5, 1023, 517, {}),
    (2048, 5, 333, 2048, {}), (4096, 5, 409, 311, {}), (4096, 2, 250, 300, dict(tile=4))])
def test_stack_transfer_functions_match_oracle(gpu_ctx, n, frames, rows, cols, kw):
    rng = np.random.default_rng(n + frames)
    base = rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    stack = np.stack([base + 0.5 * (rng.standard_normal((rows, cols))
                                    + 1j * rng.standard_normal((rows, cols)))
                      for _ in range(frames)]).astype(np.complex64)
    pad = np.zeros((n, n), complex)
    pad[:rows, :cols] = base
    goal = (np.abs(np.fft.fft2(pad)) + 0.5 * np.sqrt(rows * cols)).astype(np.float32)
    p = Plan(gpu_ctx, n, **kw)
    t = torch.from_numpy(stack).cuda()
    got = p.prtf(t).cpu().numpy()
    want = O.prtf(stack.astype(complex), n)
    assert np.linalg.norm(got - want) < 5e-6 * np.linalg.norm(want)
    got = p.rftf_stack(t, torch.from_numpy(goal).cuda()).cpu().numpy()
    want = O.rftf_stack(stack.astype(complex), goal.astype(float))
    assert np.linalg.norm(got - want) < 5e-6 * np.linalg.norm(want)
    p.close()


def test_zero_estimate_and_zero_goal(gpu_ctx):
    """|F| = 0 gives NaN (PRTF, no guard in the reference); a goal of 0 gives
    0 where |F| is not 0, NaN where it is."""
    rng = np.random.default_rng(3)
    stack = (rng.random((3, 20, 20)) + 1j * rng.random((3, 20, 20))).astype(np.complex64)
    goal = np.ones((64, 64), np.float32)
    goal[5, 7] = 0
    p = Plan(gpu_ctx, 64)
    got = p.rftf_stack(torch.from_numpy(stack).cuda(), torch.from_numpy(goal).cuda()).cpu().numpy()
    assert np.isfinite(got).all() and got[37, 39] == 0 and (got == 0).sum() == 1
    stack[1] = 0
    t = torch.from_numpy(stack).cuda()
    assert np.isnan(p.prtf(t).cpu().numpy()).all()
    got = p.rftf_stack(t, torch.from_numpy(goal).cuda()).cpu().numpy()
    assert np.isnan(got[37, 39]) and np.isnan(got).sum() == 1
    p.close()
