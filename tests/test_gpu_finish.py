"""The steps after batched trials: every frame's region in one launch, the
phase alignment's sums and rotation, the mean over many frames.

The alignment's tolerance: the angle comes from FP64 sums and the rotation is
one FP32 complex product (2-3 roundings of 6e-8): 5e-7 of the largest value.
The mean adds in FP64 and rounds once: 1e-7.
"""
import numpy as np
import pytest
import torch

from als_speckle_amd._capi import SpkError
from als_speckle_amd.device import Plan
from oracle import phasing_c128 as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,r0,c0,rows,cols,kw", [
    (16, 1, 0, 0, 16, 16, {}), (64, 7, 3, 5, 1, 59, {}), (128, 3, 127, 0, 1, 128, dict(tile=2)),
    (256, 5, 17, 201, 33, 55, dict(tile=8))])
def test_copy_roi_all_equals_single_copies(gpu_ctx, n, batch, r0, c0, rows, cols, kw):
    p = Plan(gpu_ctx, n, batch=batch, **kw)
    p.set_psi(torch.randn((batch, n, n) if batch > 1 else (n, n), dtype=torch.complex64,
                          device="cuda"), mult_support=False)
    one, many = (torch.zeros((batch + 2, rows, cols), dtype=torch.complex64, device="cuda")
                 for _ in range(2))
    for f in range(batch):
        p.copy_roi(f, one, f + 1, r0, c0, rows, cols)
    p.copy_roi_all(many, 1, r0, c0, rows, cols)
    assert torch.equal(torch.view_as_real(one), torch.view_as_real(many))
    for bad in ((3, r0, c0, rows, cols), (-1, r0, c0, rows, cols), (0, n - rows + 1, c0, rows, cols)):
        with pytest.raises(SpkError):
            p.copy_roi_all(many, *bad)
    p.close()


@pytest.mark.parametrize("frames,rows,cols", [(1, 1, 1), (3, 1, 255), (64, 16, 16), (2, 257, 1),
                                              (5, 187, 187), (1, 1030, 1021)])
def test_align_and_mean(gpu_ctx, frames, rows, cols):
    rng = np.random.default_rng(frames * rows + cols)
    z = (rng.random((frames, rows, cols)) + 0.3j * rng.standard_normal((frames, rows, cols)))
    z = (z * np.exp(1j * rng.uniform(-3, 3, (frames, 1, 1)))).astype(np.complex64)
    t = torch.from_numpy(z.copy()).cuda()
    mean = gpu_ctx.stack_mean(t).cpu().numpy()
    assert np.max(np.abs(mean - z.astype(complex).mean(0))) < 1e-7 * np.abs(z).max()
    got = gpu_ctx.align_global_phase(t).cpu().numpy()
    want = O.align_global_phase(z.astype(complex))
    assert np.max(np.abs(got - want)) < 5e-7 * np.abs(z).max()
