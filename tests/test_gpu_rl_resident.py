"""Richardson-Lucy updates in one launch (k_resident_rl): bitwise the launches
per pass, whose transforms and elementwise steps it runs in their order."""
import numpy as np
import pytest
import torch

from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows,cols,iterations,sem", [
    (64, 33, 64, 1, "numpy"), (128, 1, 77, 4, "opencl"), (256, 200, 131, 3, "numpy"),
    (512, 512, 301, 2, "numpy"), (1024, 701, 613, 3, "opencl"), (256, 100, 100, 0, "numpy")])
def test_one_launch_equals_per_pass(gpu_ctx, n, rows, cols, iterations, sem):
    g = torch.Generator(device="cuda").manual_seed(n)
    est = torch.complex(*[torch.rand((rows, cols), generator=g, device="cuda") for _ in range(2)])
    mod = torch.rand((n, n), generator=g, device="cuda") + 0.1
    got = []
    for resident in (2, 0):
        p = Plan(gpu_ctx, n, resident=resident)
        for _ in range(2):                    # the second on used work buffers
            out = p.coherence_rl(est, mod, iterations, sem)
        p.check()
        got.append(out.cpu().numpy())
        p.close()
    assert np.array_equal(got[0], got[1], equal_nan=True) and np.isfinite(got[0]).all()
