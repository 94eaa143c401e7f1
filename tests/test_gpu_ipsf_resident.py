"""Partially coherent blocks of one frame in one launch (k_resident_ipsf):
bitwise the launches per pass, whose arithmetic it runs; blocks end at
shrinkwraps and DM steps, which run as before; with a spectrum there is none.
"""
import numpy as np
import pytest
import torch

from als_speckle_amd import _capi, synth
from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu

HIO, ER, RAAR, SF, DM, IDLE = ((_capi.HIO, 0, 0.9, 0.0, 0.0), (_capi.ER, 0, 0.0, 0.0, 0.0),
                               (_capi.RAAR, 0, 0.87, 0.0, 0.0), (_capi.SF, 1, 0.0, 0.0, 0.0),
                               (_capi.DM, 0, 0.7, 0.0, 0.0), (_capi.NOOP, 0, 0.0, 0.0, 0.0))
SW = (_capi.HIO, 0, 0.9, 2.0, 0.15)
CALLS = [[HIO, HIO, ER, IDLE, RAAR, SF], [HIO], [ER, ER, HIO, SW, HIO, HIO, DM, HIO, ER]]


def run(ctx, n, resident, trace, spectrum):
    f = synth.make_frame(n, n, shape="disk", radius=n // 6, photons=1e6)
    rng = np.random.default_rng(n)
    x = np.fft.fftfreq(n) * n
    psf = np.exp(-(x[:, None] ** 2 + x[None, :] ** 2) / 8.0)
    ipsf = (np.fft.fft2(psf / psf.sum()) * np.exp(0.1j)).astype(np.complex64)
    p = Plan(ctx, n, resident=resident)
    p.set_modulus(torch.from_numpy(f.modulus).cuda())
    p.set_support(torch.from_numpy(f.support).cuda())
    p.set_ipsf(torch.from_numpy(ipsf).cuda())
    if spectrum:
        p.set_spectrum([0.98, 1.0, 1.02], [0.25, 0.5, 0.25])
    p.set_psi(torch.from_numpy((rng.random((n, n)) + 1j * rng.random((n, n)))
                               .astype(np.complex64)).cuda())
    errs = [p.iterate(c, error_trace=trace) for c in CALLS]
    p.check()
    out = [p.get_psi().cpu().numpy(), p.get_support().cpu().numpy()]
    out += [e.cpu().numpy() for e in errs if e is not None]
    counts = p.resident_counts()
    p.close()
    return out, counts


@pytest.mark.parametrize("n,trace,spectrum", [(64, True, False), (128, False, False),
                                              (256, True, False), (512, True, False),
                                              (1024, True, False), (1024, False, False),
                                              (128, True, True)])
def test_resident_ipsf_equals_per_pass(gpu_ctx, n, trace, spectrum):
    want, none = run(gpu_ctx, n, 2, trace, spectrum)
    got, counts = run(gpu_ctx, n, 0, trace, spectrum)
    # blocks: the first call's five active steps; ER, ER, HIO, SW; HIO (HIO is
    # DM's predecessor and runs per pass); HIO, ER
    assert none == (0, 0) and counts == ((0, 0) if spectrum else (3, 11))
    for a, b in zip(got, want):
        assert np.array_equal(a, b, equal_nan=True)
