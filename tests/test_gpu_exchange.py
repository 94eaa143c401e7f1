"""The resident launch's exchange of Phi by values that their readers poll
(spk_tune.exchange 4, the default) at the edges of its range: the smallest
frames (64^2: workgroups of half a wavefront; 128^2: one), every mixture of
steps with and without a column phase, launches one after another on the same
buffers, data that look like an empty slot, and a launch after one that gave
up.  Bitwise the per-pass launches, whose arithmetic it runs.
"""
import numpy as np
import pytest
import torch

from als_speckle_amd import _capi, synth
from als_speckle_amd._capi import SpkError
from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu

HIO, ER, SF, IDLE = ((_capi.HIO, 0, 0.9, 0.0, 0.0), (_capi.ER, 0, 0.0, 0.0, 0.0),
                     (_capi.SF, 1, 0.0, 0.0, 0.0), (_capi.NOOP, 0, 0.0, 0.0, 0.0))


def sw(s, sigma=2.0):
    return s[:3] + (sigma, 0.15)


CALLS = {
    "plain": [[HIO] * 5, [HIO, ER, HIO], [SF, HIO]],
    "er": [[ER] * 4 + [HIO] * 2 + [ER], [ER, ER], [HIO, ER, ER, HIO, ER, ER, ER, SF]],
    "idle": [[IDLE, HIO, IDLE, IDLE, ER, IDLE, HIO, IDLE], [HIO, HIO]],
    "shrinkwrap": [[HIO, sw(HIO), ER, ER, sw(ER), ER, HIO, sw(ER, 1.0), sw(HIO), IDLE, HIO],
                   [sw(HIO), HIO, sw(HIO)]],
}


def run(ctx, f, g, calls, trace, **kw):
    p = Plan(ctx, f.modulus.shape[0], **kw)
    p.set_modulus(torch.from_numpy(f.modulus).cuda())
    p.set_support(torch.from_numpy(f.support).cuda())
    p.set_psi(torch.from_numpy(g).cuda())
    errs = [p.iterate(c, error_trace=trace) for c in calls]
    p.check()
    out = [p.get_psi().cpu().numpy(), p.get_support().cpu().numpy()]
    out += [e.cpu().numpy() for e in errs if e is not None]
    counts = p.resident_counts()
    p.close()
    return out, counts


def case(n):
    f = synth.make_frame(n, n, shape="disk", radius=n // 6, photons=1e6)
    rng = np.random.default_rng(n)
    return f, (rng.random((n, n)) + 1j * rng.random((n, n))).astype(np.complex64)


@pytest.mark.parametrize("trace", [True, False])
@pytest.mark.parametrize("name", sorted(CALLS))
@pytest.mark.parametrize("n,tile", [(64, 0), (128, 0), (256, 2), (256, 0), (512, 2), (1024, 0)])
def test_polled_exchange_equals_per_pass(gpu_ctx, n, tile, name, trace):
    f, g = case(n)
    want, none = run(gpu_ctx, f, g, CALLS[name], trace, resident=2, tile=tile)
    got, counts = run(gpu_ctx, f, g, CALLS[name], trace, exchange=4, tile=tile)
    assert none == (0, 0) and counts[0] == len(CALLS[name])
    for a, b in zip(got, want):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("n", [64, 256])
def test_values_that_look_empty(gpu_ctx, n):
    """A guess full of the empty slot's pattern (a NaN) still ends every wait."""
    f, g = case(n)
    g.view(np.uint32)[...] = 0xFFFFFFFF
    out, counts = run(gpu_ctx, f, g, [[HIO] * 4, [ER] * 3 + [HIO]], True, exchange=4)
    assert counts[0] == 2 and np.isnan(out[0]).all() and np.isnan(out[2]).all()


def test_same_plan_after_a_launch_that_gave_up(gpu_ctx):
    """Values that a launch with a poll limit of 1 left unread do not reach the
    plan's next launch: with the limit still 1 that launch may give up again
    (and is reported again), otherwise its result is the per-pass one."""
    n = 256
    f, g = case(n)
    want, _ = run(gpu_ctx, f, g, [[HIO] * 3], True, resident=2)
    p = Plan(gpu_ctx, n, barrier_polls=1, exchange=4)
    p.set_modulus(torch.from_numpy(f.modulus).cuda())
    ok = 0
    for _ in range(3):
        p.set_support(torch.from_numpy(f.support).cuda())
        p.set_psi(torch.from_numpy(g).cuda())
        p.iterate([HIO] * 3)
        try:
            p.check()
        except SpkError as e:
            assert e.code == -2
            continue
        ok += 1
        assert np.array_equal(p.get_psi().cpu().numpy(), want[0])
    p.close()
    again, _ = run(gpu_ctx, f, g, [[HIO] * 3], True, exchange=4)
    assert np.array_equal(again[0], want[0])
