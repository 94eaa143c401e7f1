"""Resident launches of several frames with one schedule: bitwise the launches
per pass, for full and partial rounds, shared and own modulus and support,
steps with and without a column phase, blocks cut by shrinkwraps and DM steps;
and the default's choice (short blocks, many frames and per-frame schedules
run per pass).
"""
import numpy as np
import pytest
import torch

from als_speckle_amd import _capi
from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu

HIO, ER, SF, DM, IDLE = ((_capi.HIO, 0, 0.9, 0.0, 0.0), (_capi.ER, 0, 0.0, 0.0, 0.0),
                         (_capi.SF, 0, 0.0, 0.0, 0.0), (_capi.DM, 0, 0.7, 0.0, 0.0),
                         (_capi.NOOP, 0, 0.0, 0.0, 0.0))
SW = (_capi.HIO, 0, 0.9, 2.0, 0.2)


def run(ctx, n, batch, shared, calls, trace, **kw):
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    p = Plan(ctx, n, batch=batch, shared=shared, **kw)
    one, all_ = (n, n), (batch, n, n)
    own = one if shared else all_
    p.set_modulus(n * torch.rand(own, generator=g, device="cuda"))
    p.set_support((torch.rand(own, generator=g, device="cuda") > 0.6).float())
    p.set_psi(torch.complex(*[torch.rand(all_, generator=g, device="cuda") for _ in range(2)]))
    errs = [p.iterate(c, error_trace=trace) for c in calls]
    p.check()
    out = [p.get_psi().cpu().numpy(), p.get_support().cpu().numpy()]
    out += [e.cpu().numpy() for e in errs if e is not None]
    counts = p.resident_counts()
    p.close()
    return out, counts


# polled values: one round full and partial; the lean form: the first batch that
# takes it, a full round, remainders, more rounds; 1024^2 in rounds of polled
# values; workgroups of half a wavefront to eight
@pytest.mark.parametrize("n,batch,shared,tile,trace", [
    (64, 2, True, 0, True), (64, 129, False, 0, False), (128, 65, True, 0, True),
    (256, 16, False, 0, True), (256, 17, True, 0, False), (256, 5, True, 2, True),
    (64, 257, True, 0, True), (128, 130, False, 0, True), (256, 33, False, 0, True),
    (256, 35, True, 2, True), (512, 8, False, 0, False), (512, 17, True, 2, True),
    (512, 3, False, 0, True), (512, 9, True, 0, True), (1024, 2, True, 0, True),
    (1024, 3, False, 0, False)])
def test_resident_frames_equal_per_pass(gpu_ctx, n, batch, shared, tile, trace):
    calls = [[HIO] * 4 + [ER] * 3 + [IDLE, SF, HIO], [ER, ER, HIO, DM, HIO, HIO]]
    if not shared:
        calls.append([HIO, HIO, SW, HIO, ER, SW])
    want, none = run(gpu_ctx, n, batch, shared, calls, trace, resident=2, tile=tile)
    got, counts = run(gpu_ctx, n, batch, shared, calls, trace, resident=1, tile=tile)
    # one launch per block whatever the rounds: the first call; ER, ER (HIO
    # emits DM's estimate); HIO, HIO; the two blocks that shrinkwraps end
    assert none == (0, 0) and counts[0] == (3 if shared else 5)
    for a, b in zip(got, want):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("n,batch,steps,resident", [
    (256, 1, 5, False), (256, 1, 6, True), (1024, 1, 2, False), (1024, 1, 3, True),
    (256, 16, 6, True), (256, 33, 11, False), (256, 33, 12, True), (512, 25, 60, False),
    (1024, 4, 40, False)])
def test_default_choice(gpu_ctx, n, batch, steps, resident):
    p = Plan(gpu_ctx, n, batch=batch)
    p.set_modulus(torch.ones((n, n), device="cuda"))
    p.set_support(torch.ones((n, n), device="cuda"))
    p.set_psi(torch.ones((batch, n, n) if batch > 1 else (n, n), dtype=torch.complex64,
                         device="cuda"))
    p.iterate([HIO] * steps)
    assert (p.resident_counts()[0] > 0) == resident
    before = p.resident_counts()
    p.iterate([HIO] * (steps * batch), per_frame=True)   # a schedule per frame
    assert batch == 1 or p.resident_counts() == before
    p.check()
    p.close()
