"""A resident launch that gave up waiting leaves values in the exchange buffers
that nobody took.  The plan's next launch must not take them: after the report
(spk_plan_check asks for emptied buffers) and without it (the launch before
each resident one sees the flag) it gives the per-pass result, bitwise.  Up to
the report everything that leaves the plan is NaN.  The give-up is forced from the host by a poll limit of 1, back to the default after
it; every kernel ends as always."""
import numpy as np
import pytest
import torch

from als_speckle_amd import _capi
from als_speckle_amd._capi import SpkError
from als_speckle_amd.batch import phasing_batch
from als_speckle_amd.device import Plan

pytestmark = pytest.mark.gpu

HIO = (_capi.HIO, 0, 0.9, 0.0, 0.0)


def rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(shape, generator=g, device="cuda")


def crand(shape, seed):
    return torch.complex(rand(shape, seed), rand(shape, seed + 1))


def plan(ctx, n, batch, ipsf, **kw):
    p = Plan(ctx, n, batch=batch, **kw)
    p.set_modulus(n * rand((n, n), 1))
    p.set_support((rand((n, n), 2) > 0.6).float())
    if ipsf:
        p.set_ipsf(crand((n, n), 5) / n)
    return p


def give_up(p):
    with pytest.raises(SpkError) as e:
        p.check()
    assert e.value.code == -2


@pytest.mark.parametrize("reported", [True, False])
@pytest.mark.parametrize("n,batch,ipsf", [(64, 1, False), (1024, 1, False), (256, 1, True),
                                          (256, 5, False), (256, 20, False)])
def test_next_launch_after_a_give_up(gpu_ctx, n, batch, ipsf, reported):
    shape = (batch, n, n) if batch > 1 else (n, n)
    ref = plan(gpu_ctx, n, batch, ipsf, resident=2)
    ref.set_psi(crand(shape, 7))
    trace = ref.iterate([HIO] * 12)
    p = plan(gpu_ctx, n, batch, ipsf)
    p.set_barrier_polls(1)
    p.set_psi(crand(shape, 9))
    lost = p.iterate([HIO] * 100)
    roi = torch.zeros((batch, 9, 11), dtype=torch.complex64, device="cuda")
    p.copy_roi_all(roi, 0, 3, 5, 9, 11)
    assert all(x.isnan().all() for x in (lost, p.get_psi(), roi))
    if reported:
        give_up(p)
    p.set_barrier_polls(0)
    p.set_psi(crand(shape, 7))
    got = p.iterate([HIO] * 12)
    assert p.resident_counts() == (2, 112) and ref.resident_counts() == (0, 0)
    if not reported:
        assert got.isnan().all() and p.get_psi().isnan().all()
        give_up(p)
    else:
        assert torch.equal(got, trace)
    assert torch.equal(torch.view_as_real(p.get_psi()), torch.view_as_real(ref.get_psi()))
    p.check()
    p.close(), ref.close()


def test_coherence_updates_report_and_recover(gpu_ctx):
    n = 512
    est, mod = crand((300, 211), 1), rand((n, n), 3) + 0.1
    p, ref = Plan(gpu_ctx, n), Plan(gpu_ctx, n, resident=2)
    p.set_barrier_polls(1)
    assert p.coherence_rl(est, mod, 10).isnan().all()
    give_up(p)
    p.set_barrier_polls(0)
    got = p.coherence_rl(est, mod, 2)
    p.check()
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(ref.coherence_rl(est, mod, 2)))
    p.close(), ref.close()


def test_batched_trials_queue_their_blocks_and_report_where_results_are_fetched(gpu_ctx,
                                                                                monkeypatch):
    n, checks = 256, []
    check = Plan.check
    monkeypatch.setattr(Plan, "check", lambda self: (checks.append(1), check(self))[1])
    b = phasing_batch(3, gpu_info=gpu_ctx)
    sup = np.zeros((n, n), np.float32)
    sup[90:150, 80:170] = 1
    b.load((n * rand((n, n), 1)).cpu().numpy(), sup)
    b.seed(guesses=crand((3, n, n), 3))
    b.iterate(20)
    stack, mean = b.aligned_average()
    assert b._plan.resident_counts()[0] == 1 and not checks
    assert np.isfinite(b.get_error_trace()).all() and np.isfinite(b.get(mean)).all()
    b._plan.set_barrier_polls(1)
    for fetch in (b.get_error_trace, lambda: b.get(b.roi_stack())):
        b.iterate(100)
        with pytest.raises(SpkError):
            fetch()
    b.iterate(100)
    assert b.aligned_average()[1].isnan().all()
