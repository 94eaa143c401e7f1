"""The autotuner measures the launches that its caller's plans will make."""
import contextlib
import types

import torch

from als_speckle_amd import serve, tune


def test_serving_classes_are_tuned_on_the_passes_they_run(monkeypatch):
    """A serving chunk is a plan with resident=2; a shape timed on resident
    launches is another one's best (1024^2 runs 8 values per thread there, 16
    per pass)."""
    plans = []

    class Timed:
        def __init__(self, ctx, n, batch, **kw):
            plans.append(kw["resident"])

        def __getattr__(self, name):
            return lambda *a, **kw: None

    ctx = types.SimpleNamespace(device=torch.device("cpu"), sync=lambda: None)
    monkeypatch.setattr(tune, "Plan", Timed)
    monkeypatch.setattr(tune, "_cache", {})
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda dev: "device")
    monkeypatch.setattr(torch.cuda, "Stream", lambda device: None)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(serve, "Context", lambda index, stream: ctx)
    serve._Class(0, 64, 3, autotune=True)
    assert plans and set(plans) == {2}
    tried = len(plans)
    # a plan that may run resident is not given the serving class's shape
    tune.autotune(ctx, 64, 3, shared=False)
    assert set(plans[tried:]) == {0}
