"""Calls inside a caller's own stream capture: Richardson-Lucy updates, and
blocks without an error trace of several frames, are recorded as plain
launches (cooperative ones and their tables' upload stay out), and every
replay, with eager work between, gives the eager result."""
import pytest
import torch

from als_speckle_amd import _capi
from als_speckle_amd.device import Context, Plan

pytestmark = pytest.mark.gpu

N = 256


def rand(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(shape, generator=g, device="cuda")


def crand(shape, seed):
    return torch.complex(rand(shape, seed), rand(shape, seed + 1))


def captured(stream, fn):
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = fn()
    return graph, out


def test_coherence_updates_replay(gpu_ctx):
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        est, mod = crand((100, 90), 1), rand((N, N), 3) + 0.1
        p = Plan(Context(0, stream=stream), N)
        want = p.coherence_rl(est, mod, 3)       # also sizes the work buffers
    graph, out = captured(stream, lambda: p.coherence_rl(est, mod, 3))
    for _ in range(3):
        with torch.cuda.stream(stream):
            out.zero_()
            p.coherence_rl(est, 2.0 * mod, 2)    # eager work on the same buffers
            graph.replay()
        torch.cuda.synchronize()
        assert (out == want).all().item()
    p.check()
    p.close()


def test_batched_block_replays(gpu_ctx):
    hio = (_capi.HIO, 0, 0.8, 0.0, 0.0)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        p = Plan(Context(0, stream=stream), N, batch=4)
        p.set_modulus(N * rand((N, N), 1))
        p.set_support((rand((N, N), 2) > 0.6).float())
        guess = crand((4, N, N), 3)
        p.set_psi(guess)
        p.iterate([hio] * 24, error_trace=False)
        want = p.get_psi()
        p.set_psi(guess)
    graph, _ = captured(stream, lambda: p.iterate([hio] * 8, error_trace=False))
    for _ in range(2):
        with torch.cuda.stream(stream):
            p.set_psi(guess)
            graph.replay()
            p.iterate([hio] * 8, error_trace=False)
            graph.replay()
            got = p.get_psi()
        torch.cuda.synchronize()
        assert (got == want).all().item()
    p.check()
    p.close()
