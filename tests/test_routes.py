"""Which launches the library's calls make, and what they do when one fails:
its host code on a HIP of host functions (emu/fake_hip.cpp), without a GPU."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def fake_so(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "emu", "fake_hip.cpp"), "-o", so], check=True)
    return so


@pytest.fixture
def program(fake_so):
    def run(text):
        r = subprocess.run([sys.executable, os.path.join(HERE, "emu", "fake_run.py"), fake_so],
                           input=text, capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
        return r.stdout
    return run


def test_column_pass_of_four_columns_where_it_is_faster(program):
    """At 2048^2 from three columns of a band pair on (frames times projections),
    at 4096^2 always."""
    program("""
for n, batch, step, pair in [(2048, 1, HIO, 0), (2048, 2, HIO, 0), (2048, 1, DM, 0),
                             (2048, 3, HIO, 1), (2048, 2, DM, 1), (4096, 1, HIO, 1),
                             (4096, 1, DM, 1), (1024, 4, HIO, 0)]:
    p = Plan(n, batch, resident=2)
    ok(p.iterate([step] * 2))
    got = [(w[1].split("<")[0], int(w[2])) for w in launches() if "colpass" in w[1]]
    tile = 4 if n == 1024 else 2
    want = ("k_colpass_pair", n // 4) if pair else ("k_colpass", n // tile)
    assert got == [want] * 2, (n, batch, step, got)
    p.close()
""")


@pytest.mark.parametrize("ipsf", [False, True])
def test_exchange_buffers_are_emptied_after_a_launch_that_failed(program, ipsf):
    """The polled exchange takes any value that is not the empty pattern: the
    launch that empties new buffers is made again when a launch behind it failed."""
    program("""
p = Plan(256, ipsf=%r)
knob("fail_cooperative", 1)
assert p.iterate([HIO] * 8) == -2
begin = [w for w in launches() if "begin" in w]
assert len(begin) == 1 and int(begin[0][-2]) == 2 * 256 * 256 and begin[0][-1] == "1", begin
for fill in "100":
    ok(p.iterate([HIO] * 8))
    words = launches()
    assert sum(w[0] == "coop" for w in words) == 1
    assert [w[-1] for w in words if "begin" in w] == [fill], words
""" % ipsf)


def test_a_device_too_small_for_a_resident_launch_runs_the_passes(program):
    """A resident launch needs all its workgroups on the device at once: 256 at
    1024^2, 64 at 256^2 (a partition of the device has fewer compute units)."""
    program("""
for cus, n, fits in [(64, 1024, False), (255, 1024, False), (256, 1024, True), (64, 256, True),
                     (63, 256, False), (8, 64, False)]:
    knob("cus", cus)
    for resident in (0, 1):
        for ipsf in (False, True):
            p = Plan(n, ipsf=ipsf, resident=resident)
            ok(p.iterate([HIO] * 8))
            words = launches()
            assert sum(w[0] == "coop" for w in words) == fits, (cus, n, ipsf, words)
            assert sum("rowpass" in w[1] for w in words) == (0 if fits else 8)
            p.close()
        p = Plan(n, resident=resident)
        launches()
        ok(p.coherence(2))
        words = launches()
        assert sum(w[0] == "coop" for w in words) == fits, (cus, n, words)
        assert sum("colpass" in w[1] for w in words) == (3 if fits else 11)
        p.close()
""")


@pytest.mark.parametrize("n,batch", [(256, 4), (1024, 1), (64, 300)])
def test_without_memory_for_the_exchange_buffers_the_passes_run(program, n, batch):
    """A plan that fits the device is not refused for what only its resident form
    would need, and takes that form once there is room."""
    program("""
knob("occupancy", 8 if %d == 64 else 1)
p = Plan(%d, %d)
ok(p.iterate([HIO] * p.batch, per_frame=1))   # the step tables' buffers
launches()
knob("malloc_limit", fake.fake_live())
ok(p.iterate([HIO] * 40))
words = launches()
assert not any(w[0] == "coop" or "begin" in w for w in words), words
assert sum("rowpass" in w[1] for w in words) == 40
knob("malloc_limit", 0)
ok(p.iterate([HIO] * 40))
words = launches()
assert sum(w[0] == "coop" for w in words) == 1 and not any("rowpass" in w[1] for w in words)
""" % (n, n, batch))


def test_launches_in_a_callers_capture_are_plain(program):
    program("""
p, many = Plan(256), Plan(256, 4)
ok(p.coherence(2)), ok(many.iterate([HIO] * 8))
assert sum(w[0] == "coop" for w in launches()) == 2
knob("capturing", 1)
ok(p.coherence(2)), ok(many.iterate([HIO] * 8))
words = launches()
assert not any(w[0] == "coop" for w in words)
assert sum("k_colpass" in w[1] for w in words) == 11 + 8
""")


def test_plan_bytes_count_the_exchange_that_a_plan_takes(program):
    """spk_plan_bytes against what a plan and its blocks allocate, at the batches
    where the resident form changes.  The occupancies are those of a 256-CU
    device: workgroups per compute unit at 64^2, 128^2, 256^2, 512^2, 1024^2."""
    program("""
for n, occupancy in [(64, 8), (128, 8), (256, 4), (512, 2), (1024, 1)]:
    knob("occupancy", occupancy)
    fit = 256 * occupancy // (n // 4)
    for batch in sorted({1, fit - 1, fit, fit + 1, 2 * fit, 2 * fit + 1, 6 * fit, 8 * fit, 8 * fit + 1}):
        if batch < 1 or batch * n * n > 1 << 23:
            continue
        before = fake.fake_live()
        p = Plan(n, batch)
        plan = fake.fake_live() - before
        ok(p.iterate([HIO] * 120))
        taken = fake.fake_live() - before - plan      # exchange, flags; step tables (64 KB)
        if any(w[0] == "coop" for w in launches()):
            taken -= 65536
        size = ctypes.c_size_t()
        ok(lib.spk_plan_bytes(n, batch, 1, 0, ctypes.byref(size)))
        counted = size.value - plan - 65536
        # flags are counted for the most bands (tile 2); nothing else may differ
        flags = min(batch, 2 * fit) * (n // 2) * 128
        assert 0 <= counted - taken <= flags, (n, batch, counted, taken)
        p.close()
""")


def test_exchange_buffers_are_emptied_after_a_reported_give_up(program):
    program("""
p = Plan(256)
fills = []
for gave_up in (0, 1, 0):
    ok(p.iterate([HIO] * 8))
    fills += [w[-1] for w in launches() if "begin" in w]
    knob("sticky", gave_up)
    assert lib.spk_plan_check(p.h) == -2 * gave_up
assert fills == ["1", "0", "1"], fills
""")


def test_a_plan_asks_for_occupancies_with_its_first_block(program):
    """The first question about a size's kernels loads them (5 ms): a plan that
    runs no block of steps does not ask, one that does asks once."""
    program("""
for n, batch in [(1024, 1), (256, 4), (256, 20), (4096, 1)]:
    knob("queries", 0)
    p = Plan(n, batch)
    ok(p.iterate([DM]))
    assert fake.fake_get(b"queries") == 0, (n, batch)
    ok(p.iterate([HIO] * 20))
    asked = fake.fake_get(b"queries")
    assert (asked > 0) == (n < 2048)
    ok(p.iterate([HIO] * 20))
    assert fake.fake_get(b"queries") == asked
    p.close()
""")
