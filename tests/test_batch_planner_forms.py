"""CPU: the forms that the batch engine plans, in the emulator of
tests/batch_emu (see test_batch_planner.py): the tile shapes of nonlinear layers,
one cell per thread and marching strips among them, are planned and only given
to layers that take them; plans are captured after their direct passes and
replayed, except those of too many launches."""
import os
import re
import subprocess

import pytest

from test_batch_planner import driver  # noqa: F401  (the emulator's build)


def _run(driver, *args, **env):  # noqa: F811
    r = subprocess.run([driver, *map(str, args)], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1", **env))
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout


def _shapes(out):
    return [int(v) for v in re.search(r"launches by shape:([ \d]+)", out).group(1).split()]


@pytest.mark.parametrize("seed,big,want", [(11, False, 6), (12, False, 6), (21, True, 8), (25, True, 7)])
def test_shapes_of_an_untuned_batch(driver, seed, big, want):  # noqa: F811
    out = _run(driver, seed, 4 if big else 25, EMU_RULE="1", **({"EMU_BIG": "1"} if big else {}))
    n = _shapes(out)
    assert len(n) == 9 and n[want] > 0, out
    assert n[3] > 0 and not any(n[k] for k in (0, 1, 2, 4, 5)), out  # linear layers and the fallback: 64 x 8


@pytest.mark.parametrize("seed", [4, 5, 6, 9, 32, 33])
def test_plans_are_captured_after_their_direct_passes(driver, seed):  # noqa: F811
    """Captured at once, after one pass or after two (seed modulo 3): every
    scenario ends on its own step count across the switch, and graphs were
    replayed (the driver itself fails where none was)."""
    out = _run(driver, seed, 25, **({"EMU_TUNE_TWO": "1"} if seed > 30 else {}))
    m = re.search(r"(\d+) graph replays of plans captured after (\d) passes", out)
    assert int(m.group(1)) > 0 and int(m.group(2)) == seed % 3, out


def test_plans_of_too_many_launches_are_not_captured(driver):  # noqa: F811
    """Seed 11 holds nests of REL_TIME near 4000, whose root step is more than
    4096 launches: their plans run directly, others of the run from graphs."""
    out = _run(driver, 11, 25, EMU_RULE="1")
    m = re.search(r"(\d+) graph replays .* the largest of (\d+) launches, (\d+) nests too deep", out)
    assert int(m.group(1)) > 0 and int(m.group(3)) > 0, out
    assert int(m.group(2)) < 4096, out
