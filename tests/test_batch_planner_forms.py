"""CPU: the forms that the batch engine plans, in the emulator of
tests/batch_emu (see test_batch_planner.py): the tile shapes of nonlinear layers,
one cell per thread and marching strips among them, are planned and only given
to layers that take them."""
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
